// extern "C" launcher of the persistent grouped FP8 GEMM (forward / data-gradient sites), part of
// libggemm_vark.so. Validates arguments on the host, then launches either the kernel of the
// reference's geometry (grid (num_cus, 1, 1), block (512, 1, 1), 64 KiB dynamic LDS, reference
// bench.py:339-355) for the shapes it takes, the wide-tile kernel (persistent_wide.h: grid
// (num_cus, 1, 1), block (256, 1, 1), 160 KiB static LDS), or, for launches of too few such tiles, the
// mid-tile kernel (mid_gemm.h: one tile per 256-thread workgroup).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "../../include/ggemm_persistent.h"
#include "capi_common.h"
#include "mid_gemm.h"
#include "persistent_kernel.h"
#include "persistent_wide.h"
#include "transpose_tile.h"

GGEMM_DEFINE_PERSISTENT_LIB_KERNEL(_grouped_fp8_persistent_gemm_kernel, false)
GGEMM_DEFINE_PERSISTENT_LIB_KERNEL(_grouped_fp8_persistent_gemm_kernel_e5m2, true)
GGEMM_DEFINE_PERSISTENT_WIDE_KERNEL(_grouped_fp8_persistent_gemm_kernel_wide, false)
GGEMM_DEFINE_PERSISTENT_WIDE_KERNEL(_grouped_fp8_persistent_gemm_kernel_wide_e5m2, true)
GGEMM_DEFINE_MID_GEMM_KERNEL(_grouped_fp8_gemm_kernel_mid64, false, 64)
GGEMM_DEFINE_MID_GEMM_KERNEL(_grouped_fp8_gemm_kernel_mid64_e5m2, true, 64)
GGEMM_DEFINE_MID_GEMM_KERNEL(_grouped_fp8_gemm_kernel_mid128, false, 128)
GGEMM_DEFINE_MID_GEMM_KERNEL(_grouped_fp8_gemm_kernel_mid128_e5m2, true, 128)

static_assert(GGEMM_PERSISTENT_MAX_GROUPS == ggemm::nt::kMaxGroups, "header and kernel agree");

namespace {

using ggemm::host::aligned;
using ggemm::host::device_cus;

int validate(const void* a, const void* b, const void* out, const void* as, const void* bs, const int64_t* offs,
             int G, int N, int K, int sam, int sbg, int sbn, int scm, int scn, int fmt, int64_t M_total) {
  if (!a || !b || !out || !as || !bs || !offs) return GGEMM_E_NULL;
  if (fmt != GGEMM_FP8_E4M3 && fmt != GGEMM_FP8_E5M2) return GGEMM_E_FORMAT;
  if (G <= 0 || G > ggemm::nt::kMaxGroups || N <= 0 || K <= 0 || N % 16 || K % 16) return GGEMM_E_SHAPE;
  if (M_total < 0 || M_total > ggemm::nt::kMaxRow) return GGEMM_E_SHAPE;
  // 32-bit tile indices: every group adds at most one partial M-tile
  const int64_t tiles = (M_total / ggemm::kTileM + G) * (int64_t)((N + 319) / 320);
  if (tiles > ggemm::nt::kMaxTiles) return GGEMM_E_SHAPE;
  if (scn != 1) return GGEMM_E_STRIDE;
  if (sam < K || sbn < K || sam % 16 || sbn % 16 || sbg % 16) return GGEMM_E_STRIDE;
  if ((int64_t)sbg < (int64_t)(N - 1) * sbn + K) return GGEMM_E_STRIDE;
  if (scm < N || scm % 8) return GGEMM_E_STRIDE;
  // 32-bit buffer offsets of a stage: 192 A rows, up to 384 B rows, below the out-of-range offset
  if ((int64_t)sam * ggemm::kTileM >= ggemm::nt::kOob || (int64_t)sbn * 384 >= ggemm::nt::kOob)
    return GGEMM_E_SHAPE;
  if (!aligned(a, 16) || !aligned(b, 16) || !aligned(out, 16)) return GGEMM_E_ALIGN;
  return GGEMM_OK;
}

// Byte transpose over 128 x 128 tiles (ggemm_persistent_transpose_u8), the tile scheme of the
// quantize-and-transpose producer (transpose_tile.h: LDS map tt_off, byte_col): thread t loads 16
// bytes of each of the tile rows t / 8 + 32h (h = 0..3, all loads issued first) into the LDS tile;
// after a barrier it reads the dwords of tile columns 4 (t / 8) .. +3 in tile rows 16 (t % 8) ..
// +15 and writes 16 bytes to each of those four destination rows, so a store instruction's 8
// threads of a column group write one whole 128-byte line. Edge tiles hold whole 16-byte segments.
constexpr int kXT = 128, kXThreads = 256;
typedef unsigned int xv4u __attribute__((ext_vector_type(4)));

__global__ void __launch_bounds__(kXThreads) transpose_u8_kernel(const uint8_t* src, int batch, int rows, int cols,
                                                                 int64_t sb, int64_t sr, uint8_t* dst, int64_t db,
                                                                 int64_t dr) {
  __shared__ __attribute__((aligned(16))) uint8_t s_t[kXT * kXT];
  const int tid = threadIdx.x;
  const int tr = tid >> 3, tc = 16 * (tid & 7);
  const int cg = tid >> 3, rj = tid & 7;
  const int rt = (rows + kXT - 1) / kXT, ct = (cols + kXT - 1) / kXT;
  const int per = rt * ct;
  const int64_t tiles = (int64_t)batch * per;
  for (int64_t it = blockIdx.x; it < tiles; it += gridDim.x) {
    const int b = (int)(it / per);
    const int rem = (int)(it - (int64_t)b * per);
    const int r0 = (rem / ct) * kXT, c0 = (rem % ct) * kXT;
    xv4u v[4];
#pragma unroll
    for (int h = 0; h < 4; ++h)
      if (c0 + tc < cols && r0 + tr + 32 * h < rows)
        v[h] = __builtin_nontemporal_load((const xv4u*)(src + b * sb + (int64_t)(r0 + tr + 32 * h) * sr + c0 + tc));
#pragma unroll
    for (int h = 0; h < 4; ++h)
      if (c0 + tc < cols && r0 + tr + 32 * h < rows) *(xv4u*)(s_t + ggemm::qt::tt_off(tr + 32 * h, tc)) = v[h];
    __syncthreads();
    if (r0 + 16 * rj < rows && c0 + 4 * cg < cols) {
      uint32_t dw[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) dw[i] = *(const uint32_t*)(s_t + ggemm::qt::tt_off(16 * rj + i, 4 * cg));
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        using ggemm::qt::byte_col;
        uint8_t* out = dst + b * db + (int64_t)(c0 + 4 * cg + k) * dr + r0 + 16 * rj;
        __builtin_nontemporal_store(xv4u{byte_col(dw[0], dw[1], dw[2], dw[3], k), byte_col(dw[4], dw[5], dw[6], dw[7], k),
                                          byte_col(dw[8], dw[9], dw[10], dw[11], k),
                                          byte_col(dw[12], dw[13], dw[14], dw[15], k)},
                                    (xv4u*)out);
      }
    }
    __syncthreads();
  }
}

// ggemm_persistent_clear_tail on its own: the rows that a GEMM left as they were.
constexpr int kTailThreads = 256;

__global__ void __launch_bounds__(kTailThreads) clear_tail_kernel(uint16_t* out, int64_t stride_cm, int N,
                                                                  const int64_t* group_offs, int G,
                                                                  int64_t m_total) {
  ggemm::nt::clear_tail_rows(out, stride_cm, N, group_offs, G, m_total);
}

// The wide-tile kernel takes N % 320 == 0 and K % 64 == 0 (persistent_wide.h); its 32-bit buffer
// offsets: 256 A rows and 320 B rows per stage below the out-of-range offset, a C tile's 256 rows
// within num_records.
bool wide_fits(int N, int K, int sam, int sbn, int scm) {
  return ggemm::pw::fits(N, K) && (int64_t)sam * ggemm::pw::kTM < ggemm::nt::kOob &&
         (int64_t)sbn * ggemm::pw::kTN < ggemm::nt::kOob && (int64_t)scm * 2 * ggemm::pw::kTM < ggemm::nt::kOob;
}

// The automatic choice: the wide kernel wherever it fits. Against the 512-thread kernel it measured
// faster at all four fwd / dgrad sites on both row layouts: on the reference's contiguous K = 2880
// rows (half the 128-byte row segments straddle two lines) 2-6 % (5.690 against 5.999 ms over the
// four sites, same box), on line-aligned rows more.
bool wide_preferred(int N, int K, int sam, int sbn, int scm) { return wide_fits(N, K, sam, sbn, scm); }

int64_t mid_tiles(int rows, int G, int N, int64_t M_total) {
  return (M_total / rows + (G < M_total ? G : M_total)) * ((N + 127) / 128);
}

// The second look at a launch of more than four groups that the estimate of mid_preferred gives to 128-row
// tiles: both sides in whole rounds, for rows spread evenly over the groups and for any (half a row tile more
// for each group), and the mean of the two. Of 1553 drawn launches on 128 rows (1 to 64 groups, 1 to 60000 rows,
// features 64 to 5760, even, exponential and Zipf lengths) 35 were more than 3 % slower than before there were mid
// tiles, 16 more than 10 %: 13 groups, 5788 rows, N = K = 2880 75 us, 51 on the wide tiles; 15, 7007, N = 2560, K
// = 5760 112, 85. With this rule 27 and 9 are, and 7 lose a gain of 20 % or more. For up to four groups it lost
// as often as it gained.
bool rows128_faster(int N, double M, double g, double stages, double mem, bool wide, int cus) {
  constexpr int kRun = ggemm::mid::kXcdRun;
  const int tn = wide ? 320 : ggemm::wide_tiles(N, false) ? 384 : 320;
  double mid = 0, big = 0;
  for (const bool even : {true, false}) {
    auto tiles = [&](double h, double w) {
      return (even ? g * std::ceil(M / g / h) : std::max(1.0, M / h + g / 2)) * std::ceil(N / w);
    };
    const double t = tiles(128, 128), all = ggemm::kXcds * kRun, runs = std::floor(t / all);
    // half rounds of two workgroups on every CU of the XCD that takes most tiles (tile_of_block)
    const double most = kRun * runs + std::min<double>(kRun, t - runs * all);
    const double half = std::ceil(most * ggemm::kXcds / cus);
    mid += 6.6 + (0.976 * half / 2 - 0.28) * (stages + 2) + 0.33 * mem;
    const double r = std::ceil(tiles(wide ? ggemm::pw::kTM : ggemm::kTileM, tn) / cus);
    big += wide        ? 2.6 + r * (1.19 * stages + 6.1) + 0.32 * mem
           : tn == 320 ? 2.0 + r * (1.12 * stages + 6.8) + 0.29 * mem
                       : 4.6 + r * (1.27 * stages + 5.0) + 0.43 * mem;
  }
  return mid < 1.05 * big;
}

// The mid-tile kernel's row-tile height (64 or 128) where it is the faster one, else 0: the estimated
// microseconds of each kernel compared. The lengths of the groups are on the device; M_total rows over
// G groups are taken to make max(g, M_total / height + g / 2) row tiles, g the groups that can have a
// row. Per 128-byte K stage and tile: 1.85 us (wide) or 1.75 us (512-thread) for the persistent kernels,
// their tiles one to a CU in whole rounds; 0.69 / 1.06 us for the mid tiles of 64 / 128 rows with two
// workgroups on every CU (0.41 / 0.64 with few), and they feel the memory's time too; 4 us around
// either. Measured (us, the better of 512-thread and wide kernel -> the choice): N = 5760, K = 2880, G =
// 32: 256 rows 149 -> 95 (64), 3072 rows 148 -> 118 (128), 6144 rows 162, mid 182 (stays); N = K = 2880,
// G = 4: 512 rows 38 -> 14, 8192 rows 83 -> 75, 16384 rows 132, mid 153 (stays); N = 2048, K = 1424, G =
// 7: 512 rows 25 -> 9, 5003 rows 28, mid 31 (stays); N = 512, K = 1024, G = 8: 100000 rows 92 -> 77.
int mid_preferred(int G, int N, int K, int scm, int64_t M_total, bool wide, int cus) {
  if (G > ggemm::mid::kMaxGroups || M_total <= 0 || mid_tiles(64, G, N, M_total) > (1 << 22)) return 0;
  if ((int64_t)scm * 2 * 64 >= (int64_t)ggemm::nt::kOob) return 0;   // a wave's rows of C: 32-bit offsets
  const double M = (double)M_total, g = G < M ? G : M;
  const double stages = (K + 127) / 128 + 2;                          // two more for the tile's ends
  const double mem = (M * K + g * N * K + 2 * M * N) / 5.1e6;
  auto tiles = [&](double h, double w) { return std::max(g, M / h + g / 2) * std::ceil(N / w); };
  double big;
  if (wide) {
    big = 4 + std::ceil(tiles(256, 320) / cus) * stages * 1.85;
  } else {
    const int tn = ggemm::wide_tiles(N, false) ? 384 : 320;
    big = 4 + std::ceil(tiles(192, tn) / cus) * stages * (tn == 384 ? 1.75 : 1.58) + 0.2 * mem;
  }
  const double f64 = tiles(64, 128) / (2 * cus), f128 = tiles(128, 128) / (2 * cus);
  const double c64 = 4 + std::max(1.0, f64) * stages * (0.41 + 0.28 * std::min(1.0, f64)) + 0.3 * mem;
  const double c128 = 4 + std::max(1.0, f128) * stages * (0.64 + 0.42 * std::min(1.0, f128)) + 0.3 * mem;
  if (std::min(c64, c128) >= 0.92 * big) return 0;   // near the line the estimate is a few per cent off
  if (c64 < 0.97 * c128) return 64;
  return g <= 4 || rows128_faster(N, M, g, (K + 127) / 128, mem, wide, cus) ? 128 : 0;
}

int launch(const void* a, const void* b, void* out, const float* a_scale, const float* b_scale,
           const int64_t* group_offs, int G, int N, int K, int sam, int sbg, int sbn, int scm, int scn, int fmt,
           int64_t M_total, int kernel, void* stream) {
  int rc = validate(a, b, out, a_scale, b_scale, group_offs, G, N, K, sam, sbg, sbn, scm, scn, fmt, M_total);
  if (rc) return rc;
  const bool fits = wide_fits(N, K, sam, sbn, scm);
  const int zero_tail = (kernel & GGEMM_PERSISTENT_ZERO_TAIL) != 0;
  if (kernel >= 0) kernel &= ~GGEMM_PERSISTENT_ZERO_TAIL;
  const bool automatic = kernel == GGEMM_PERSISTENT_KERNEL_AUTO;
  if (automatic)
    kernel = wide_preferred(N, K, sam, sbn, scm) ? GGEMM_PERSISTENT_KERNEL_WIDE : GGEMM_PERSISTENT_KERNEL_512;
  if (kernel == GGEMM_PERSISTENT_KERNEL_WIDE && !fits) return GGEMM_E_SHAPE;
  if (kernel < GGEMM_PERSISTENT_KERNEL_AUTO || kernel > GGEMM_PERSISTENT_KERNEL_WIDE) return GGEMM_E_SHAPE;
  int cus = 0;
  rc = device_cus(&cus);
  if (rc) return rc;
  if (M_total == 0) return GGEMM_OK;   // no rows: nothing to write
  const bool e5m2 = fmt == GGEMM_FP8_E5M2;
  const int mid = automatic ? mid_preferred(G, N, K, scm, M_total, kernel == GGEMM_PERSISTENT_KERNEL_WIDE, cus) : 0;
  if (mid) {
    auto kern = mid == 64 ? (e5m2 ? _grouped_fp8_gemm_kernel_mid64_e5m2 : _grouped_fp8_gemm_kernel_mid64)
                          : (e5m2 ? _grouped_fp8_gemm_kernel_mid128_e5m2 : _grouped_fp8_gemm_kernel_mid128);
    // at most one partial row tile per group, none for a group without rows; whole runs of 8 XCDs
    const int64_t tiles = mid_tiles(mid, G, N, M_total), run = ggemm::kXcds * ggemm::mid::kXcdRun;
    hipLaunchKernelGGL(kern, dim3((uint32_t)((tiles + run - 1) / run * run)), dim3(ggemm::mid::kNT), 0,
                       (hipStream_t)stream, (const uint8_t*)a, (const uint8_t*)b, (uint16_t*)out, a_scale, b_scale,
                       group_offs, G, N, K, sam, sbg, sbn, scm, scn, (void*)nullptr, (void*)nullptr, M_total, zero_tail);
    return (int)hipGetLastError();
  }
  if (kernel == GGEMM_PERSISTENT_KERNEL_WIDE) {
    auto kern = e5m2 ? _grouped_fp8_persistent_gemm_kernel_wide_e5m2 : _grouped_fp8_persistent_gemm_kernel_wide;
    hipLaunchKernelGGL(kern, dim3(cus), dim3(ggemm::pw::kNT), 0, (hipStream_t)stream, (const uint8_t*)a,
                       (const uint8_t*)b, (uint16_t*)out, a_scale, b_scale, group_offs, G, N, K, sam, sbg, sbn, scm,
                       scn, (void*)nullptr, (void*)nullptr, M_total, zero_tail);
    return (int)hipGetLastError();
  }
  auto kern = e5m2 ? _grouped_fp8_persistent_gemm_kernel_e5m2 : _grouped_fp8_persistent_gemm_kernel;
  hipLaunchKernelGGL(kern, dim3(cus), dim3(ggemm::kThreads), ggemm::kDynLdsBytes, (hipStream_t)stream,
                     (const uint8_t*)a, (const uint8_t*)b, (uint16_t*)out, a_scale, b_scale, group_offs, G, N, K, sam,
                     sbg, sbn, scm, scn, (void*)nullptr, (void*)nullptr, M_total, zero_tail);
  return (int)hipGetLastError();
}

}  // namespace

extern "C" {

int ggemm_persistent_fp8(const void* a, const void* b, void* out, const float* a_scale, const float* b_scale,
                         const int64_t* group_offs, int32_t G, int32_t N, int32_t K, int32_t stride_am,
                         int32_t stride_bg, int32_t stride_bn, int32_t stride_cm, int32_t stride_cn,
                         int32_t a_format, int64_t M_total, void* stream) {
  return launch(a, b, out, a_scale, b_scale, group_offs, G, N, K, stride_am, stride_bg, stride_bn, stride_cm,
                stride_cn, a_format, M_total, GGEMM_PERSISTENT_KERNEL_AUTO, stream);
}

int ggemm_persistent_fp8_kernel(const void* a, const void* b, void* out, const float* a_scale, const float* b_scale,
                                const int64_t* group_offs, int32_t G, int32_t N, int32_t K, int32_t stride_am,
                                int32_t stride_bg, int32_t stride_bn, int32_t stride_cm, int32_t stride_cn,
                                int32_t a_format, int64_t M_total, int32_t kernel, void* stream) {
  return launch(a, b, out, a_scale, b_scale, group_offs, G, N, K, stride_am, stride_bg, stride_bn, stride_cm,
                stride_cn, a_format, M_total, kernel, stream);
}

int32_t ggemm_persistent_selected_kernel(int32_t N, int32_t K, int32_t stride_am, int32_t stride_bn,
                                         int32_t stride_cm) {
  return wide_preferred(N, K, stride_am, stride_bn, stride_cm) ? GGEMM_PERSISTENT_KERNEL_WIDE
                                                               : GGEMM_PERSISTENT_KERNEL_512;
}

int32_t ggemm_persistent_tile_rows(int32_t G, int32_t N, int32_t K, int32_t stride_am, int32_t stride_bn,
                                   int32_t stride_cm, int64_t M_total, int32_t num_cus) {
  const bool wide = wide_preferred(N, K, stride_am, stride_bn, stride_cm);
  const int mid = mid_preferred(G, N, K, stride_cm, M_total, wide, num_cus);
  return mid ? mid : wide ? ggemm::pw::kTM : ggemm::kTileM;
}

int ggemm_persistent_clear_tail(void* out, int32_t N, int32_t stride_cm, const int64_t* group_offs, int32_t G,
                                int64_t M_total, void* stream) {
  if (!out || !group_offs) return GGEMM_E_NULL;
  if (G <= 0 || G > ggemm::nt::kMaxGroups || N <= 0 || N % 16 || M_total < 0 || M_total > ggemm::nt::kMaxRow)
    return GGEMM_E_SHAPE;
  if (stride_cm < N || stride_cm % 8) return GGEMM_E_STRIDE;
  if (!aligned(out, 16)) return GGEMM_E_ALIGN;
  int cus = 0;
  const int rc = device_cus(&cus);
  if (rc) return rc;
  if (M_total == 0) return GGEMM_OK;
  hipLaunchKernelGGL(clear_tail_kernel, dim3(4 * cus), dim3(kTailThreads), 0, (hipStream_t)stream,
                     static_cast<uint16_t*>(out), (int64_t)stride_cm, N, group_offs, G, M_total);
  return (int)hipGetLastError();
}

int ggemm_persistent_transpose_u8(const void* src, int32_t batch, int32_t rows, int32_t cols, int64_t src_bstride,
                                  int64_t src_rstride, void* dst, int64_t dst_bstride, int64_t dst_rstride,
                                  void* stream) {
  if (!src || !dst) return GGEMM_E_NULL;
  if (batch < 0 || rows <= 0 || cols <= 0 || rows % 16 || cols % 16) return GGEMM_E_SHAPE;
  if (src_rstride < cols || dst_rstride < rows || src_rstride % 16 || dst_rstride % 16 || src_bstride % 16 ||
      dst_bstride % 16)
    return GGEMM_E_STRIDE;
  if (batch > 1 && (src_bstride < (int64_t)rows * src_rstride || dst_bstride < (int64_t)cols * dst_rstride))
    return GGEMM_E_STRIDE;
  const int64_t per = (int64_t)((rows + kXT - 1) / kXT) * ((cols + kXT - 1) / kXT);
  if ((int64_t)batch * per > 0x7fffffffLL) return GGEMM_E_SHAPE;
  if (!aligned(src, 16) || !aligned(dst, 16)) return GGEMM_E_ALIGN;
  if (batch == 0) return GGEMM_OK;
  int cus = 0;
  const int rc = device_cus(&cus);
  if (rc) return rc;
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(transpose_u8_kernel),
                                                   kXThreads, 0) != hipSuccess ||
      per_cu < 1)
    per_cu = 1;
  if (per_cu > 3) per_cu = 3;   // as the transposing quantizer: 3 per CU beats the 4 or more that fit
  const int64_t tiles = (int64_t)batch * per, cap = (int64_t)cus * per_cu;
  const int grid = (int)(tiles < cap ? tiles : cap);
  hipLaunchKernelGGL(transpose_u8_kernel, dim3(grid), dim3(kXThreads), 0, (hipStream_t)stream,
                     static_cast<const uint8_t*>(src), batch, rows, cols, src_bstride, src_rstride,
                     static_cast<uint8_t*>(dst), dst_bstride, dst_rstride);
  return (int)hipGetLastError();
}

}  // extern "C"
