// extern "C" launcher library for the variable-K FP8 grouped wgrad kernels (libggemm_vark.so).
// Validates arguments on the host, then launches the persistent kernel with the reference's
// geometry: grid (num_cus, 1, 1), block (512, 1, 1), 64 KiB dynamic LDS
// (reference launcher.cpp:142-171, bench.py:388-398), or the wide-tile (vark_wide.h) or the mid-tile
// kernel (mid_wgrad.h) where it serves the launch better.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "../../include/ggemm_vark.h"
#include "capi_common.h"
#include "mid_wgrad.h"
#include "vark_kernel.h"
#include "vark_wide.h"

GGEMM_DEFINE_TENSORWISE_LIB_KERNEL(_grouped_variable_k_gemm_kernel, false, uint16_t, ggemm::kOutBF16, false)
GGEMM_DEFINE_TENSORWISE_LIB_KERNEL(_grouped_variable_k_gemm_kernel_k32, true, uint16_t, ggemm::kOutBF16, false)
GGEMM_DEFINE_MX_KERNEL(_grouped_variable_k_mxfp8_gemm_kernel)
GGEMM_DEFINE_TENSORWISE_LIB_KERNEL(_grouped_variable_k_gemm_kernel_f32, false, float, ggemm::kOutF32, false)
GGEMM_DEFINE_TENSORWISE_LIB_KERNEL(_grouped_variable_k_gemm_kernel_f32_acc, false, float, ggemm::kOutF32Acc, false)
GGEMM_DEFINE_WIDE_KERNEL(_grouped_variable_k_gemm_kernel_wide, 256, 384, uint16_t, ggemm::kOutBF16, false)
GGEMM_DEFINE_WIDE_KERNEL(_grouped_variable_k_gemm_kernel_wide320, 320, 320, uint16_t, ggemm::kOutBF16, false)
GGEMM_DEFINE_WIDE_KERNEL(_grouped_variable_k_gemm_kernel_wide320_f32, 320, 320, float, ggemm::kOutF32, false)
GGEMM_DEFINE_WIDE_KERNEL(_grouped_variable_k_gemm_kernel_wide320_f32_acc, 320, 320, float, ggemm::kOutF32Acc, false)
GGEMM_DEFINE_TENSORWISE_LIB_KERNEL(_grouped_variable_k_gemm_kernel_swapped, false, uint16_t, ggemm::kOutBF16, true)
GGEMM_DEFINE_WIDE_KERNEL(_grouped_variable_k_gemm_kernel_wide_swapped, 256, 384, uint16_t, ggemm::kOutBF16, true)
GGEMM_DEFINE_WIDE_KERNEL(_grouped_variable_k_gemm_kernel_wide320_swapped, 320, 320, uint16_t, ggemm::kOutBF16, true)
GGEMM_DEFINE_MID_WGRAD_KERNEL(_grouped_variable_k_gemm_kernel_mid, uint16_t, ggemm::kOutBF16, false)
GGEMM_DEFINE_MID_WGRAD_KERNEL(_grouped_variable_k_gemm_kernel_mid_swapped, uint16_t, ggemm::kOutBF16, true)
GGEMM_DEFINE_MID_WGRAD_KERNEL(_grouped_variable_k_gemm_kernel_mid_f32, float, ggemm::kOutF32, false)
GGEMM_DEFINE_MID_WGRAD_KERNEL(_grouped_variable_k_gemm_kernel_mid_f32_acc, float, ggemm::kOutF32Acc, false)
GGEMM_DEFINE_WIDE_MX_KERNEL(_grouped_variable_k_mxfp8_gemm_kernel_wide320)

namespace {

using ggemm::host::aligned;
using ggemm::host::device_cus;

int validate_common(const void* lhs, const void* rhs, const void* out, const void* ls, const void* rs,
                    const int64_t* offs, int G, int OUT_M, int OUT_N, int slm, int srm, int scg, int scm,
                    int scn) {
  if (!lhs || !rhs || !out || !ls || !rs || !offs) return GGEMM_E_NULL;
  if (G <= 0 || OUT_M <= 0 || OUT_N <= 0) return GGEMM_E_SHAPE;
  if (OUT_M % 16 || OUT_N % 16) return GGEMM_E_SHAPE;
  if (scn != 1) return GGEMM_E_STRIDE;
  if (slm < OUT_M || srm < OUT_N || slm % 16 || srm % 16) return GGEMM_E_STRIDE;
  if (scm < OUT_N || scm % 4 || scg % 4) return GGEMM_E_STRIDE;
  if ((int64_t)scg < (int64_t)(OUT_M - 1) * scm + OUT_N) return GGEMM_E_STRIDE;
  // the kernel forms 32-bit buffer offsets of up to 128 rows of a stage
  if ((int64_t)slm * 129 > INT32_MAX || (int64_t)srm * 129 > INT32_MAX) return GGEMM_E_SHAPE;
  // ... and 32-bit tile indices: at most 2^30 output tiles (counted with the narrower 320 tile)
  const int64_t tiles = (int64_t)((OUT_M + ggemm::kTileM - 1) / ggemm::kTileM) * ((OUT_N + 319) / 320);
  if ((int64_t)G * tiles > (int64_t(1) << 30)) return GGEMM_E_SHAPE;
  if (!aligned(lhs, 16) || !aligned(rhs, 16) || !aligned(out, 8)) return GGEMM_E_ALIGN;
  return GGEMM_OK;
}

// Wide-tile kernels (tile = its OUT_M height): 320 x 320 where it divides both output dims (no
// partial tiles), else 256 x 384 where OUT_N is a multiple of 384 (N-ragged tiles would need
// per-lane store masks; rows past OUT_M fall outside the C buffer resource); a group of C must be
// addressable with 32-bit byte offsets. 0: no wide kernel takes the shape.
int wide_tile_for(int OUT_M, int OUT_N, int scm) {
  if ((int64_t)OUT_M * scm * 2 >= INT32_MAX) return 0;
  if (OUT_M % 320 == 0 && OUT_N % 320 == 0) return 320;
  if (OUT_N % 384 == 0) return 256;
  return 0;
}

// The wide kernels' epilogues store 16-byte chunks of C rows: every row and group must start on 16
// bytes. scm / scg in bf16 elements (twice the fp32 strides for an fp32 C).
bool wide_rows_aligned(const void* out, int64_t scm, int64_t scg) {
  return aligned(out, 16) && scm % 8 == 0 && scg % 8 == 0;
}

// The bf16 entry points run a wide-tile kernel where one takes the shape, C rows start on 16 bytes
// and the problem is large enough to fill its tiles (OUT_M >= 1024); otherwise the 192 x 384 /
// 192 x 320 kernel.
int wide_selected(int OUT_M, int OUT_N, int64_t scm, int64_t scg, const void* out) {
  return OUT_M >= 1024 && wide_rows_aligned(out, scm, scg) ? wide_tile_for(OUT_M, OUT_N, (int)scm) : 0;
}

int64_t mid_tiles(int G, int OUT_M, int OUT_N) {
  return (int64_t)G * ((OUT_M + ggemm::mid::kWT - 1) / ggemm::mid::kWT) *
         ((OUT_N + ggemm::mid::kWT - 1) / ggemm::mid::kWT);
}

// The second look at a launch that the estimate of mid_preferred gives to the mid tiles, where both features
// are over 1280: with tiles of equal lengths both sides run in whole rounds, which that estimate, made for the
// tails of many unlike tiles, spreads out, and the larger tiles' rates and fixed costs are those of launches
// without the read of the dispatch packet. Mid tiles: 1.15 of a tile's time a round of two to a CU, 0.8 the last
// one with one to a CU, on the XCD that takes most of them (tile_of_block); 192-row ones: 1.62, and 1.1 to 1.6
// for a last round; wide 1.67. Of 7661 drawn launches for the mid tiles (1 to 64 groups, 1 to 131072 tokens,
// features 64 to 5760, even, exponential and Zipf lengths) 136 were more than 3 % slower than before there were
// mid tiles, 73 more than 10 %: [1, 2880, 2880] of 100930 tokens 1843 us, 1403 on the large tiles; [5, 2544,
// 1744] of 17692 122, 94; [2, 2880, 3312] of 106369 1574, 1122. With this rule 78 and 35 are, and 4 lose a gain
// of 20 % or more. Narrower outputs stay with the mid tiles: of those that the same line would take back the even
// lengths are slower on them (0.90 in the median), the unlike ones, whose longest group alone counts, faster
// (1.2).
bool whole_rounds_faster(int G, int OUT_M, int OUT_N, bool f32, double stages, int wide_tile, int cus) {
  constexpr int kRun = ggemm::mid::kXcdRun;
  const int64_t t = mid_tiles(G, OUT_M, OUT_N), all = ggemm::kXcds * kRun;
  const double slots = 2.0 * cus / ggemm::kXcds;             // of an XCD
  const double r = (kRun * (t / all) + std::min<int64_t>(kRun, t % all)) / slots, rest = r - std::floor(r);
  const double c_us = (double)G * OUT_M * OUT_N * (f32 ? 6 : 2) / 5e6;   // C written; fp32: the two modes' mean
  const double mid = 3.5 + (1.15 * std::floor(r) + (rest == 0 ? 0 : rest <= 0.5 ? 0.8 : 1.15)) * (0.88 * stages + 3.3) +
                     (f32 ? 0.2 * c_us : 0);
  auto rounds = [&](int h, int n) { return (double)G * ((OUT_M + h - 1) / h) * ((OUT_N + n - 1) / n) / cus; };
  double big;
  if (wide_tile) {
    big = 9 + std::ceil(wide_tile == 320 ? rounds(320, 320) : rounds(256, 384)) * (1.67 * stages + 4) +
          (f32 ? 0.7 * c_us : 0);
  } else {
    const double b = rounds(ggemm::kTileM, ggemm::wide_tiles(OUT_N, false) ? 384 : 320), last = b - std::floor(b);
    big = 10 + (1.62 * std::floor(b) + (last == 0 ? 0 : b < 1 ? 1.2 + 0.55 * last : 1.1 + 0.5 * last)) * (stages + 1) +
          0.85 * c_us;
  }
  return mid < 0.95 * big;
}

// Whether the mid-tile kernel is the faster one: the estimated microseconds of both sides compared,
// M_total / G tokens in every group. Per 128-token stage and tile: 2.06 us for a wide tile and 1.2
// (few CUs busy) to 2.1 us for a 192-row one, tiles one to a CU in whole rounds; 0.55 (few) to 1.27 us
// (two workgroups on every CU) for a mid tile; a tile's ends cost 3 stages more (an fp32 C: 4; wide 7
// us, fp32 16, between the 9 of writing and the 30 of accumulating); 4 to 7 us around all. wide_tile: the
// wide kernel the entry would run, 0 the 192-row kernel. Measured (us, large -> mid): 64 x 128, 512
// tokens, G = 4: 14 -> 5.3; 512 x 1024, G = 8: 1000 tokens 15 -> 6.3, 100000 tokens 137 -> 69; 1024 x 2048,
// G = 2, 8000 tokens 51 -> 25; 2880 x 2880, G = 4: 4096 tokens 54, mid 63 (stays), accumulated fp32 1024
// tokens 77 -> 52; 1600 x 1600, G = 12: 1000 tokens 24, mid 24 (stays), accumulated 63 -> 42, 100000
// tokens 294, mid 354 (stays). The fp32 modes take one line for both, so that accumulating adds exactly
// what the fp32 mode writes. No token count (INT64_MAX): the large kernels.
bool mid_preferred(int G, int OUT_M, int OUT_N, int64_t scm, int64_t scg, const void* out, bool f32, int64_t M_total,
                   int wide_tile, int cus) {
  const int64_t w = f32 ? 2 : 1;                             // strides in bf16 elements
  if (G > ggemm::mid::kMaxGroups || M_total > INT32_MAX || !wide_rows_aligned(out, w * scm, w * scg)) return false;
  if (scm * 2 * w * 64 >= (int64_t)ggemm::mid::kOob) return false;   // a wave's rows of C: 32-bit offsets
  if (mid_tiles(G, OUT_M, OUT_N) > (1 << 22)) return false;
  const double stages = (double)M_total / G / ggemm::kKStep + 0.5;
  auto tiles = [&](int h, int n) { return (double)G * ((OUT_M + h - 1) / h) * ((OUT_N + n - 1) / n); };
  const double f = tiles(ggemm::mid::kWT, ggemm::mid::kWT) / (2 * cus);
  const double mid = 4 + std::max(1.0, f) * (stages + (f32 ? 4 : 3)) * (0.55 + 0.72 * std::min(1.0, f));
  double big;
  if (wide_tile) {
    const double t = wide_tile == 320 ? tiles(320, 320) : tiles(256, 384);
    big = 5 + std::ceil(t / cus) * (stages * 2.06 + (f32 ? 16 : 7));
  } else {
    const double t = tiles(ggemm::kTileM, ggemm::wide_tiles(OUT_N, false) ? 384 : 320) / cus;
    big = 7 + std::ceil(t) * (stages + 3) * (1.2 + 0.9 * std::min(1.0, t));
  }
  if (mid >= 0.92 * big) return false;                       // near the line the estimate is a few per cent off
  return std::min(OUT_M, OUT_N) <= 1280 || whole_rounds_faster(G, OUT_M, OUT_N, f32, stages, wide_tile, cus);
}

// swapped: e5m2 LHS, e4m3 RHS (bf16 C only)
int launch_wide(bool swapped, int tile, int out_mode, const void* lhs, const void* rhs, void* out,
                const float* lhs_scale, const float* rhs_scale, const int64_t* group_offs, int32_t G, int32_t OUT_M,
                int32_t OUT_N, int32_t slm, int32_t srm, int32_t scg, int32_t scm, int32_t scn, int64_t M_total, void* stream) {
  int cus = 0;
  int rc = device_cus(&cus);
  if (rc) return rc;
  // the kernels keep token counts in 32 bits: a group never exceeds 2^31 - 1 tokens
  const int64_t m_total = M_total < INT32_MAX ? M_total : INT32_MAX;
  const dim3 grid(cus), block(ggemm::wide::kNT);
  if (out_mode == GGEMM_OUT_BF16) {
    auto kern = swapped ? (tile == 320 ? _grouped_variable_k_gemm_kernel_wide320_swapped
                                       : _grouped_variable_k_gemm_kernel_wide_swapped)
                        : (tile == 320 ? _grouped_variable_k_gemm_kernel_wide320 : _grouped_variable_k_gemm_kernel_wide);
    hipLaunchKernelGGL(kern, grid, block, 0, (hipStream_t)stream, (const uint8_t*)lhs, (const uint8_t*)rhs,
                       (uint16_t*)out, lhs_scale, rhs_scale, group_offs, G, OUT_M, OUT_N, slm, srm, scg, scm, scn,
                       (void*)nullptr, (void*)nullptr, m_total);
  } else {
    auto kern = out_mode == GGEMM_OUT_F32 ? _grouped_variable_k_gemm_kernel_wide320_f32
                                          : _grouped_variable_k_gemm_kernel_wide320_f32_acc;
    hipLaunchKernelGGL(kern, grid, block, 0, (hipStream_t)stream, (const uint8_t*)lhs, (const uint8_t*)rhs,
                       (float*)out, lhs_scale, rhs_scale, group_offs, G, OUT_M, OUT_N, slm, srm, scg, scm, scn,
                       (void*)nullptr, (void*)nullptr, m_total);
  }
  return (int)hipGetLastError();
}

// The mid-tile kernel's launch, arguments as for the entry points; out_mode GGEMM_OUT_*.
int launch_mid(bool swapped, int out_mode, const void* lhs, const void* rhs, void* out, const float* lhs_scale,
               const float* rhs_scale, const int64_t* group_offs, int32_t G, int32_t OUT_M, int32_t OUT_N, int32_t slm,
               int32_t srm, int32_t scg, int32_t scm, int32_t scn, int64_t M_total, void* stream) {
  const int64_t tiles = mid_tiles(G, OUT_M, OUT_N), run = ggemm::kXcds * ggemm::mid::kXcdRun;
  const dim3 grid((uint32_t)((tiles + run - 1) / run * run)), block(ggemm::mid::kNT);
  if (out_mode == GGEMM_OUT_BF16) {
    auto kern = swapped ? _grouped_variable_k_gemm_kernel_mid_swapped : _grouped_variable_k_gemm_kernel_mid;
    hipLaunchKernelGGL(kern, grid, block, 0, (hipStream_t)stream, (const uint8_t*)lhs, (const uint8_t*)rhs,
                       (uint16_t*)out, lhs_scale, rhs_scale, group_offs, G, OUT_M, OUT_N, slm, srm, scg, scm, scn,
                       (void*)nullptr, (void*)nullptr, M_total);
  } else {
    auto kern = out_mode == GGEMM_OUT_F32 ? _grouped_variable_k_gemm_kernel_mid_f32
                                          : _grouped_variable_k_gemm_kernel_mid_f32_acc;
    hipLaunchKernelGGL(kern, grid, block, 0, (hipStream_t)stream, (const uint8_t*)lhs, (const uint8_t*)rhs,
                       (float*)out, lhs_scale, rhs_scale, group_offs, G, OUT_M, OUT_N, slm, srm, scg, scm, scn,
                       (void*)nullptr, (void*)nullptr, M_total);
  }
  return (int)hipGetLastError();
}

}  // namespace

extern "C" {

enum class Mfma { kK128, kK32, kK128Swapped };   // swapped: e5m2 LHS, e4m3 RHS

// m_total: the token count group offsets are clamped to on the device (INT64_MAX for the entry
// points with the reference's argument list, which carries none).
static int launch_tensorwise(Mfma mfma, const void* lhs, const void* rhs, void* out, const float* lhs_scale,
                             const float* rhs_scale, const int64_t* group_offs, int32_t G, int32_t OUT_M,
                             int32_t OUT_N, int32_t slm, int32_t srm, int32_t scg, int32_t scm, int32_t scn,
                             int64_t m_total, void* stream) {
  int rc = validate_common(lhs, rhs, out, lhs_scale, rhs_scale, group_offs, G, OUT_M, OUT_N, slm, srm, scg, scm,
                           scn);
  if (rc) return rc;
  if (m_total < 0) return GGEMM_E_SHAPE;
  int cus = 0;
  rc = device_cus(&cus);
  if (rc) return rc;
  const int tile = mfma == Mfma::kK32 ? 0 : wide_selected(OUT_M, OUT_N, scm, scg, out);
  if (mfma != Mfma::kK32 && mid_preferred(G, OUT_M, OUT_N, scm, scg, out, false, m_total, tile, cus))
    return launch_mid(mfma == Mfma::kK128Swapped, GGEMM_OUT_BF16, lhs, rhs, out, lhs_scale, rhs_scale, group_offs, G,
                      OUT_M, OUT_N, slm, srm, scg, scm, scn, m_total, stream);
  if (tile)
    return launch_wide(mfma == Mfma::kK128Swapped, tile, GGEMM_OUT_BF16, lhs, rhs, out, lhs_scale, rhs_scale,
                       group_offs, G, OUT_M, OUT_N, slm, srm, scg, scm, scn, m_total, stream);
  auto kern = mfma == Mfma::kK32          ? _grouped_variable_k_gemm_kernel_k32
              : mfma == Mfma::kK128Swapped ? _grouped_variable_k_gemm_kernel_swapped
                                           : _grouped_variable_k_gemm_kernel;
  hipLaunchKernelGGL(kern, dim3(cus), dim3(ggemm::kThreads), ggemm::kDynLdsBytes, (hipStream_t)stream,
                     (const uint8_t*)lhs, (const uint8_t*)rhs, (uint16_t*)out, lhs_scale, rhs_scale, group_offs, G,
                     OUT_M, OUT_N, slm, srm, scg, scm, scn, (void*)nullptr, (void*)nullptr, m_total);
  return (int)hipGetLastError();
}

int ggemm_vark_wgrad_fp8_wide(const void* lhs, const void* rhs, void* out, const float* lhs_scale,
                              const float* rhs_scale, const int64_t* group_offs, int32_t G, int32_t OUT_M,
                              int32_t OUT_N, int32_t stride_lhs_m, int32_t stride_rhs_m, int32_t stride_cg,
                              int32_t stride_cm, int32_t stride_cn, int64_t M_total, int32_t tile_m,
                              int32_t out_mode, void* stream) {
  if (out_mode != GGEMM_OUT_BF16 && out_mode != GGEMM_OUT_F32 && out_mode != GGEMM_OUT_F32_ACCUM)
    return GGEMM_E_FORMAT;
  int rc = validate_common(lhs, rhs, out, lhs_scale, rhs_scale, group_offs, G, OUT_M, OUT_N, stride_lhs_m,
                           stride_rhs_m, stride_cg, stride_cm, stride_cn);
  if (rc) return rc;
  if (M_total < 0) return GGEMM_E_SHAPE;
  // fp32 C: the same byte bound as a bf16 C twice as wide
  const int fit = wide_tile_for(OUT_M, OUT_N, out_mode == GGEMM_OUT_BF16 ? stride_cm : 2 * stride_cm);
  int tile = tile_m == 0 ? fit : tile_m;
  if (tile == 320 && (OUT_M % 320 || OUT_N % 320)) tile = 0;
  if (tile == 256 && (OUT_N % 384 || out_mode != GGEMM_OUT_BF16)) tile = 0;   // fp32 epilogues: 320 x 320
  if ((tile != 256 && tile != 320) || fit == 0) return GGEMM_E_SHAPE;
  const int64_t w = out_mode == GGEMM_OUT_BF16 ? 1 : 2;   // strides in bf16 elements
  if (!wide_rows_aligned(out, w * stride_cm, w * stride_cg)) return GGEMM_E_ALIGN;   // 16-byte row chunks
  return launch_wide(false, tile, out_mode, lhs, rhs, out, lhs_scale, rhs_scale, group_offs, G, OUT_M, OUT_N, stride_lhs_m,
                     stride_rhs_m, stride_cg, stride_cm, stride_cn, M_total, stream);
}

int ggemm_vark_wgrad_fp8(const void* lhs, const void* rhs, void* out, const float* lhs_scale, const float* rhs_scale,
                         const int64_t* group_offs, int32_t G, int32_t OUT_M, int32_t OUT_N, int32_t stride_lhs_m,
                         int32_t stride_rhs_m, int32_t stride_cg, int32_t stride_cm, int32_t stride_cn,
                         void* stream) {
  return launch_tensorwise(Mfma::kK128, lhs, rhs, out, lhs_scale, rhs_scale, group_offs, G, OUT_M, OUT_N, stride_lhs_m,
                           stride_rhs_m, stride_cg, stride_cm, stride_cn, INT64_MAX, stream);
}

int ggemm_vark_wgrad_fp8_k32(const void* lhs, const void* rhs, void* out, const float* lhs_scale,
                             const float* rhs_scale, const int64_t* group_offs, int32_t G, int32_t OUT_M,
                             int32_t OUT_N, int32_t stride_lhs_m, int32_t stride_rhs_m, int32_t stride_cg,
                             int32_t stride_cm, int32_t stride_cn, void* stream) {
  return launch_tensorwise(Mfma::kK32, lhs, rhs, out, lhs_scale, rhs_scale, group_offs, G, OUT_M, OUT_N, stride_lhs_m,
                           stride_rhs_m, stride_cg, stride_cm, stride_cn, INT64_MAX, stream);
}

int ggemm_vark_wgrad_fp8_out(const void* lhs, const void* rhs, void* out, const float* lhs_scale,
                             const float* rhs_scale, const int64_t* group_offs, int32_t G, int32_t OUT_M,
                             int32_t OUT_N, int32_t stride_lhs_m, int32_t stride_rhs_m, int32_t stride_cg,
                             int32_t stride_cm, int32_t stride_cn, int32_t out_mode, int64_t M_total,
                             void* stream) {
  if (out_mode == GGEMM_OUT_BF16)
    return launch_tensorwise(Mfma::kK128, lhs, rhs, out, lhs_scale, rhs_scale, group_offs, G, OUT_M, OUT_N, stride_lhs_m,
                             stride_rhs_m, stride_cg, stride_cm, stride_cn, M_total, stream);
  if (out_mode != GGEMM_OUT_F32 && out_mode != GGEMM_OUT_F32_ACCUM) return GGEMM_E_FORMAT;
  int rc = validate_common(lhs, rhs, out, lhs_scale, rhs_scale, group_offs, G, OUT_M, OUT_N, stride_lhs_m,
                           stride_rhs_m, stride_cg, stride_cm, stride_cn);
  if (rc) return rc;
  if (M_total < 0) return GGEMM_E_SHAPE;
  if (!aligned(out, 16)) return GGEMM_E_ALIGN;    // 16-byte fp32 row segments
  int cus = 0;
  rc = device_cus(&cus);
  if (rc) return rc;
  // fp32 C takes the 320 x 320 wide-tile kernel where the bf16 C of the same shape would
  const bool wide = wide_selected(OUT_M, OUT_N, 2 * (int64_t)stride_cm, 2 * (int64_t)stride_cg, out) == 320;
  if (mid_preferred(G, OUT_M, OUT_N, stride_cm, stride_cg, out, true, M_total, wide ? 320 : 0, cus))
    return launch_mid(false, out_mode, lhs, rhs, out, lhs_scale, rhs_scale, group_offs, G, OUT_M, OUT_N, stride_lhs_m,
                      stride_rhs_m, stride_cg, stride_cm, stride_cn, M_total, stream);
  if (wide)
    return launch_wide(false, 320, out_mode, lhs, rhs, out, lhs_scale, rhs_scale, group_offs, G, OUT_M, OUT_N,
                       stride_lhs_m, stride_rhs_m, stride_cg, stride_cm, stride_cn, M_total, stream);
  auto kern = out_mode == GGEMM_OUT_F32 ? _grouped_variable_k_gemm_kernel_f32 : _grouped_variable_k_gemm_kernel_f32_acc;
  hipLaunchKernelGGL(kern, dim3(cus), dim3(ggemm::kThreads), ggemm::kDynLdsBytes, (hipStream_t)stream,
                     (const uint8_t*)lhs, (const uint8_t*)rhs, (float*)out, lhs_scale, rhs_scale, group_offs, G, OUT_M,
                     OUT_N, stride_lhs_m, stride_rhs_m, stride_cg, stride_cm, stride_cn, (void*)nullptr, (void*)nullptr,
                     M_total);
  return (int)hipGetLastError();
}

int ggemm_vark_wgrad_fp8_swapped(const void* lhs, const void* rhs, void* out, const float* lhs_scale,
                                 const float* rhs_scale, const int64_t* group_offs, int32_t G, int32_t OUT_M,
                                 int32_t OUT_N, int32_t stride_lhs_m, int32_t stride_rhs_m, int32_t stride_cg,
                                 int32_t stride_cm, int32_t stride_cn, int64_t M_total, void* stream) {
  return launch_tensorwise(Mfma::kK128Swapped, lhs, rhs, out, lhs_scale, rhs_scale, group_offs, G, OUT_M, OUT_N,
                           stride_lhs_m, stride_rhs_m, stride_cg, stride_cm, stride_cn, M_total, stream);
}

// tile_m: 0 = the wide 320 x 320 kernel where the bf16 tensorwise entry would run it, else the
// 192-row kernel; 320 / 192 = that kernel (320 only for shapes it takes)
static int launch_mx(int32_t tile_m, const void* lhs, const void* rhs, void* out, const uint8_t* lhs_scale,
                     const uint8_t* rhs_scale, const int64_t* group_offs, int32_t G, int32_t OUT_M, int32_t OUT_N,
                     int32_t stride_lhs_m, int32_t stride_rhs_m, int32_t stride_cg, int32_t stride_cm,
                     int32_t stride_cn, int32_t stride_lhs_scale, int32_t stride_rhs_scale, int64_t M_total,
                     void* stream) {
  int rc = validate_common(lhs, rhs, out, lhs_scale, rhs_scale, group_offs, G, OUT_M, OUT_N, stride_lhs_m,
                           stride_rhs_m, stride_cg, stride_cm, stride_cn);
  if (rc) return rc;
  if (M_total < 0) return GGEMM_E_SHAPE;
  if (stride_lhs_scale < OUT_M || stride_rhs_scale < OUT_N || stride_lhs_scale % 16 || stride_rhs_scale % 16)
    return GGEMM_E_STRIDE;
  if (!aligned(lhs_scale, 16) || !aligned(rhs_scale, 16)) return GGEMM_E_ALIGN;
  if (tile_m != 0 && tile_m != 320 && tile_m != 192) return GGEMM_E_SHAPE;
  bool wide = tile_m == 0 ? wide_selected(OUT_M, OUT_N, stride_cm, stride_cg, out) == 320 : tile_m == 320;
  if (tile_m == 320) {
    if (wide_tile_for(OUT_M, OUT_N, stride_cm) != 320) return GGEMM_E_SHAPE;
    if (!wide_rows_aligned(out, stride_cm, stride_cg)) return GGEMM_E_ALIGN;    // 16-byte row chunks
  }
  int cus = 0;
  rc = device_cus(&cus);
  if (rc) return rc;
  if (wide) {
    // the kernels keep token counts in 32 bits: a group never exceeds 2^31 - 1 tokens
    const int64_t m_total = M_total < INT32_MAX ? M_total : INT32_MAX;
    hipLaunchKernelGGL(_grouped_variable_k_mxfp8_gemm_kernel_wide320, dim3(cus), dim3(ggemm::wide::kNT), 0,
                       (hipStream_t)stream, (const uint8_t*)lhs, (const uint8_t*)rhs, (uint16_t*)out, lhs_scale,
                       rhs_scale, group_offs, G, OUT_M, OUT_N, stride_lhs_m, stride_rhs_m, stride_cg, stride_cm,
                       stride_cn, stride_lhs_scale, stride_rhs_scale, m_total);
    return (int)hipGetLastError();
  }
  hipLaunchKernelGGL(_grouped_variable_k_mxfp8_gemm_kernel, dim3(cus), dim3(ggemm::kThreads), ggemm::kDynLdsBytes,
                     (hipStream_t)stream, (const uint8_t*)lhs, (const uint8_t*)rhs, (uint16_t*)out, lhs_scale,
                     rhs_scale, group_offs, G, OUT_M, OUT_N, stride_lhs_m, stride_rhs_m, stride_cg, stride_cm,
                     stride_cn, stride_lhs_scale, stride_rhs_scale, (void*)nullptr, (void*)nullptr, M_total);
  return (int)hipGetLastError();
}

int ggemm_vark_wgrad_mxfp8(const void* lhs, const void* rhs, void* out, const uint8_t* lhs_scale,
                           const uint8_t* rhs_scale, const int64_t* group_offs, int32_t G, int32_t OUT_M,
                           int32_t OUT_N, int32_t stride_lhs_m, int32_t stride_rhs_m, int32_t stride_cg,
                           int32_t stride_cm, int32_t stride_cn, int32_t stride_lhs_scale, int32_t stride_rhs_scale,
                           int64_t M_total, void* stream) {
  return launch_mx(0, lhs, rhs, out, lhs_scale, rhs_scale, group_offs, G, OUT_M, OUT_N, stride_lhs_m, stride_rhs_m,
                   stride_cg, stride_cm, stride_cn, stride_lhs_scale, stride_rhs_scale, M_total, stream);
}

int ggemm_vark_wgrad_mxfp8_tile(const void* lhs, const void* rhs, void* out, const uint8_t* lhs_scale,
                                const uint8_t* rhs_scale, const int64_t* group_offs, int32_t G, int32_t OUT_M,
                                int32_t OUT_N, int32_t stride_lhs_m, int32_t stride_rhs_m, int32_t stride_cg,
                                int32_t stride_cm, int32_t stride_cn, int32_t stride_lhs_scale,
                                int32_t stride_rhs_scale, int64_t M_total, int32_t tile_m, void* stream) {
  return launch_mx(tile_m, lhs, rhs, out, lhs_scale, rhs_scale, group_offs, G, OUT_M, OUT_N, stride_lhs_m,
                   stride_rhs_m, stride_cg, stride_cm, stride_cn, stride_lhs_scale, stride_rhs_scale, M_total, stream);
}

int ggemm_vark_check_offsets(const int64_t* offs, int32_t G, int64_t M_total, int32_t mx) {
  if (!offs || G <= 0) return GGEMM_E_OFFSETS;
  if (offs[0] != 0) return GGEMM_E_OFFSETS;
  for (int g = 0; g < G; ++g) {
    if (offs[g + 1] < offs[g]) return GGEMM_E_OFFSETS;
    if (mx && (offs[g] % 32)) return GGEMM_E_MX_ALIGN;
  }
  if (offs[G] > M_total) return GGEMM_E_OFFSETS;
  return GGEMM_OK;
}

int ggemm_vark_num_cus(int32_t device, int32_t* num_cus) {
  if (!num_cus) return GGEMM_E_NULL;
  int v = 0;
  hipError_t e = hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, device);
  if (e != hipSuccess) return (int)e;
  *num_cus = v;
  return GGEMM_OK;
}

const char* ggemm_vark_strerror(int32_t code) {
  switch (code) {
    case GGEMM_OK: return "success";
    case GGEMM_E_NULL: return "a required pointer is NULL";
    case GGEMM_E_SHAPE:
      return "invalid shape (G, OUT_M, OUT_N must be > 0, OUT_M/OUT_N multiples of 16, row strides below "
             "2^31/129, at most 2^30 output tiles)";
    case GGEMM_E_STRIDE: return "invalid strides (row strides >= width and multiples of 16, stride_cn == 1)";
    case GGEMM_E_ALIGN: return "misaligned pointer (LHS/RHS 16-byte, C 8-byte)";
    case GGEMM_E_OFFSETS: return "invalid group offsets (must start at 0, be non-decreasing, end <= M_total)";
    case GGEMM_E_DEVICE: return "current device is not a usable gfx950 (MI355X) GPU";
    case GGEMM_E_MX_ALIGN: return "MXFP8 groups must start on 32-token block boundaries";
    case GGEMM_E_FORMAT: return "unknown fp8 format code (A: GGEMM_FP8_E4M3 or GGEMM_FP8_E5M2)";
    default: break;
  }
  if (code > 0) return hipGetErrorString((hipError_t)code);
  return "unknown error";
}

int32_t ggemm_vark_abi_version(void) { return GGEMM_VARK_ABI_VERSION; }

int32_t ggemm_vark_bf16_kernel(int32_t OUT_M, int32_t OUT_N, int32_t stride_cm, const void* out) {
  return wide_selected(OUT_M, OUT_N, stride_cm, (int64_t)OUT_M * stride_cm, out);
}

int32_t ggemm_vark_tile_rows(int32_t G, int32_t OUT_M, int32_t OUT_N, int32_t stride_cm, int32_t out_mode,
                             int64_t M_total, int32_t num_cus) {
  const bool f32 = out_mode != GGEMM_OUT_BF16;
  const int64_t scm = stride_cm, scg = scm * OUT_M, w = f32 ? 2 : 1;
  int tile = wide_selected(OUT_M, OUT_N, w * scm, w * scg, nullptr);
  if (f32 && tile != 320) tile = 0;
  if (mid_preferred(G, OUT_M, OUT_N, scm, scg, nullptr, f32, M_total, tile, num_cus)) return ggemm::mid::kWT;
  return tile ? tile : ggemm::kTileM;
}

void ggemm_vark_launch_geometry(int32_t out_n, int32_t* block_threads, int32_t* dynamic_lds, int32_t* tile_m,
                                int32_t* tile_n, int32_t* k_step) {
  if (block_threads) *block_threads = ggemm::kThreads;
  if (dynamic_lds) *dynamic_lds = ggemm::kDynLdsBytes;
  if (tile_m) *tile_m = ggemm::kTileM;
  if (tile_n) *tile_n = (out_n > 0 && ggemm::wide_tiles(out_n, false)) ? 384 : 320;
  if (k_step) *k_step = ggemm::kKStep;
}

}  // extern "C"
