// Wide-tile persistent grouped FP8 GEMM (forward and data-gradient sites) for gfx950, library only:
//
//   C[r, :] = s_a * s_b * A[r, :] @ B[g]^T      for every row r of group g: offs[g] <= r < offs[g+1]
//
// Same semantics, operands and schedule as the 512-thread kernel (persistent_kernel.h), outside the
// reference's launch contract: one 256-thread workgroup per CU, one wave per SIMD, so a wave owns
// 512 registers and the output tile grows to 256 rows x 320 columns (128 x 160 per wave, 320 fp32
// accumulators: 256 in AGPRs, 64 in VGPRs). Per 128-byte K stage a CU asks for 576 row segments
// for 21.0 MFLOP (the 512-thread kernel: 576 for 18.9 MFLOP at 192 x 384) and every wave reads 36
// KiB of LDS for 40 MFMAs of 32x32x64, 5.2 MFLOP (the 512-thread kernel: 24 KiB for 36 of
// 16x16x128, 2.4 MFLOP, i.e. 1.5 times the LDS bytes per FLOP).
//
// The HIP code here runs the schedule (group tables, XCD slices, tile_of with 256-row tiles) and
// the per-lane set-up; each tile is one inline assembly statement generated by gen_vark_wide.py
// (the K-major configurations): the compiler cannot hold 320 accumulators per wave in one register
// class. The statement's operands carry the operand pipeline between tiles (slot of the next
// tile's first stage, whether it is in flight, the per-wave model of outstanding vector-memory
// operations).
//
// Requirements (the library routes other shapes to the 512-thread kernel): N % 320 == 0, K % 64 ==
// 0 (a stage is 128 bytes; K % 128 == 64 makes each tile's last stage a half stage), strides and
// bases as for the 512-thread kernel.
//
// LDS (static, 160 KiB): two 72 KiB stage slots (256 A rows then 320 B rows of 128 bytes; logical
// chunk c of row r at physical chunk c ^ (r & 7) ^ ((r >> 3) & 1), the 512-thread kernel's
// swizzle), then the group tables (tile prefix sums, then offsets, 8 KiB each). The epilogue stages
// C in the freed slot as the wgrad's wide kernels do (32-row x 64-column passes, whole 128-byte
// lines; the line the two wave halves share goes through a joint pass).
#pragma once

#include "persistent_kernel.h"
#include "vark_wide.h"

namespace ggemm {
namespace pw {

constexpr int kNT = 256;                              // threads: one wave per SIMD
constexpr int kTM = 256, kTN = 320;                   // tile rows (A rows) x columns (B rows)
constexpr int kKS = 128;                              // K bytes per stage
constexpr int kSlot = (kTM + kTN) * kKS, kSlots = 2;  // 72 KiB
constexpr int kPreOff = kSlots * kSlot;
constexpr int kOffsOff = kPreOff + 4 * (nt::kMaxGroups + 1);
constexpr int kLdsBytes = kOffsOff + 4 * (nt::kMaxGroups + 1);
constexpr int kNL = kTM * kKS / 4096, kNR = kTN * kKS / 4096;   // LDS-DMA instructions per wave and stage
static_assert(kLdsBytes <= 160 * 1024, "gfx950 LDS");
static_assert(GGEMM_WIDE_NOPERANDS_pk256x320_e4m3 == 60 && GGEMM_WIDE_NOPERANDS_pk256x320_e5m2 == 60,
              "operand list of vark_wide_asm.inc");
static_assert(8 * kNT <= kSlot, "the group scan's scratch fits slot 1");

// Shapes the wide kernel takes (the host also checks strides and bases as for every launch).
__host__ __device__ constexpr bool fits(int N, int K) { return N % kTN == 0 && K % 64 == 0 && K > 0; }

}  // namespace pw

template <bool kAE5M2>
__device__ __forceinline__ void persistent_wide_body(const nt::Args& a, GG_LDS uint8_t* lds) {
  using namespace pw;
  GG_LDS int* s_pre = (GG_LDS int*)(lds + kPreOff);
  GG_LDS int* s_offs = (GG_LDS int*)(lds + kOffsOff);
  GG_LDS int64_t* s_scan = (GG_LDS int64_t*)(lds + kSlot);   // slot 1: no stage is issued before the scan ends

  const int num_wg = nt::workgroups(a);
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  const int G = a.G;
  const int n_tn = a.N / kTN;
  if (!nt::group_tables<kNT, kTM>(a, n_tn, s_pre, s_offs, s_scan)) return;
  const nt::Slices sl = nt::xcd_slices(s_pre[G], num_wg);
  const uint32_t lds_base = lds_u32(lds);

  // LDS-DMA: instruction j of this wave fills slot bytes [1024 (wave + 4 j), +1024), operand rows
  // 8 (wave + 4 j) + l / 8 (A rows for j < kNL, then B rows), lane l writing physical chunk l % 8.
  // The row's swizzle is (l / 8) ^ (wave & 1) in every instruction, so a lane loads one logical
  // chunk throughout.
  const int lc = (lane & 7) ^ (lane >> 3) ^ (wave & 1);
  int voffl[kNL], voffr[kNR];
#pragma unroll
  for (int j = 0; j < kNL; ++j) voffl[j] = (8 * (wave + 4 * j) + (lane >> 3)) * a.stride_am + 16 * lc;
#pragma unroll
  for (int j = 0; j < kNR; ++j) voffr[j] = (8 * (wave + 4 * j) + (lane >> 3)) * a.stride_bn + 16 * lc;

  // Operand reads (32x32x64): lane l takes row l % 32 of a 32-row block, K bytes 32 h .. 32 h + 31
  // of the K-half (h = l / 32): logical chunks 4 kh + 2 h (lo) and 4 kh + 2 h + 1 (hi). Block rows
  // start at multiples of 16, so the swizzle depends on l % 32 alone; block b is 4096 b further.
  const int rr = lane & 31, hh = lane >> 5, sw = nt::swz(rr);
  const int arow = (int)lds_base + (128 * wm + rr) * kKS;
  const int brow = (int)lds_base + kTM * kKS + (160 * wn + rr) * kKS;
  int rd[2][2][2];   // [side][kh][lo / hi]
#pragma unroll
  for (int kh = 0; kh < 2; ++kh)
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const int chunk = (4 * kh + 2 * hh + x) ^ sw;
      rd[0][kh][x] = arow + 16 * chunk;
      rd[1][kh][x] = brow + 16 * chunk;
    }

  // Epilogue: as in the wgrad's wide kernels (vark_wide.h): staging writes at row l % 32, half
  // l / 32; read-back k gives lane l row 8 k + l / 8, chunk l % 8.
  const int rl = lane & 31, hl = lane >> 5;
  const int ew_base = rl * 128 + 8 * hl, ew_s = (rl >> 1) & 7;
  const int er = lane >> 3, ec = lane & 7, es = (er >> 1) & 7;
  const int rb_even = er * 128 + 16 * (ec ^ es);
  const int rb_odd = (8 + er) * 128 + 16 * (ec ^ (es ^ 4));
  const int gb = (er * a.stride_cm + 8 * ec) * 2;
  const uint32_t sw_epi = (uint32_t)(128 * wm * a.stride_cm + 160 * wn) * 2u;
  const uint32_t alpha_bits = __builtin_amdgcn_readfirstlane(__float_as_uint(*a.a_scale * *a.b_scale));
  const uint32_t cm2 = (uint32_t)a.stride_cm * 2u;
  const uint32_t w1k = (uint32_t)wave * 1024u;
  const uint32_t klen = (uint32_t)a.K;
  const int nsteps = (a.K + kKS - 1) / kKS;

  uint32_t c0 = 0, nis = 0, vmt = 0, q0 = 0, q1 = 0, q2 = 0, np = 0;
  int t = sl.t_begin;
  if (t >= sl.t_end) return;
  nt::Tile T = nt::tile_of<kTM, kTN>(s_pre, s_offs, G, n_tn, t);
  for (;;) {
    const int t_next = t + sl.t_step;
    const bool has_next = t_next < sl.t_end;
    nt::Tile N = T;
    if (has_next) N = nt::tile_of<kTM, kTN>(s_pre, s_offs, G, n_tn, t_next);
    // stage bases at K = 0; num_records without the stage's K bytes: (valid rows - 1) x stride
    const uint8_t* blt = a.a + (int64_t)(T.row_base + T.m0) * a.stride_am;
    const uint8_t* brt = a.b + (int64_t)T.g * a.stride_bg + (int64_t)T.n0 * a.stride_bn;
    const uint8_t* bln = a.a + (int64_t)(N.row_base + N.m0) * a.stride_am;
    const uint8_t* brn = a.b + (int64_t)N.g * a.stride_bg + (int64_t)N.n0 * a.stride_bn;
    const uint32_t rat = (uint32_t)((T.rows - 1) * a.stride_am), rbt = (uint32_t)((kTN - 1) * a.stride_bn);
    const uint32_t ran = (uint32_t)((N.rows - 1) * a.stride_am);
    const uint32_t kln = has_next ? klen : 0u;
    const uint16_t* ct = a.c + (int64_t)(T.row_base + T.m0) * a.stride_cm + T.n0;
    const uint32_t crec = (uint32_t)(((int64_t)T.rows * a.stride_cm - T.n0) * 2);
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
#define GGEMM_PW_OPERANDS                                                                                       \
  : "+s"(c0), "+s"(nis), "+s"(vmt), "+s"(q0), "+s"(q1), "+s"(q2), "+s"(np)                                        \
  : "s"(lds_base), "s"(w1k), "s"(lo32(blt)), "s"(hi32(blt)), "s"(lo32(brt)), "s"(hi32(brt)), "s"(klen), "s"(rat), \
    "s"(rbt), "s"(lo32(bln)), "s"(hi32(bln)), "s"(lo32(brn)), "s"(hi32(brn)), "s"(kln), "s"(ran), "s"(rbt),        \
    "s"(lo32(ct)), "s"(hi32(ct)), "s"(crec), "s"(cm2), "s"(alpha_bits), "s"(sw_epi), "v"(voffl[0]),             \
    "v"(voffl[1]), "v"(voffl[2]), "v"(voffl[3]), "v"(voffl[4]), "v"(voffl[5]), "v"(voffl[6]), "v"(voffl[7]),     \
    "v"(voffr[0]), "v"(voffr[1]), "v"(voffr[2]), "v"(voffr[3]), "v"(voffr[4]), "v"(voffr[5]), "v"(voffr[6]),     \
    "v"(voffr[7]), "v"(voffr[8]), "v"(voffr[9]), "v"(rd[0][0][0]), "v"(rd[0][0][1]), "v"(rd[0][1][0]),           \
    "v"(rd[0][1][1]), "v"(rd[1][0][0]), "v"(rd[1][0][1]), "v"(rd[1][1][0]), "v"(rd[1][1][1]), "v"(ew_base),      \
    "v"(ew_s), "v"(rb_even), "v"(rb_odd), "v"(gb)
    if constexpr (kAE5M2)
      asm volatile(GGEMM_WIDE_ASM_pk256x320_e5m2 GGEMM_PW_OPERANDS : GGEMM_WIDE_CLOBBERS_pk256x320_e5m2);
    else
      asm volatile(GGEMM_WIDE_ASM_pk256x320_e4m3 GGEMM_PW_OPERANDS : GGEMM_WIDE_CLOBBERS_pk256x320_e4m3);
#undef GGEMM_PW_OPERANDS
#pragma clang diagnostic pop
    c0 = (c0 + (uint32_t)nsteps) & 1u;
    if (!has_next) break;
    t = t_next;
    T = N;
  }
}

}  // namespace ggemm

// Library kernel: the 512-thread kernel's 16 arguments plus M_total and zero_tail, 256 threads, 160 KiB of static
// LDS and no dynamic LDS.
#define GGEMM_DEFINE_PERSISTENT_WIDE_KERNEL(NAME, AE5M2)                                                 \
  extern "C" __global__ __launch_bounds__(ggemm::pw::kNT) __attribute__((amdgpu_waves_per_eu(1, 1)))     \
  void NAME(GGEMM_PERSISTENT_PARAMS, int64_t m_total, int zero_tail) {                                   \
    __shared__ __attribute__((aligned(1024))) uint8_t ggemm_pw_lds[ggemm::pw::kLdsBytes];                \
    ggemm::nt::Args args{a, b, c, a_scale, b_scale, group_offs, G, N, K,                                 \
                         stride_am, stride_bg, stride_bn, stride_cm, stride_cn, m_total, zero_tail,      \
                         (int)gridDim.x};                                                               \
    (void)global_scratch; (void)profile_scratch;                                                        \
    if (G > 0 && G <= ggemm::nt::kMaxGroups && ggemm::pw::fits(N, K))                                   \
      ggemm::persistent_wide_body<AE5M2>(ggemm::nt::without_tail(args), (GG_LDS uint8_t*)ggemm_pw_lds);  \
    ggemm::nt::clear_tail_rows(args);                                                                   \
  }
