// Wide-tile FP8 grouped wgrad for gfx950 (library only; bf16 C, and at 320 x 320 also fp32 C, fp32
// C += and MXFP8 block scales):
//
//   C[g] = s_lhs * s_rhs * LHS[offs[g]:offs[g+1], :]^T  @  RHS[offs[g]:offs[g+1], :]
//
// Same semantics and schedule as the 192 x 384 kernel (vark_kernel.h), outside the reference's
// 512-thread launch contract: one 256-thread workgroup per CU, one wave per SIMD, so a wave owns
// 512 registers and the output tile grows to 256 x 384 or 320 x 320 (OUT_M x OUT_N). Per 64-token
// stage a CU then asks the L1 -> L2 stream for 64 x 5 (256 x 384) or 64 x 6 (320 x 320) line
// requests for 12.6 / 13.1 MFLOP, against 64 x 5 for 9.4 MFLOP at 192 x 384, and reads ~35 % fewer
// LDS bytes per FLOP. 320 x 320 divides 2880 and 5760 exactly (no partial tiles at the MoE shapes);
// 256 x 384 leaves a quarter-height last M-tile at OUT_M = 2880.
//
// The HIP code here runs the schedule (make_sched / tile_at with 64-token stages) and the
// per-lane address set-up; each tile is computed by one inline assembly statement generated by
// gen_vark_wide.py (vark_wide_asm.inc): the compiler cannot allocate 384-400 accumulators per wave
// (it puts every MFMA of a kernel in one accumulator register class, at most 256 AGPRs), so the
// assembly keeps 256 in AGPRs and the rest in VGPRs by hand. The statement's operands carry the
// operand pipeline from one tile to the next (slot of the next tile's first stage, how many of its
// stages are already in flight, the per-wave model of outstanding vector-memory operations).
//
// LDS (static, 136 KiB): three 40 KiB stage slots (64 rows of the tile's LHS bytes, then 64 rows
// of its RHS bytes), then the schedule tables. Chunk swizzles (16-byte chunk c of token row t
// stored at c ^ swz(t)): 256-byte rows swz = (t & 7) << 1, 384-byte rows ((t >> 1) & 3) << 1,
// 320-byte rows ((t >> 2) & 1) << 1 -- the 8 tokens x 2 chunks x 2 halves of a 32-lane half of a
// transposed read land in 32 distinct 8-byte bank pairs, and tokens t + 8, t + 32, t + 40 share t's
// swizzle. Epilogue staging rows (128 B, 64 bf16): chunk c of row r at c ^ ((r >> 1) & 7). The
// fp32 epilogues stage one 32 x 32 block per pass (128-byte rows, chunk c of row r at
// c ^ (((r >> 1) & 3) << 1)); accumulating, the old C of the next two passes is in flight while a
// pass waits for its own.
#pragma once

#include "vark_kernel.h"
#include "vark_wide_asm.inc"

namespace ggemm {
namespace wide {

constexpr int kNT = 256;                          // threads: one wave per SIMD
constexpr int kKS = 64;                           // tokens per stage
constexpr int kSlot = 40960, kSlots = 3;
constexpr int kMiscOff = kSlots * kSlot;
constexpr int kLdsBytes = kMiscOff + kMiscBytes;  // 136 KiB
// MXFP8: three 2.5 KiB scale slots right after the stage slots (the one that goes with stage slot
// byte offset o starts at kScaleOff + o / 16): a stage's e8m0 rows, 320 bytes each from the tile's
// column, LHS token blocks 0 and 1 at +0 and +320, RHS blocks at +1024 and +1344. LDS-DMA
// destinations stay below 128 KiB, where the operand slots have always been (the DMA's M0 offset is
// not exercised above it), so the schedule tables, read with plain LDS reads, move above them.
constexpr int kScaleOff = kMiscOff, kScaleSlot = kSlot / 16;
constexpr int kMiscOffMX = 128 * 1024;
constexpr int kLdsBytesMX = kMiscOffMX + kMiscBytes;   // 144 KiB
constexpr int kEpiW = 3;                          // a tile's epilogue, in 64-token stages
static_assert(kLdsBytesMX <= 160 * 1024, "gfx950 LDS");
static_assert(kScaleOff == 122880 && kScaleSlot >= 2048 && kScaleOff + kSlots * kScaleSlot <= kMiscOffMX,
              "scale slots of vark_wide_asm.inc, below 128 KiB");
static_assert(GGEMM_WIDE_NOPERANDS_256x384 == 56 && GGEMM_WIDE_NOPERANDS_320x320 == 50 &&
                  GGEMM_WIDE_NOPERANDS_320x320_f32 == 49 && GGEMM_WIDE_NOPERANDS_320x320_f32acc == 49 &&
                  GGEMM_WIDE_NOPERANDS_320x320_mx == 54,
              "operand lists of vark_wide_asm.inc");

template <int kPitch>
__device__ __forceinline__ int swz(int t) {
  static_assert(kPitch == 256 || kPitch == 320 || kPitch == 384, "row pitch");
  if constexpr (kPitch == 256) return (t & 7) << 1;
  else if constexpr (kPitch == 384) return ((t >> 1) & 3) << 1;
  else return ((t >> 2) & 1) << 1;
}

}  // namespace wide

__device__ __forceinline__ uint32_t lo32(const void* p) { return (uint32_t)reinterpret_cast<uintptr_t>(p); }
__device__ __forceinline__ uint32_t hi32(const void* p) {
  return (uint32_t)(reinterpret_cast<uintptr_t>(p) >> 32);
}

// The asm statement of one tile (shape TM x TN); its 31 scalar operands come first, then the
// per-lane ones in the order gen_vark_wide.py lists them.
#define GGEMM_WIDE_SCALAR_OPERANDS                                                                      \
  : "+s"(c0), "+s"(nis), "+s"(vmt), "+s"(q0), "+s"(q1), "+s"(q2), "+s"(np)                                  \
  : "s"(lds_base), "s"(w1k), "s"(lo32(blt)), "s"(hi32(blt)), "s"(lo32(brt)), "s"(hi32(brt)), "s"(klt),       \
    "s"(T.m0), "s"(T.n0), "s"(lo32(bln)), "s"(hi32(bln)), "s"(lo32(brn)), "s"(hi32(brn)), "s"(kln), "s"(N.m0), \
    "s"(N.n0), "s"(lo32(ct)), "s"(hi32(ct)), "s"(crec), "s"(stride_l), "s"(stride_r), "s"(cm2),             \
    "s"(alpha_bits), "s"(sw_epi)

// OUT: kOutBF16 (bf16 C), kOutF32 (fp32 C) or kOutF32Acc (fp32 C += result); the fp32 modes are
// built for 320 x 320 tiles. MX: e8m0 block scales (one per 32 tokens and column) applied by the
// scaled MFMA, bf16 C, 320 x 320 tiles. SWAPPED: e5m2 LHS and e4m3 RHS (dW[g] = dy_g^T x_g in the
// weight's own [N, K] orientation), bf16 C.
template <int TM, int TN, int OUT = kOutBF16, bool MX = false, bool SWAPPED = false>
__device__ __forceinline__ void vark_wide_body(const VarKArgs& a, GG_LDS uint8_t* lds) {
  using namespace wide;
  static_assert(OUT == kOutBF16 || (TM == 320 && TN == 320), "fp32 epilogues of the 320 x 320 tile");
  static_assert(!MX || (OUT == kOutBF16 && TM == 320 && TN == 320), "MX: bf16 C, 320 x 320 tiles");
  static_assert(!SWAPPED || (OUT == kOutBF16 && !MX), "swapped formats: bf16 C");
  using CT = std::conditional_t<OUT == kOutBF16, uint16_t, float>;
  constexpr int kCB = sizeof(CT);                 // bytes per C element
  constexpr int BM = TM / 64, BN = TN / 64;       // 32-wide blocks per wave, 2 x 2 waves
  constexpr int kRhsOff = kKS * TM;
  constexpr int NL = kKS * TM / 4096, NR = kKS * TN / 4096;   // LDS-DMA instructions per wave
  static_assert(kKS * (TM + TN) == kSlot, "slot layout");
  GG_LDS uint8_t* misc = lds + (MX ? kMiscOffMX : kMiscOff);
  GG_LDS int* s_order = (GG_LDS int*)misc;
  GG_LDS int* s_kb = (GG_LDS int*)(misc + kKbOffset);
  const Sched S = make_sched<TN, kKS, kEpiW, TM, kNT, OUT == kOutBF16 ? 0 : OUT == kOutF32 ? 16 : 32>(
      a, s_order, s_kb, (GG_LDS int*)(misc + kFlagOffset), (GG_LDS int64_t*)(misc + kBoundOffset));
  if (!S.valid) {
    poison_c<OUT>(a);
    return;
  }
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  const uint32_t lds_base = lds_u32(lds);

  // Transposed operand reads (32x32x64 layout): lane l reads token tb0 + {0, 8, 32, 40}, 8 bytes
  // at half hb of chunk 2 b + cb of its block b (the hardware returns column l % 32 of 8 tokens).
  const int g16 = lane >> 4, t16 = lane & 15, cb = g16 & 1, hh = g16 >> 1;
  const int tb0 = 16 * hh + (t16 >> 1), hb = t16 & 1;
  int amb[BM], bnb[BN];
#pragma unroll
  for (int i = 0; i < BM; ++i)
    amb[i] = (int)lds_base + tb0 * TM + 16 * ((2 * BM * wm + 2 * i + cb) ^ swz<TM>(tb0)) + 8 * hb;
#pragma unroll
  for (int j = 0; j < BN; ++j)
    bnb[j] = (int)lds_base + kRhsOff + tb0 * TN + 16 * ((2 * BN * wn + 2 * j + cb) ^ swz<TN>(tb0)) + 8 * hb;

  // LDS-DMA: instruction j of this wave fills operand bytes [1024 (wave + 4 j), +1024): chunk
  // q = 64 (wave + 4 j) + l, token row q / (pitch / 16), physical chunk q % (pitch / 16), which
  // holds logical chunk (q % (pitch / 16)) ^ swz(row).
  int voffl[NL], voffr[NR];
#pragma unroll
  for (int j = 0; j < NL; ++j) {
    const int q = 64 * (wave + 4 * j) + lane, row = q / (TM / 16), pc = q - (TM / 16) * row;
    voffl[j] = row * a.stride_lhs_m + 16 * (pc ^ swz<TM>(row));
  }
#pragma unroll
  for (int j = 0; j < NR; ++j) {
    const int q = 64 * (wave + 4 * j) + lane, row = q / (TN / 16), pc = q - (TN / 16) * row;
    voffr[j] = row * a.stride_rhs_m + 16 * (pc ^ swz<TN>(row));
  }

  // Epilogue: a pass stages 32 rows x 64 columns (one m-block, two n-blocks) in a private 4 KiB
  // region; lane (r = l % 32, h = l / 32) writes 8-byte halves of chunks 4 jj + g; read-back k
  // (0..3) gives lane l row 8 k + l / 8, chunk l % 8 -- 8 lanes cover one whole 128-byte row. With
  // an odd BN the line the two wave halves share is staged by both in a common region (the left
  // half's last block in chunks 0-3, the right half's first in 4-7) and read back the same way.
  const int rl = lane & 31, hl = lane >> 5;
  const int ew_base = rl * 128 + 8 * hl, ew_s = (rl >> 1) & 7;
  const int rr = lane >> 3, rc = lane & 7, rs = (rr >> 1) & 7;
  const int rb_even = rr * 128 + 16 * (rc ^ rs);                 // rows rr, 16 + rr (+2048)
  const int rb_odd = (8 + rr) * 128 + 16 * (rc ^ (rs ^ 4));      // rows 8 + rr, 24 + rr
  const int gb = (rr * a.stride_cm + 8 * rc) * 2;
  // fp32 epilogue: one 32 x 32 block per pass in a private 4 KiB region; lane (r = l % 32,
  // h = l / 32) writes chunk 2 g + h of row r (chunk c stored at c ^ (((r >> 1) & 3) << 1)), i.e.
  // at fw_base + 32 (g ^ fw_s); read-back k gives lane l row 8 k + l / 8, chunk l % 8.
  const int fw_base = rl * 128 + 16 * hl, fw_s = (rl >> 1) & 3;
  const int frb = rr * 128 + 16 * (rc ^ (((rr >> 1) & 3) << 1));
  const int fgb = (rr * a.stride_cm + 4 * rc) * 4;
  const uint32_t sw_epi = (uint32_t)(32 * BM * wm * a.stride_cm + 32 * BN * wn) * (uint32_t)kCB;
  // MX: the block scales are in the products; the epilogue's factor is 1
  const float alpha = MX ? 1.0f : *(const float*)a.lhs_scale * *(const float*)a.rhs_scale;
  const uint32_t alpha_bits = __builtin_amdgcn_readfirstlane(__float_as_uint(alpha));

  // MX: waves 0, 1 load the stage's two LHS e8m0 rows, waves 2, 3 the RHS rows (both waves of a
  // side write the same bytes), lanes 0-39 one 16-byte chunk each (row l / 20, chunk l % 20; the
  // other lanes' offsets are out of range) at scw + 16 l; lane l reads its scale of block b from
  // row l / 32 at column 160 wm + 32 b + l % 32 (LHS) or 160 wn + 32 b + l % 32 (RHS, scrd further)
  const int sside = wave >> 1;
  const uint8_t* scale_base = static_cast<const uint8_t*>(sside ? a.rhs_scale : a.lhs_scale);
  const uint32_t stride_sc = (uint32_t)(sside ? a.stride_rhs_scale : a.stride_lhs_scale);
  const int vsc = lane < 40 ? (lane / 20) * (int)stride_sc + 16 * (lane % 20) : (int)0x80000000;
  const int vscb = (int)lds_base + kScaleOff + 320 * (lane >> 5) + 160 * wm + (lane & 31);
  const uint32_t scrd = (uint32_t)(1024 + 160 * (wn - wm));
  const uint32_t scw = lds_base + (uint32_t)kScaleOff + 1024u * (uint32_t)sside;

  const uint8_t* lhs = static_cast<const uint8_t*>(a.lhs);
  const uint8_t* rhs = static_cast<const uint8_t*>(a.rhs);
  CT* out = static_cast<CT*>(a.out);
  const uint32_t stride_l = (uint32_t)a.stride_lhs_m, stride_r = (uint32_t)a.stride_rhs_m;
  const uint32_t cm2 = (uint32_t)a.stride_cm * 2u;
  const uint32_t w1k = (uint32_t)wave * 1024u;

  // pipeline state carried between tiles
  uint32_t c0 = 0, nis = 0, vmt = 0, q0 = 0, q1 = 0, q2 = 0, np = 0;
  int t = S.t_first, d = S.d0, d_alt = S.d1;
  if (!S.has(t)) return;
  Tile T = tile_at<TN, kKS, TM>(S, a, s_order, s_kb, t);
  for (;;) {
    const int t_next = t + d;
    const bool has_next = S.has(t_next);
    Tile N{};
    if (has_next) N = tile_at<TN, kKS, TM>(S, a, s_order, s_kb, t_next);
    const uint8_t* blt = lhs + T.kb * (int64_t)stride_l + T.m0;
    const uint8_t* brt = rhs + T.kb * (int64_t)stride_r + T.n0;
    const uint8_t* bln = lhs + N.kb * (int64_t)stride_l + N.m0;
    const uint8_t* brn = rhs + N.kb * (int64_t)stride_r + N.n0;
    const CT* ct = out + (int64_t)T.g * a.stride_cg + (int64_t)T.m0 * a.stride_cm + T.n0;
    const uint32_t crec = (uint32_t)(((int64_t)(a.OUT_M - T.m0) * a.stride_cm - T.n0) * kCB);
    const uint32_t klt = (uint32_t)T.klen, kln = has_next ? (uint32_t)N.klen : 0u;
    const uint8_t* sct = scale_base + (T.kb >> 5) * (int64_t)stride_sc + (sside ? T.n0 : T.m0);
    const uint8_t* scn = scale_base + (N.kb >> 5) * (int64_t)stride_sc + (sside ? N.n0 : N.m0);
    // m0 is written only by these statements' LDS-DMA set-up (as in dma16); clang warns that a
    // reserved register is on the clobber list
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
    if constexpr (TM == 256 && TN == 384) {
#define GGEMM_WIDE_OPERANDS_256x384 \
  GGEMM_WIDE_SCALAR_OPERANDS, \
    "v"(voffl[0]), "v"(voffl[1]), "v"(voffl[2]), "v"(voffl[3]), "v"(voffr[0]), "v"(voffr[1]), \
    "v"(voffr[2]), "v"(voffr[3]), "v"(voffr[4]), "v"(voffr[5]), "v"(amb[0]), "v"(amb[1]), \
    "v"(amb[2]), "v"(amb[3]), "v"(bnb[0]), "v"(bnb[1]), "v"(bnb[2]), "v"(bnb[3]), "v"(bnb[4]), \
    "v"(bnb[5]), "v"(ew_base), "v"(ew_s), "v"(rb_even), "v"(rb_odd), "v"(gb)
      if constexpr (SWAPPED)
        asm volatile(GGEMM_WIDE_ASM_256x384_swapped GGEMM_WIDE_OPERANDS_256x384 : GGEMM_WIDE_CLOBBERS_256x384_swapped);
      else
        asm volatile(GGEMM_WIDE_ASM_256x384 GGEMM_WIDE_OPERANDS_256x384 : GGEMM_WIDE_CLOBBERS_256x384);
#undef GGEMM_WIDE_OPERANDS_256x384
    } else if constexpr (MX) {
      const int amb0 = amb[0], amb1 = amb[1] - 32, bnb0 = bnb[0], bnb1 = bnb[1] - 32;
      asm volatile(GGEMM_WIDE_ASM_320x320_mx GGEMM_WIDE_SCALAR_OPERANDS,
                   "v"(voffl[0]), "v"(voffl[1]), "v"(voffl[2]), "v"(voffl[3]), "v"(voffl[4]), "v"(voffr[0]),
                   "v"(voffr[1]), "v"(voffr[2]), "v"(voffr[3]), "v"(voffr[4]), "v"(amb0), "v"(amb1), "v"(bnb0),
                   "v"(bnb1), "s"(lo32(sct)), "s"(hi32(sct)), "s"(lo32(scn)), "s"(hi32(scn)), "s"(stride_sc),
                   "s"(scrd), "s"(scw), "v"(vsc), "v"(vscb)
                   : GGEMM_WIDE_CLOBBERS_320x320_mx);
    } else if constexpr (OUT == kOutF32) {
      const int amb0 = amb[0], amb1 = amb[1] - 32, bnb0 = bnb[0], bnb1 = bnb[1] - 32;
      asm volatile(GGEMM_WIDE_ASM_320x320_f32 GGEMM_WIDE_SCALAR_OPERANDS,
                   "v"(voffl[0]), "v"(voffl[1]), "v"(voffl[2]), "v"(voffl[3]), "v"(voffl[4]), "v"(voffr[0]),
                   "v"(voffr[1]), "v"(voffr[2]), "v"(voffr[3]), "v"(voffr[4]), "v"(amb0), "v"(amb1), "v"(bnb0),
                   "v"(bnb1), "v"(fw_base), "v"(fw_s), "v"(frb), "v"(fgb)
                   : GGEMM_WIDE_CLOBBERS_320x320_f32);
    } else if constexpr (OUT == kOutF32Acc) {
      const int amb0 = amb[0], amb1 = amb[1] - 32, bnb0 = bnb[0], bnb1 = bnb[1] - 32;
      asm volatile(GGEMM_WIDE_ASM_320x320_f32acc GGEMM_WIDE_SCALAR_OPERANDS,
                   "v"(voffl[0]), "v"(voffl[1]), "v"(voffl[2]), "v"(voffl[3]), "v"(voffl[4]), "v"(voffr[0]),
                   "v"(voffr[1]), "v"(voffr[2]), "v"(voffr[3]), "v"(voffr[4]), "v"(amb0), "v"(amb1), "v"(bnb0),
                   "v"(bnb1), "v"(fw_base), "v"(fw_s), "v"(frb), "v"(fgb)
                   : GGEMM_WIDE_CLOBBERS_320x320_f32acc);
    } else {
      static_assert(TM == 320 && TN == 320, "tile shapes of vark_wide_asm.inc");
      // two read bases per side: block b reads at base[b & 1] + 32 b (the one-bit swizzle of
      // 320-byte rows moves a chunk pair by +-32 bytes with the parity of its index)
      const int amb0 = amb[0], amb1 = amb[1] - 32, bnb0 = bnb[0], bnb1 = bnb[1] - 32;
#define GGEMM_WIDE_OPERANDS_320x320 \
  GGEMM_WIDE_SCALAR_OPERANDS, \
    "v"(voffl[0]), "v"(voffl[1]), "v"(voffl[2]), "v"(voffl[3]), "v"(voffl[4]), "v"(voffr[0]), \
    "v"(voffr[1]), "v"(voffr[2]), "v"(voffr[3]), "v"(voffr[4]), "v"(amb0), "v"(amb1), "v"(bnb0), \
    "v"(bnb1), "v"(ew_base), "v"(ew_s), "v"(rb_even), "v"(rb_odd), "v"(gb)
      if constexpr (SWAPPED)
        asm volatile(GGEMM_WIDE_ASM_320x320_swapped GGEMM_WIDE_OPERANDS_320x320 : GGEMM_WIDE_CLOBBERS_320x320_swapped);
      else
        asm volatile(GGEMM_WIDE_ASM_320x320 GGEMM_WIDE_OPERANDS_320x320 : GGEMM_WIDE_CLOBBERS_320x320);
#undef GGEMM_WIDE_OPERANDS_320x320
    }
#pragma clang diagnostic pop
    c0 = (c0 + (uint32_t)T.nsteps) % 3u;
    if (!has_next) break;
    t = t_next;
    const int d_was = d;
    d = d_alt;
    d_alt = d_was;
    T = N;
  }
}

}  // namespace ggemm

// Library kernels: the tensorwise kernel's 16 arguments plus M_total, 256 threads, 136 KiB of
// static LDS and no dynamic LDS. CT / OUT: bf16 C (kOutBF16) or fp32 C (kOutF32, kOutF32Acc);
// SWAPPED: e5m2 LHS, e4m3 RHS.
#define GGEMM_DEFINE_WIDE_KERNEL(NAME, TM, TN, CT, OUT, SWAPPED)                                         \
  extern "C" __global__ __launch_bounds__(ggemm::wide::kNT) __attribute__((amdgpu_waves_per_eu(1, 1)))   \
  void NAME(GGEMM_VARK_TW_PARAMS(CT), int64_t m_total) {                                                \
    __shared__ __attribute__((aligned(1024))) uint8_t ggemm_wide_lds[ggemm::wide::kLdsBytes];            \
    ggemm::VarKArgs a{lhs, rhs, out, lhs_scale, rhs_scale, group_offs, G, OUT_M, OUT_N,                  \
                      stride_lhs_m, stride_rhs_m, stride_cg, stride_cm, stride_cn, 0, 0, m_total,        \
                      (int)gridDim.x};                                                                  \
    (void)global_scratch; (void)profile_scratch;                                                        \
    if (G > 0) ggemm::vark_wide_body<TM, TN, OUT, false, SWAPPED>(a, (GG_LDS uint8_t*)ggemm_wide_lds);   \
  }

// MXFP8 library kernel, 320 x 320 tiles: the MX kernel's arguments without the scratch pointers,
// 144 KiB of static LDS.
#define GGEMM_DEFINE_WIDE_MX_KERNEL(NAME)                                                               \
  extern "C" __global__ __launch_bounds__(ggemm::wide::kNT) __attribute__((amdgpu_waves_per_eu(1, 1)))   \
  void NAME(const uint8_t* lhs, const uint8_t* rhs, uint16_t* out, const uint8_t* lhs_scale,             \
            const uint8_t* rhs_scale, const int64_t* group_offs, int G, int OUT_M, int OUT_N,             \
            int stride_lhs_m, int stride_rhs_m, int stride_cg, int stride_cm, int stride_cn,               \
            int stride_lhs_scale, int stride_rhs_scale, int64_t m_total) {                                \
    __shared__ __attribute__((aligned(1024))) uint8_t ggemm_wide_lds[ggemm::wide::kLdsBytesMX];          \
    ggemm::VarKArgs a{lhs, rhs, out, lhs_scale, rhs_scale, group_offs, G, OUT_M, OUT_N,                  \
                      stride_lhs_m, stride_rhs_m, stride_cg, stride_cm, stride_cn,                      \
                      stride_lhs_scale, stride_rhs_scale, m_total, (int)gridDim.x};                     \
    if (G > 0) ggemm::vark_wide_body<320, 320, ggemm::kOutBF16, true>(a, (GG_LDS uint8_t*)ggemm_wide_lds); \
  }
