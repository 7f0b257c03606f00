// Mid-tile FP8 grouped wgrad for gfx950, library only:
//
//   C[g] = s_lhs * s_rhs * LHS[offs[g]:offs[g+1], :]^T  @  RHS[offs[g]:offs[g+1], :]
//
// Same semantics as vark_kernel.h, for the launches that its 192 x 384 and the wide kernels' 320 x 320
// tiles serve badly (mid_common.h): one 128 x 128 tile of one group per 256-thread workgroup, two
// workgroups per CU, the groups' tiles handed out largest group first. The K partition (128-token
// stages from the group's start), the MFMA (16x16x128) and the tokens in its lanes are the 192-row
// kernel's, so the results are its bits.
//
// Stages of 128 tokens, 128 LHS then 128 RHS bytes each, loaded by LDS-DMA: two 32 KiB slots, one
// barrier per stage, four waves of 64 x 64. Rows of 128 bytes: chunk c of token t at c ^ ((t >> 1) & 7),
// which puts the 16 tokens of a half-wave's transposed read on 16 distinct 16-byte bank slots.
#pragma once

#include "mid_common.h"

namespace ggemm {
namespace mid {

constexpr int kWT = 128;                                     // tile edge, and tokens per stage
constexpr int kWSide = kWT * kKStep;                         // 16 KiB of one operand
constexpr int kWSlot = 2 * kWSide, kWStages = 2;
constexpr int kWPerWave = kWSlot / 1024 / 4;                 // 8 LDS-DMA instructions, four per side

template <int kOut, bool kSwapped>
__device__ __forceinline__ void wgrad_body(const VarKArgs& a, GG_LDS uint8_t* lds) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n_tm = (a.OUT_M + kWT - 1) / kWT, n_tn = (a.OUT_N + kWT - 1) / kWT, tpg = n_tm * n_tn;

  // ---- this workgroup's tile. Up to 64 groups, one to a lane of every wave, are ranked by descending
  // length, so that the longest tiles start first; more are taken in their own order. (Ranking 256
  // groups four to a lane took 1.5 us of every workgroup, as long as a stage.)
  const int t = tile_of_block(blockIdx.x);
  if (t >= a.G * tpg) return;
  const int slot = t / tpg;
  int g = slot;
  if (a.G <= 64) {
    const int64_t lo = clamp_off(a.group_offs[min(lane, a.G)], a.m_total);
    const int64_t hi = clamp_off(a.group_offs[min(lane + 1, a.G)], a.m_total);
    const int len = hi > lo ? (int)(hi - lo) : 0;
    int rank = 0;
    for (int o = 0; o < a.G; ++o) {
      const int other = __builtin_amdgcn_readlane(len, o);
      rank += other > len || (other == len && o < lane);
    }
    g = __builtin_ctzll(__ballot(rank == slot && lane < a.G));   // ranks are a permutation of 0 .. G - 1
  }
  const int kb = (int)clamp_off(uniform64(a.group_offs[g]), a.m_total);
  const int klen = max((int)clamp_off(uniform64(a.group_offs[g + 1]), a.m_total) - kb, 0);
  const int in_g = t - slot * tpg;
  constexpr int kBandN = 8;
  const int band = in_g / (n_tm * kBandN);
  const int r = in_g - band * n_tm * kBandN;
  const int bw = min(kBandN, n_tn - band * kBandN);
  const int tm = r / bw;
  const int m0 = tm * kWT, n0 = (band * kBandN + r - tm * bw) * kWT;

  // ---- stage loads: instruction j of the wave fills token rows 8 (wave + 4 j) + lane / 8 of a side
  const int lc = (lane & 7) ^ (4 * (wave & 1) + (lane >> 4));
  const int vl = (8 * wave + (lane >> 3)) * a.stride_lhs_m + 16 * lc;
  const int vr = (8 * wave + (lane >> 3)) * a.stride_rhs_m + 16 * lc;
  const uint8_t* pl = a.lhs + (int64_t)kb * a.stride_lhs_m + m0;
  const uint8_t* pr = a.rhs + (int64_t)kb * a.stride_rhs_m + n0;
  auto issue = [&](int step, int sl) {
    const int64_t k0 = (int64_t)step * kKStep;
    const int valid = (int)min((int64_t)kKStep, klen - k0);
    // num_records ends with the last valid token's row: tokens past the group read as zero
    const v4i rl = make_rsrc(pl + k0 * a.stride_lhs_m, valid * a.stride_lhs_m - m0);
    const v4i rr = make_rsrc(pr + k0 * a.stride_rhs_m, valid * a.stride_rhs_m - n0);
    const uint32_t base = lds_u32(lds) + sl * kWSlot + 1024 * wave;
#pragma unroll
    for (int j = 0; j < kWPerWave / 2; ++j) dma16(rl, base + 4096 * j, vl + 32 * j * a.stride_lhs_m);
#pragma unroll
    for (int j = 0; j < kWPerWave / 2; ++j) dma16(rr, base + kWSide + 4096 * j, vr + 32 * j * a.stride_rhs_m);
  };

  // ---- operand reads as in vark_kernel.h (read_operand), on 128-byte rows
  const int wm = wave & 1, wn = wave >> 1, q = lane >> 4, s16 = lane & 15;
  const int rbase = 32 * (q >> 1) + 8 * (q & 1) + (s16 >> 1), swz = (rbase >> 1) & 7;
  int off_m[4], off_n[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    off_m[i] = rbase * kWT + 16 * ((4 * wm + i) ^ swz) + 8 * (s16 & 1);
    off_n[i] = kWSide + rbase * kWT + 16 * ((4 * wn + i) ^ swz) + 8 * (s16 & 1);
  }

  v4f acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

  const int nsteps = (klen + kKStep - 1) / kKStep;
  if constexpr (kOut == kOutF32Acc)
    if (nsteps == 0) return;                                 // C += 0: reading and writing it took 199 us for
                                                             // 16 groups of 2880 x 2880 and two tokens, not 42
  if (nsteps > 0) issue(0, 0);
  int cur = 0;
  for (int s = 0; s < nsteps; ++s) {
    wait_vmcnt<0>();                                         // stage s has landed for this wave
    lds_barrier();                                           // ... and for all; stage s - 1's slot is free
    if (s + 1 < nsteps) issue(s + 1, cur ^ 1);
    const GG_LDS uint8_t* sb = lds + cur * kWSlot;
    v8i bn[4], am[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) bn[j] = read_operand<kWT>(sb + off_n[j]);
#pragma unroll
    for (int i = 0; i < 4; ++i) am[i] = read_operand<kWT>(sb + off_m[i]);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = mfma<false, 0, 0, kSwapped>(bn[j], am[i], acc[i][j], 0, 0);
    cur ^= 1;
  }

  // ---- epilogue, through the slot that the next stage would have taken (cur): every wave has passed
  // the last stage's barrier, so none reads it any more
  // (an empty group's C is zero whatever the scales are: a NaN among them would turn 0 * alpha to NaN)
  const float alpha = nsteps > 0 ? *(const float*)a.lhs_scale * *(const float*)a.rhs_scale : 0.f;
  const int64_t c0 = (int64_t)g * a.stride_cg + (int64_t)(m0 + 64 * wm) * a.stride_cm + n0 + 64 * wn;
  const int rows = a.OUT_M - m0 - 64 * wm, cols = a.OUT_N - n0 - 64 * wn;
  GG_LDS uint8_t* reg = lds + cur * kWSlot + wave * (kWSlot / 4);
  if constexpr (kOut == kOutBF16) {
    store_bf16<4>(acc, alpha, reg, static_cast<uint16_t*>(a.out) + c0, a.stride_cm, rows, cols, lane);
  } else {
    store_f32<kOut == kOutF32Acc>(acc, alpha, reg, static_cast<float*>(a.out) + c0, a.stride_cm, rows, cols, lane);
  }
}

}  // namespace mid
}  // namespace ggemm

#define GGEMM_DEFINE_MID_WGRAD_KERNEL(NAME, CT, OUT, SWAPPED)                                            \
  extern "C" __global__ __launch_bounds__(ggemm::mid::kNT, 2) void NAME(GGEMM_VARK_TW_PARAMS(CT),        \
                                                                        int64_t m_total) {               \
    __shared__ __attribute__((aligned(1024))) uint8_t ggemm_mid_lds[ggemm::mid::kWStages * ggemm::mid::kWSlot]; \
    ggemm::VarKArgs a{lhs, rhs, out, lhs_scale, rhs_scale, group_offs, G, OUT_M, OUT_N,                  \
                      stride_lhs_m, stride_rhs_m, stride_cg, stride_cm, stride_cn, 0, 0, m_total};       \
    (void)global_scratch; (void)profile_scratch;                                                        \
    if (G > 0 && G <= ggemm::mid::kMaxGroups)                                                            \
      ggemm::mid::wgrad_body<OUT, SWAPPED>(a, (GG_LDS uint8_t*)ggemm_mid_lds);                            \
  }
