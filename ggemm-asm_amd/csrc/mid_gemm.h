// Mid-tile grouped FP8 GEMM (forward and data-gradient sites) for gfx950, library only:
//
//   C[r, :] = s_a * s_b * A[r, :] @ B[g]^T      for every row r of group g: offs[g] <= r < offs[g+1]
//
// Same semantics and operands as persistent_kernel.h, for the launches that its 192 x 384 and the
// wide kernel's 256 x 320 tiles serve badly (mid_common.h): one tile of BM = 64 or 128 rows of one
// group x 128 columns per 256-thread workgroup, two workgroups per CU. A decoding step's few rows per
// expert are bound by reading the weights once: at BM = 64 a stage is 16 KiB of B beside 8 KiB of A
// and two stages per workgroup are in flight, 96 KiB per CU.
//
// Stages of 128 K bytes, BM rows of A then 128 rows of B, loaded by LDS-DMA with the 512-thread
// kernel's swizzle (chunk c of row r at c ^ nt::swz(r)); kStages slots, one barrier per stage. The
// MFMA is that kernel's 16x16x128 with the same K bytes in the same lanes, so the results are its
// bits. Waves: 1 x 4 of 64 x 32 (BM = 64) or 2 x 2 of 64 x 64 (BM = 128).
#pragma once

#include "mid_common.h"
#include "persistent_kernel.h"

namespace ggemm {
namespace mid {

template <int kBM>
struct GemmCfg {
  static_assert(kBM == 64 || kBM == 128, "tile heights");
  static constexpr int BN = 128, Row = 128;
  static constexpr int Stages = kBM == 64 ? 3 : 2;
  static constexpr int Slot = (kBM + BN) * Row;              // 24 or 32 KiB
  static constexpr int PerWave = Slot / 1024 / 4;            // LDS-DMA instructions per wave and stage
  static constexpr int LhsJ = kBM / 32;                      // the first of them carry A rows
  static constexpr int WM = kBM / 64, WN = 4 / WM;           // waves along rows and columns
  static constexpr int MB = 4, NB = BN / WN / 16;            // 16-wide blocks per wave
  static constexpr int LdsBytes = Stages * Slot;             // 72 or 64 KiB: two workgroups per CU
  static_assert(4 * 64 * 2 * 16 * NB <= Slot, "epilogue staging fits a slot");
  static constexpr int BandN = 8;                            // column tiles of a band, rows tiles walked inside
};

template <bool kAE5M2, int kBM>
__device__ __forceinline__ void gemm_body(const nt::Args& a, GG_LDS uint8_t* lds) {
  using C = GemmCfg<kBM>;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n_tn = (a.N + C::BN - 1) / C::BN;

  // ---- this workgroup's tile: groups hold ceil(len / BM) n_tn consecutive tiles each
  const int t = tile_of_block(blockIdx.x);
  bool negative;
  const Groups gr = load_groups(a.group_offs, a.G, a.m_total, lane, &negative);
  if (negative) return;                                      // as the persistent kernels: nothing is written
  int cnt[4], sum = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    cnt[k] = (gr.len[k] + kBM - 1) / kBM * n_tn;
    sum += cnt[k];
  }
  const int incl = wave_scan(sum, lane);
  const uint64_t past = __ballot(incl > t);
  if (past == 0) return;                                     // more workgroups than tiles
  const int gl = __builtin_ctzll(past);
  int in_g = t - __builtin_amdgcn_readlane(incl - sum, gl), gx = 0;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const int c = __builtin_amdgcn_readlane(cnt[k], gl);
    if (gx == k && in_g >= c) {
      in_g -= c;
      gx = k + 1;
    }
  }
  const int row_base = pick(gr.start, gl, gx), len = pick(gr.len, gl, gx);
  const int n_tm = (len + kBM - 1) / kBM;
  const int band = in_g / (n_tm * C::BandN);
  const int r = in_g - band * n_tm * C::BandN;
  const int bw = min(C::BandN, n_tn - band * C::BandN);
  const int tm = r / bw;
  const int m0 = tm * kBM, n0 = (band * C::BandN + r - tm * bw) * C::BN;
  const int rows = min(kBM, len - m0), cols = min(C::BN, a.N - n0);
  const uint8_t* pa = a.a + (int64_t)(row_base + m0) * a.stride_am;
  const uint8_t* pb = a.b + (int64_t)(4 * gl + gx) * a.stride_bg + (int64_t)n0 * a.stride_bn;
  const int rec_a = rows * a.stride_am, rec_b = cols * a.stride_bn;

  // ---- stage loads: instruction i = wave + 4 j fills operand rows 8 i' + lane / 8 (A for j < LhsJ)
  const int lc = (lane & 7) ^ (lane >> 3) ^ (wave & 1);      // nt::swz of those rows, for every j
  const int va = (8 * wave + (lane >> 3)) * a.stride_am + 16 * lc;
  const int vb = (8 * wave + (lane >> 3)) * a.stride_bn + 16 * lc;
  auto issue = [&](int step, int slot) {
    const int k0 = step * C::Row;
    const v4i ra = make_rsrc(pa + k0, rec_a - k0), rb = make_rsrc(pb + k0, rec_b - k0);
    const bool dead = 16 * lc >= a.K - k0;                   // chunks at or past K read as zero
    const uint32_t base = lds_u32(lds) + slot * C::Slot + 1024 * wave;
#pragma unroll
    for (int j = 0; j < C::PerWave; ++j) {
      const bool lhs = j < C::LhsJ;
      const int voff = lhs ? va + 32 * j * a.stride_am : vb + 32 * (j - C::LhsJ) * a.stride_bn;
      dma16(lhs ? ra : rb, base + 4096 * j, dead ? (int)kOob : voff);
    }
  };

  // ---- operand reads: lane 16 q + s takes row s of a block, logical chunks 2 q and 2 q + 1
  const int wm = wave % C::WM, wn = wave / C::WM;
  const int q = lane >> 4, s16 = lane & 15;
  const int sw = 16 * ((2 * q) ^ nt::swz(s16));
  const int off_a = (64 * wm + s16) * C::Row + sw;
  const int off_b = (kBM + 16 * C::NB * wn + s16) * C::Row + sw;

  v4f acc[C::MB][C::NB];
#pragma unroll
  for (int i = 0; i < C::MB; ++i)
#pragma unroll
    for (int j = 0; j < C::NB; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

  const int nsteps = (a.K + C::Row - 1) / C::Row;
#pragma unroll
  for (int s = 0; s < C::Stages - 1; ++s)
    if (s < nsteps) issue(s, s);
  int cur = 0, nxt = C::Stages - 1;
  for (int s = 0; s < nsteps; ++s) {
    // stage s has landed for this wave (the stages after it may be in flight), then for all waves;
    // the slot of stage s - 1 is free
    if (s + C::Stages - 1 <= nsteps)
      wait_vmcnt<(C::Stages - 2) * C::PerWave>();
    else
      wait_vmcnt<0>();
    lds_barrier();
    if (s + C::Stages - 1 < nsteps) issue(s + C::Stages - 1, nxt);
    const GG_LDS uint8_t* sa = lds + cur * C::Slot;
    const GG_LDS uint8_t* a_lo = sa + off_a;
    const GG_LDS uint8_t* a_hi = sa + (off_a ^ 16);
    const GG_LDS uint8_t* b_lo = sa + off_b;
    const GG_LDS uint8_t* b_hi = sa + (off_b ^ 16);
    v8i bn[C::NB], am[C::MB];
#pragma unroll
    for (int j = 0; j < C::NB; ++j) bn[j] = nt::read_nt(b_lo + 2048 * j, b_hi + 2048 * j);
#pragma unroll
    for (int i = 0; i < C::MB; ++i) am[i] = nt::read_nt(a_lo + 2048 * i, a_hi + 2048 * i);
#pragma unroll
    for (int i = 0; i < C::MB; ++i)
#pragma unroll
      for (int j = 0; j < C::NB; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bn[j], am[i], acc[i][j], 0, kAE5M2 ? 1 : 0, 0, 0,
                                                                     0, 0);
    nxt = cur;
    cur = cur + 1 == C::Stages ? 0 : cur + 1;
  }

  // ---- epilogue, through the slot that the next stage would have taken: every wave has passed the
  // last stage's barrier, so none reads it any more
  const float alpha = *a.a_scale * *a.b_scale;
  constexpr int kCols = 16 * C::NB;
  store_bf16<C::NB>(acc, alpha, lds + cur * C::Slot + wave * (64 * 2 * kCols),
                    a.c + (int64_t)(row_base + m0 + 64 * wm) * a.stride_cm + n0 + kCols * wn, a.stride_cm,
                    rows - 64 * wm, cols - kCols * wn, lane);
}

}  // namespace mid
}  // namespace ggemm

// Library kernel: the 512-thread kernel's 16 arguments plus M_total and zero_tail; 256 threads, static
// LDS, one tile per workgroup (workgroups past the last tile have none).
#define GGEMM_DEFINE_MID_GEMM_KERNEL(NAME, AE5M2, BM)                                                    \
  extern "C" __global__ __launch_bounds__(ggemm::mid::kNT, 2) void NAME(GGEMM_PERSISTENT_PARAMS,          \
                                                                        int64_t m_total, int zero_tail) { \
    __shared__ __attribute__((aligned(1024))) uint8_t ggemm_mid_lds[ggemm::mid::GemmCfg<BM>::LdsBytes];   \
    ggemm::nt::Args args{a, b, c, a_scale, b_scale, group_offs, G, N, K,                                 \
                         stride_am, stride_bg, stride_bn, stride_cm, stride_cn, m_total, zero_tail};     \
    (void)global_scratch; (void)profile_scratch;                                                        \
    if (G > 0 && G <= ggemm::mid::kMaxGroups && K > 0 && N > 0)                                          \
      ggemm::mid::gemm_body<AE5M2, BM>(ggemm::nt::without_tail(args), (GG_LDS uint8_t*)ggemm_mid_lds);    \
    ggemm::nt::clear_tail_rows(args);                                                                   \
  }
