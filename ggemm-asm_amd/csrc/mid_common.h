// What the two mid-tile kernels share (mid_gemm.h, mid_wgrad.h): one output tile per 256-thread
// workgroup, several workgroups per CU, no persistent schedule. The wide and the 512-thread kernels
// hold one tile of 240-400 KiB of accumulators on each CU for as long as it takes; problems of fewer
// such tiles than CUs, of short groups or of small feature sizes leave most of that idle. Here the
// tiles are a quarter of that size or less, the hardware hands them out as workgroups finish, and
// the other workgroups of a CU compute while one waits for its loads, starts or stores its results.
#pragma once

#include "vark_kernel.h"

namespace ggemm {
namespace mid {

constexpr int kNT = 256;            // threads: four waves
constexpr int kMaxGroups = 256;     // groups a wave holds, four to a lane
constexpr int kXcdRun = 32;         // consecutive tiles that one XCD takes
constexpr uint32_t kOob = 0x7fff0000u;   // buffer offset past every num_records (host-checked)

// Tile of workgroup b: the hardware deals workgroups round robin over the 8 XCDs; runs of kXcdRun
// consecutive tiles go to one XCD, whose L2 then holds the operand rows that they share. The grid is
// a multiple of 8 kXcdRun.
__device__ __forceinline__ int tile_of_block(int b) {
  const int run = kXcds * kXcdRun;
  const int r = b % run;
  return b - r + (r % kXcds) * kXcdRun + r / kXcds;
}

// Four groups per lane: lane l of every wave holds groups 4 l .. 4 l + 3. Their offsets clamped to
// [0, m_total]; each wave reads them for itself, so no barrier and no LDS is needed. Where offsets decrease and
// rise again, rows belong to the first group that holds them: the groups then have no more rows in all than
// there are, nor more tiles than the launch has workgroups, and every row that a group holds is written (the
// offsets begin with zero, so the rows up to the largest one so far are all held).
struct Groups {
  int start[4], len[4];             // first row and row count (0 for g >= G and for decreasing offsets)
};
__device__ __forceinline__ Groups load_groups(const int64_t* offs, int G, int64_t m_total, int lane,
                                              bool* any_negative) {
  int64_t o[5];
  bool neg = false;
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    o[k] = offs[min(4 * lane + k, G)];
    neg |= o[k] < 0;
  }
  *any_negative = __ballot(neg) != 0;
  Groups r;
  int end[4];
  bool falls = false;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    r.start[k] = (int)clamp_off(o[k], m_total);
    end[k] = (int)clamp_off(o[k + 1], m_total);
    r.len[k] = max(end[k] - r.start[k], 0);
    falls |= end[k] < r.start[k];
  }
  if (__ballot(falls) != 0) {
    int past = max(max(end[0], end[1]), max(end[2], end[3]));   // end of the rows held up to here
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int v = __shfl_up(past, d, 64);
      if (lane >= d) past = max(past, v);
    }
    past = __shfl_up(past, 1, 64);
    if (lane == 0) past = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      r.start[k] = max(r.start[k], past);
      r.len[k] = max(end[k] - r.start[k], 0);
      past = max(past, end[k]);
    }
  }
  return r;
}

// Inclusive sum over the lanes of a wave.
__device__ __forceinline__ int wave_scan(int v, int lane) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int o = __shfl_up(v, d, 64);
    if (lane >= d) v += o;
  }
  return v;
}

// Slot x of lane l of a four-per-lane table, for wave-uniform l and x.
__device__ __forceinline__ int pick(const int (&v)[4], int lane, int x) {
  const int s = x == 0 ? v[0] : x == 1 ? v[1] : x == 2 ? v[2] : v[3];
  return __builtin_amdgcn_readlane(s, lane);
}

// Results of a wave: 4 x NB blocks of v_mfma_f32_16x16x128 with C columns on the A side: lane 16 q + s
// holds row 16 i + s, columns 16 j + 4 q .. + 3 in acc[i][j]. They pass through a wave-private LDS
// region and leave as 16-byte chunks in row order, so that the lanes of a store instruction cover
// whole 128-byte lines of C. rows and cols: the part of the wave's block inside C, cols a multiple of
// 16.

typedef unsigned v4u32 __attribute__((ext_vector_type(4)));

// The rows of C that a wave stores, as a buffer: rows past it are neither read nor written. A row's offset
// goes into the lane offset, which the range check compares with num_records; with it in the scalar offset
// the check subtracts that from num_records, and rows past the block are those where this is negative.
struct CBlock {
  __amdgpu_buffer_rsrc_t rsrc;
  int pitch;                        // bytes between rows (64 of them within kOob: host-checked)
  template <typename T>
  __device__ __forceinline__ CBlock(T* c, int64_t stride, int rows)
      : rsrc(__builtin_amdgcn_make_buffer_rsrc(c, 0, max(0, min(rows, 64)) * (int)(stride * sizeof(T)), kRsrcWord3)),
        pitch((int)(stride * sizeof(T))) {}
  __device__ __forceinline__ v4i load(uint32_t off) const {
    return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)off, 0, 0));
  }
  __device__ __forceinline__ void store(v4i v, uint32_t off) const {   // non-temporal
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u32, v), rsrc, (int)off, 0, 2);
  }
};

template <int NB>
__device__ __forceinline__ void store_bf16(const v4f (&acc)[4][NB], float alpha, GG_LDS uint8_t* reg, uint16_t* c,
                                           int64_t stride, int rows, int cols, int lane) {
  // 64 rows of 32 NB bytes, chunk k of row r at k ^ ((r >> 1) & (2 NB - 1))
  constexpr int kChunks = 2 * NB, kRow = 16 * kChunks;
  const int q = lane >> 4, s16 = lane & 15;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const v4f v = acc[i][j];
      const v2i pk = v2i{(int)(f32_to_bf16_rne(v[0] * alpha) | (f32_to_bf16_rne(v[1] * alpha) << 16)),
                         (int)(f32_to_bf16_rne(v[2] * alpha) | (f32_to_bf16_rne(v[3] * alpha) << 16))};
      const int r = 16 * i + s16, k = 2 * j + (q >> 1);
      *(GG_LDS v2i*)(reg + r * kRow + 16 * (k ^ ((r >> 1) & (kChunks - 1))) + 8 * (q & 1)) = pk;
    }
  // row 64 n / kChunks + lane / kChunks, chunk lane % kChunks: rows past the block fall outside the
  // resource, the other columns' lanes too
  const CBlock b(c, stride, rows);
  const uint32_t v = 8 * (lane % kChunks) < cols ? lane / kChunks * b.pitch + 16 * (lane % kChunks) : kOob;
#pragma unroll
  for (int n = 0; n < kChunks; ++n) {
    const int f = 64 * n + lane, r = f / kChunks, k = f % kChunks;
    b.store(*(const GG_LDS v4i*)(reg + r * kRow + 16 * (k ^ ((r >> 1) & (kChunks - 1)))),
            v + (uint32_t)(n * (64 / kChunks) * b.pitch));
  }
}

// fp32, 64 columns: two passes of 32 rows of 256 bytes, chunk k of row r at k ^ (r & 15).
// kAdd: added to the C there, the scaled value rounded first.
template <bool kAdd>
__device__ __forceinline__ void store_f32(const v4f (&acc)[4][4], float alpha, GG_LDS uint8_t* reg, float* c,
                                          int64_t stride, int rows, int cols, int lane) {
  const int q = lane >> 4, s16 = lane & 15;
  const CBlock b(c, stride, rows);
  const uint32_t v = 4 * s16 < cols ? q * b.pitch + 16 * s16 : kOob;
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    v4f old[8];
    if constexpr (kAdd) {
#pragma unroll
      for (int n = 0; n < 8; ++n) old[n] = __builtin_bit_cast(v4f, b.load(v + (uint32_t)((32 * p + 4 * n) * b.pitch)));
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int r = 16 * i + s16;
        *(GG_LDS v4f*)(reg + r * 256 + 16 * ((4 * j + q) ^ s16)) = acc[2 * p + i][j] * alpha;
      }
#pragma unroll
    for (int n = 0; n < 8; ++n) {
      const int r = 4 * n + q;
      v4f x = *(const GG_LDS v4f*)(reg + r * 256 + 16 * (s16 ^ (r & 15)));
      if constexpr (kAdd) x += old[n];
      b.store(__builtin_bit_cast(v4i, x), v + (uint32_t)((32 * p + 4 * n) * b.pitch));
    }
  }
}

}  // namespace mid
}  // namespace ggemm
