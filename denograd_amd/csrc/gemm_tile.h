// What the tiled several-row kernels share (gemm_tile.hip, gemm_group.hip): a launch's arguments, the order of its tiles, where the
// weight rows of a tile lie, and how eight neighbouring outputs of a row are stored.
#pragma once
#include "gemm.h"

namespace jsg {

constexpr int TILE_BK = 64;
constexpr int TILE_THREADS = 512;

struct TileArgs {
  GemmArgs g;                          // output side: y, residual, rope, cache, M, N, K
  const void *b[3];                    // weight rows (fp16, or codes), up to three matrices on top of each other
  const _Float16 *s[3];                // codes: their scales
  int b_end[2];                        // ends of the first two (SWIGLU: b[0] is w1, b[1] is w3, row for row)
  int split;                           // K parts
  int whole = 0;                       // 256 x 256: tiles of whole K, in front of those that come in parts
  float *ws;                           // split > 1: [tile][part][BM * BN] floats
  int *counters;                       // split > 1: one per tile, zero, and zero again afterwards
};

template <int N> __device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
__device__ __forceinline__ void turn_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}
// ... after this wavefront's LDS reads have arrived
__device__ __forceinline__ void turn_barrier_lds() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// Block id -> tile (and K part): blocks are dealt to the eight XCDs round-robin, so ids are first made contiguous per XCD; K
// parts of a tile are neighbours, then GROUP row tiles share each column tile, so that the blocks resident on one XCD share
// operand tiles in its L2.  (GROUP 2 / 4 / 8 / 16 at 32768 x 4096 x 14336: 1453 / 1451 / 1413 / 1334 TFLOP/s, at
// 32768 x 28672 x 4096: 1392 / 1422 / 1440 / 1318.)
struct TileId { int tile, part, m0, col; };
// The first `whole` tiles are a block each and come first.
template <int BM, int CW> __device__ __forceinline__ TileId tile_id(const TileArgs &t, int whole = 0) {
  constexpr int GROUP = 4;
  const int tiles_m = (t.g.M + BM - 1) / BM, tiles_n = t.g.N / CW;
  const bool in_parts = (int)blockIdx.x >= whole;
  const int split = in_parts ? t.split : 1, nblocks = in_parts ? (tiles_m * tiles_n - whole) * split : whole;
  int bid = (int)blockIdx.x - (in_parts ? whole : 0);
  const int per = nblocks / 8;
  if (bid < per * 8) bid = (bid & 7) * per + (bid >> 3);
  TileId r;
  r.part = bid % split;
  r.tile = (in_parts ? whole : 0) + bid / split;
  const int in_group = GROUP * tiles_n, first_m = (r.tile / in_group) * GROUP, gsz = min(tiles_m - first_m, GROUP);
  r.m0 = (first_m + (r.tile % in_group) % gsz) * BM;
  r.col = ((r.tile % in_group) / gsz) * CW;
  return r;
}

// Where row r of a weight tile of BN rows lies: the matrix and its row.  Boundaries are multiples of 64, so the 8 or 16 rows of a
// load, or of a fragment, never straddle two matrices.
struct WeightRow { int mat, row; };
template <int EPI, int BN> __device__ __forceinline__ WeightRow weight_row(const TileArgs &t, int col, int r) {
  if constexpr (EPI == GEPI_SWIGLU) return r < BN / 2 ? WeightRow{0, col + r} : WeightRow{1, col + r - BN / 2};
  else {
    const int n = col + r;
    if (n < t.b_end[0]) return {0, n};
    if (n < t.b_end[1]) return {1, n - t.b_end[0]};
    return {2, n - t.b_end[1]};
  }
}
template <typename T> __device__ __forceinline__ const T *pick(const T *const (&p)[3], int i) { return i == 0 ? p[0] : (i == 1 ? p[1] : p[2]); }
template <int EPI, int BN> __device__ __forceinline__ const unsigned char *weight_ptr(const TileArgs &t, int col, int r, size_t row_bytes) {
  const WeightRow w = weight_row<EPI, BN>(t, col, r);
  return (const unsigned char *)pick(t.b, w.mat) + (size_t)w.row * row_bytes;
}

// Eight neighbouring outputs of row m, columns n .. n + 7, as 16 bytes.  SWIGLU: v is the product already; STORE: res is the residual's piece.
template <int EPI> __device__ __forceinline__ void store_piece(const GemmArgs &a, int m, int n, h8_t v, h8_t res) {
  if constexpr (EPI == GEPI_SWIGLU) {
    *(h8_t *)&a.y[(size_t)m * a.N + n] = v;
  } else if constexpr (EPI == GEPI_STORE) {
    h8_t o = v;
    if (a.residual) {
#pragma unroll
      for (int c = 0; c < 8; c++) o[c] = (_Float16)((float)res[c] + (float)v[c]);
    }
    *(h8_t *)&a.y[(size_t)m * a.N + n] = o;
  } else {
    // wq | wk | wv columns; q and k get the interleaved-pair rotation (llama.ts:17-32), k and v go to the cache rows.
    // Eight neighbouring columns are four pairs of one head of one matrix (every boundary is a multiple of 8).
    const int b = m / a.seq_len, pos = a.start_pos + m % a.seq_len;
    const int which = n < a.n0 ? 0 : (n < a.n0 + a.n1 ? 1 : 2);
    const int nl = which == 0 ? n : (which == 1 ? n - a.n0 : n - a.n0 - a.n1);
    h8_t o = v;
    if (which < 2) {
      const int pair = (nl % a.head_dim) >> 1;
      const h8_t cs = *(const h8_t *)(a.rope_table + ((size_t)pos * (a.head_dim / 2) + pair) * 2);   // cos, sin of four pairs
#pragma unroll
      for (int h = 0; h < 4; h++) {
        const float ev = (float)v[2 * h], od = (float)v[2 * h + 1];
        const float c = (float)cs[2 * h], d = (float)cs[2 * h + 1];
        o[2 * h] = (_Float16)(ev * c - od * d);
        o[2 * h + 1] = (_Float16)(ev * d + od * c);
      }
    }
    if (which == 0) *(h8_t *)&a.y[(size_t)m * a.n0 + nl] = o;
    else {
      _Float16 *cache = which == 1 ? a.cache_k : a.cache_v;
      *(h8_t *)&cache[((size_t)b * a.max_context + pos) * a.n1 + nl] = o;
    }
  }
}
// silu(w1 x) * (w3 x), each GEMM output and the product stored as fp16 (llama.ts:108-110)
__device__ __forceinline__ float swiglu(float gate, float up) { return silu_act<_Float16>(rn16(gate)) * rn16(up); }

// The arguments of a launch without K parts
inline TileArgs tile_args(int epi, const GemmArgs &a, int *counters) {
  TileArgs t = {};
  t.g = a;
  t.b[0] = a.w0; t.b[1] = a.w1; t.b[2] = a.w2;
  t.s[0] = a.s0; t.s[1] = a.s1; t.s[2] = a.s2;
  t.b_end[0] = epi == GEPI_ROPE_KV ? a.n0 : a.N;
  t.b_end[1] = t.b_end[0] + (epi == GEPI_ROPE_KV ? a.n1 : 0);
  t.split = 1;
  t.counters = counters;
  return t;
}

// gemm_group.hip: at most 64 rows.  The estimate of its fastest shape for a call; shape < 0: not for this call.
struct GroupChoice { float us = 0.0f; int shape = -1, split = 1; };
GroupChoice choose_group(int epi, int kind, const GemmArgs &a);
int run_group(int epi, int kind, const GemmArgs &a, const GroupChoice &c, int prof_kind);

}  // namespace jsg
