// Arguments and entry points that the several-row kernels share (gemm.hip: few rows, gemm_tile.hip: more than that).
#pragma once
#include "common.h"

namespace jsg {

typedef _Float16 h4_t __attribute__((ext_vector_type(4)));

enum { GEPI_STORE = 0, GEPI_ROPE_KV = 1, GEPI_SWIGLU = 2 };

struct GemmArgs {
  const void *w0, *w1, *w2;           // up to three weight matrices stacked along N (wq|wk|wv, or w1|w3)
  const _Float16 *s0, *s1, *s2;       // their scales (int8: per row; nf4: per 64 elements)
  int n0, n1, n2;                     // their row counts
  int M, N, K;                        // N = columns of the output this launch produces
  const _Float16 *x;                  // [M][K]
  _Float16 *y;                        // [M][N]  (ROPE_KV: q rows [M][n0])
  const _Float16 *residual;           // [M][N] or null
  // ROPE_KV
  const _Float16 *rope_table;         // [2*max_context][hd/2][2]
  _Float16 *cache_k, *cache_v;        // [B][max_context][n1]
  int seq_len, start_pos, head_dim, max_context;
};

__device__ __forceinline__ uint32_t pk_mul_h2(uint32_t a, h2_t s) {
  h2_t r = as_h2(a) * s;
  return __builtin_bit_cast(uint32_t, r);
}

// 4 int8 codes (one dword) -> 4 exact fp16 values: byte | 0x6400 is 1024 + (code ^ 0x80), minus 1152 leaves the code
__device__ __forceinline__ void i8x4_to_h2x2(uint32_t q, uint32_t &lo, uint32_t &hi) {
  const uint32_t u = q ^ 0x80808080u;
  const h2_t bias = {(_Float16)1152.0f, (_Float16)1152.0f};
  h2_t a = as_h2(__builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) - bias;   // bytes 0,1
  h2_t b = as_h2(__builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) - bias;   // bytes 2,3
  lo = __builtin_bit_cast(uint32_t, a);
  hi = __builtin_bit_cast(uint32_t, b);
}

// gemm_tile.hip: the tiled kernels, any number of rows; epi: GEPI_*
int gemm_tiled(int epi, int kind, const GemmArgs &a, int prof_kind);
// gemm.hip: 8 MiB of device memory that belong to the several-row kernels (one launch at a time: the stream orders them)
int gemm_scratch(void **host_out, size_t *host_out_bytes);

}  // namespace jsg
