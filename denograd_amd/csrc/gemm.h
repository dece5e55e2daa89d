// What the several-row kernels share: gemm.hip (few rows), gemm_tile.hip and gemm_staged.hip (more than that), prefill.hip (causal attention).
#pragma once
#include <stdlib.h>
#include <string.h>
#include <unistd.h>

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
  // x is to be RMSNorm'ed first: gemm_few.hip does that in registers, for the others x is normed in memory
  const _Float16 *norm_w;             // [K] or null
  float eps, inv_k;                   // inv_k: float(1 / K)
  bool pins;                          // some variable of the environment begins with JSG_: a test may want a certain kernel or tile
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

// ---- direct global-to-LDS loads
typedef int i4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ i4_t dma_rsrc(const void *p) {
  const uint64_t v = (uint64_t)p;
  i4_t r;
  r.x = __builtin_amdgcn_readfirstlane((int)(uint32_t)v);
  r.y = __builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
  r.z = -1;                            // callers keep their offsets in bounds
  r.w = 0x00020000;
  return r;
}
// 64 lanes x 16 bytes from rs + voff(lane) + soff to LDS bytes [lds, lds + 1024) in lane order.  M0 holds the LDS address; one
// wait state between writing it and the load that reads it.
__device__ __forceinline__ void dma16(i4_t rs, uint32_t voff, uint32_t soff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(lds), "v"(voff), "s"(rs), "s"(soff) : "memory");
}
// the same for bytes that are read once
__device__ __forceinline__ void dma16_stream(i4_t rs, uint32_t voff, uint32_t soff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds" ::"s"(lds), "v"(voff), "s"(rs), "s"(soff) : "memory");
}
// the same with four bytes per lane
__device__ __forceinline__ void dma4(i4_t rs, uint32_t voff, uint32_t soff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds" ::"s"(lds), "v"(voff), "s"(rs), "s"(soff) : "memory");
}

// RMSNorm.call (nn/index.ts:586-588) with the rounding points of rmsnorm_rows_kernel: the factor of a row with this sum of squares, and
// eight elements of it
__device__ __forceinline__ float norm_factor(const GemmArgs &a, float sum) { return __fsqrt_rn(__fdiv_rn(1.0f, __fadd_rn(__fmul_rn(sum, a.inv_k), a.eps))); }
__device__ __forceinline__ h8_t norm_piece(h8_t x, float r, h8_t w) {
  h8_t n;
#pragma unroll
  for (int e = 0; e < 8; e++) n[e] = (_Float16)__fmul_rn((float)x[e], r);
  return n * w;
}
// Plus the squares of eight elements, one by one (products of halves are exact, so each costs one rounding).  v_dot2_f32_f16 adds two at once and its sums are
// further off: of 85 M normed elements of rows of 1024 to 4096, 4472 were not the nearest half, one by one 4176.  What that costs, us, 5 rows, two | one:
// norm and wq|wk|wv of 3072 x 2048 5.6 | 5.9, w1|w3 of 8192 x 2048 14.6 | 14.6, int8 w1|w3 of 8192 x 3072 12.2 | 12.4.
__device__ __forceinline__ float square_sum(h8_t x, float s) {
#pragma unroll
  for (int e = 0; e < 8; e++) s = fmaf((float)x[e], (float)x[e], s);
  return s;
}

// What a test asks for, or null.  Looking a variable up costs a walk through the environment, so a call makes one walk for all of them.
inline bool any_pins() {
  for (char **e = environ; e && *e; e++)                     // null behind clearenv()
    if (!strncmp(*e, "JSG_", 4)) return true;
  return false;
}
inline const char *pin_env(const GemmArgs &a, const char *name) { return a.pins ? getenv(name) : nullptr; }

// gemm_few.hip: at most 16 rows, weights streamed past x in registers; *taken false: not for this call, nothing launched
int gemm_few(int epi, int kind, const GemmArgs &a, int prof_kind, bool *taken);
// gemm_group.hip: at most 32 rows, wherever the weight-streaming kernels of gemm.hip are slower; *taken as above
int gemm_group(int epi, int kind, const GemmArgs &a, int prof_kind, bool *taken);
// gemm_tile.hip: the tiled kernels, any number of rows; epi: GEPI_*
int gemm_tiled(int epi, int kind, const GemmArgs &a, int prof_kind);
// gemm_staged.hip: quantised weights dequantised on their way into LDS, any number of rows; tiles of bm x bn: 32x128 (not for w1|w3),
// 128x128, 256x128 or 256x256 (the output, w1 and w3 counted together, is then a multiple of 256)
int gemm_staged(int epi, int kind, int bm, int bn, const GemmArgs &a, int prof_kind);

}  // namespace jsg
