// Several-position kernels for fp16 activations: causal grouped-query attention on the matrix cores for S > 1 new
// positions per sequence (batched prefill), and the row-wise companions of the one-row kernels (embedding gather,
// RMSNorm, greedy argmax) for [rows][...] inputs.
//
// Reference semantics: Attention.call with a mask (/root/reference/jsgrad/models/llama.ts:61-97, mask :208 =
// triu(start_pos + 1) of -inf), repeat_kv :34-39, scaled_dot_product_attention /root/reference/jsgrad/tensor.ts:3920-3934
// (float32 scores and softmax, probabilities cast to fp16, float32 P.V sum, fp16 out).
#include "gemm.h"

namespace jsg {

typedef float f16_t __attribute__((ext_vector_type(16)));
typedef short s4_t __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------- causal attention, S new positions
//
// Block = 4 wavefronts = 128 query rows of one kv head of one sequence: its n_rep query heads side by side, row = position *
// n_rep + head, so that a wavefront's 32 rows are a few positions (little is computed above the diagonal) and a short prompt
// still fills its rows.  Keys are walked in tiles of 64.  Scores are computed TRANSPOSED, S^T = K . Q^T (A operand = K rows from
// LDS, B operand = the lane's query row held in registers), so that a lane holds 32 scores of ONE query row per tile: the
// online-softmax statistics are lane-local (plus one exchange between the two lane halves), and the fp16 probabilities are
// already laid out as the B operand of O^T = V^T . P^T.  The k-slot order of an MFMA operand is free as long as both
// operands agree.
// K and V tiles come by direct global-to-LDS loads into one of two buffers, rows as they are in the cache, the 16-byte pieces
// of a row exchanged by row number so that fragment reads hit different banks.  V^T fragments come out of the row-major tile
// by transposing LDS reads: within 16 lanes, lane i gets element i of four rows, row j being what lanes 4j .. 4j+3 address.
// One barrier per tile: tile t + 1 is asked for behind the barrier of tile t, into the buffer of tile t - 1.
// What bounds it: per tile a wavefront has 32 matrix instructions (1100 cycles) and ~1000 cycles of vector work (a
// quarter-rate exponential per score); two blocks per CU, so that one wavefront of a SIMD computes under the other's softmax.
// Measured (TFLOP/s of visible scores, head_dim 128, 32 heads, 8 kv heads): 16 x 2048 positions 799, 1 x 4096 800 (437 and 463 for
// the kernel with tiles through registers, V transposed on the way into LDS and one query head per block).
// A grid that does not fill the chip is split along the keys: every part leaves its running sums in a workspace and the last
// of a wavefront's parts to arrive folds them in order.
constexpr int PF_THREADS = 256, PF_QROWS = 128, PF_KEYS = 64;
constexpr int PF_COUNTERS = 4096;
static __device__ int pf_counters[PF_COUNTERS];

// x / d for 0 <= x < 2^30: a division in full is 30 instructions that wait for each other, and a block of a short prompt has eight
// of them in front of its one tile (57 positions, 24 heads of 128: 5.6 us, 5.5 without).
struct Divisor {
  uint32_t d, mul, shift;
  __device__ int div(int x) const { return mul ? (int)(__umulhi((uint32_t)x, mul) >> shift) : x; }
};
static Divisor divisor(uint32_t d) {
  Divisor r = {d, 0, 0};
  if (d == 1) return r;
  int s = 1;
  while ((1u << s) < d) s++;
  const int n = s < 2 ? 32 : 30 + s;                          // mul = ceil(2^n / d) <= 2^31, off by less than d <= 2^s
  r.mul = (uint32_t)((((uint64_t)1 << n) + d - 1) / d);
  r.shift = n - 32;
  return r;
}

struct PrefillAttnArgs {
  const _Float16 *q;                 // [B*S][H*HD]
  const _Float16 *cache_k, *cache_v; // [B][max_context][KV][HD]
  _Float16 *out;                     // [B*S][H*HD]
  int S, start_pos, max_context;
  Divisor n_rep, n_kv_heads, tile_div;
  int tiles, pairs;                  // query tiles per (sequence, kv head); sequences x kv heads
  int parts;                         // key parts
  float *ws;                         // parts > 1: [block][part][wavefront][HD / 2 + 2 values][64 lanes]
  int *counters;                     // parts > 1: one per (block, wavefront), zero, and zero again afterwards
  float scale_log2;                  // float(1/sqrt(HD)) * log2(e)
};

template <int HD> __global__ __launch_bounds__(PF_THREADS, 2) void attn_prefill_kernel(PrefillAttnArgs a) {
  constexpr int ROWB = HD * 2, PPR = HD / 8;                 // bytes and 16-byte pieces of a cache row of one head
  constexpr int TILE = PF_KEYS * ROWB, BUF = 2 * TILE;       // K tile, then V tile
  constexpr int LOADS = TILE / 1024 / 4;                     // a wavefront's loads per tile of K, and of V
  constexpr int RPL = 64 / PPR;                              // rows per load
  constexpr int NT = HD / 32;                                // 32-feature tiles of the output
  __shared__ __align__(16) unsigned char lds[2 * BUF];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, lg = lane >> 5;
  // Blocks are dealt to the eight XCDs round-robin: ids are made contiguous per XCD, so that the query tiles of a (sequence,
  // kv head) run on one XCD and share its K and V in that L2; within one the tiles with the most keys come first.
  const int nblocks = a.tiles * a.pairs * a.parts;
  int bid = blockIdx.x;
  const int per = nblocks / 8;
  if (bid < per * 8) bid = (bid & 7) * per + (bid >> 3);
  int part = 0, blk = bid;
  if (a.parts > 1) {
    part = bid % a.parts;
    blk = bid / a.parts;
  }
  const int pair = a.tile_div.div(blk), qt = a.tiles - 1 - (blk - pair * a.tiles);
  const int n_rep = (int)a.n_rep.d, n_kv_heads = (int)a.n_kv_heads.d;
  const int b = a.n_kv_heads.div(pair), g = pair - b * n_kv_heads;
  const int rows = a.S * n_rep;
  const int q0 = qt * PF_QROWS, qw0 = q0 + wave * 32;
  const int n_tiles = (a.start_pos + a.n_rep.div(min(q0 + PF_QROWS, rows) - 1)) / PF_KEYS + 1;
  int t_lo = 0, t_hi = n_tiles;
  if (a.parts > 1) {
    t_lo = part * n_tiles / a.parts;
    t_hi = (part + 1) * n_tiles / a.parts;
  }
  // this wavefront's first and last position; rows past the end repeat the last one and are never stored
  const int pos_lo = a.start_pos + a.n_rep.div(min(qw0, rows - 1)), pos_hi = a.start_pos + a.n_rep.div(min(qw0 + 31, rows - 1));
  const bool q_valid = qw0 + l32 < rows;
  const int qrow = min(qw0 + l32, rows - 1), qs = a.n_rep.div(qrow), qpos = a.start_pos + qs;   // keys <= qpos are visible
  const size_t q_off = ((size_t)b * a.S + qs) * (n_kv_heads * n_rep) * HD + (size_t)(g * n_rep + qrow - qs * n_rep) * HD;

  const uint32_t row_stride = (uint32_t)n_kv_heads * ROWB;
  const size_t base = (size_t)b * a.max_context * row_stride + (size_t)g * ROWB;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)lds + wave * LOADS * 1024;
  const int lrow = lane / PPR, lp = lane % PPR, last_row = a.max_context - 1;
  // where piece p of row r of a tile is kept: K by all pieces of a row, V by pairs of pieces (a transposing read takes 32 bytes of
  // eight rows)
  auto k_at = [](int r, int p) { return HD == 128 ? p ^ (r & 15) : p ^ (r & 7); };
  auto v_at = [](int r, int p) { return HD == 128 ? p ^ ((r & 7) << 1) : p ^ (((r >> 1) & 3) << 1); };
  auto issue = [&](int t, int buf) {
    const uint32_t to = lds0 + buf * BUF;
    // the tile's first row is in the descriptors: a sequence's cache may be longer than 32-bit offsets reach
    const size_t tile = base + (size_t)t * PF_KEYS * row_stride;
    const i4_t rk = dma_rsrc((const unsigned char *)a.cache_k + tile), rv = dma_rsrc((const unsigned char *)a.cache_v + tile);
#pragma unroll
    for (int i = 0; i < LOADS; i++) {
      const int r = (wave * LOADS + i) * RPL + lrow;          // row of the tile this lane brings a piece of
      const uint32_t key = (uint32_t)min(r, last_row - t * PF_KEYS) * row_stride;   // behind the cache's end: masked, any row will do
      dma16(rk, key + k_at(r, lp) * 16, 0, to + i * 1024);
      dma16(rv, key + v_at(r, lp) * 16, 0, to + TILE + i * 1024);
    }
  };

  if (t_lo < t_hi) issue(t_lo, 0);
  // query row fragments: chunk c covers features [16c, 16c+16), the lane half picks 8 of them
  h8_t qf[HD / 16];
  {
    const _Float16 *qp = a.q + q_off + lg * 8;
#pragma unroll
    for (int c = 0; c < HD / 16; c++) qf[c] = *(const h8_t *)(qp + c * 16);
  }
#pragma unroll
  for (int c = 0; c < HD / 16; c++) asm volatile("" : "+v"(qf[c]));   // waited for here, in front of the loop

  f16_t o_acc[NT];
#pragma unroll
  for (int t = 0; t < NT; t++)
#pragma unroll
    for (int r = 0; r < 16; r++) o_acc[t][r] = 0.0f;
  // the maximum starts finite: a part of the keys may hold none that a row sees, and -inf minus -inf is not a number
  float m_run = -1e30f, l_run = 0.0f;

  // K fragment of key l32 (+ 32): chunk 2c + lg of its row; V: lane -> row (lane / 4 % 4) of its half's four keys, 8 bytes
  const unsigned char *const kp = lds + l32 * ROWB;
  const int vrow = 4 * lg + ((lane >> 2) & 3), vcol = ((lane >> 4) & 1) * 32 + (lane & 3) * 8;   // byte column inside 64 (32 features)

  for (int t = t_lo, buf = 0; t < t_hi; t++, buf ^= 1) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();                                            // tile t is there, everyone is done with tile t - 1
    if (t + 1 < t_hi) issue(t + 1, buf ^ 1);
    const int k0 = t * PF_KEYS;
    if (k0 > pos_hi) continue;                                // every key of the tile is masked for this wavefront (uniform)

    // S^T tile: 64 keys x 32 query rows
    f16_t s[2];
#pragma unroll
    for (int tk = 0; tk < 2; tk++) {
#pragma unroll
      for (int r = 0; r < 16; r++) s[tk][r] = 0.0f;
#pragma unroll
      for (int c = 0; c < HD / 16; c++) {
        const h8_t kf = *(const h8_t *)(kp + buf * BUF + tk * 32 * ROWB + k_at(l32, 2 * c + lg) * 16);
        s[tk] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[c], s[tk], 0, 0, 0);
      }
    }
    // accumulator r of s[tk] is key k0 + tk*32 + 8*(r/4) + 4*lg + r%4 for query row l32.  Only a tile that reaches past
    // the first query row of the wavefront has masked keys (uniform test); the scale is positive, so the maximum is
    // taken over the raw scores and the scale folded into the exponent: exp2(s * scale - max * scale).
    if (k0 + PF_KEYS - 1 > pos_lo) {
#pragma unroll
      for (int tk = 0; tk < 2; tk++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
          const int key = k0 + tk * 32 + 8 * (r / 4) + 4 * lg + (r % 4);
          if (key > qpos) s[tk][r] = -INFINITY;
        }
    }
    float mx = m_run;
#pragma unroll
    for (int tk = 0; tk < 2; tk++)
#pragma unroll
      for (int r = 0; r < 16; r += 2) mx = fmaxf(fmaxf(mx, s[tk][r]), s[tk][r + 1]);
    mx = max_xor32(mx);
    // The sums are rescaled when some row's maximum has moved (uniform branch; two tiles in three), so that the largest
    // probability of a row is 1 and its fp16 rounding exact.  Rescaled only after growth by 2^8 the kernel is faster (838 and 832
    // TFLOP/s), but every probability is rounded: relative error against float64 2.48e-4 instead of 2.21e-4 with scores of
    // deviation 3, 2.61e-4 instead of 2.54e-4 with deviation 1 (2048 positions).
    if (__builtin_amdgcn_ballot_w64(mx > m_run)) {
      const float alpha = __builtin_amdgcn_exp2f((m_run - mx) * a.scale_log2);   // first visible tile: 0
      m_run = mx;
      l_run *= alpha;
#pragma unroll
      for (int td = 0; td < NT; td++)
#pragma unroll
        for (int r = 0; r < 16; r++) o_acc[td][r] *= alpha;
    }
    const float mxs = m_run * a.scale_log2;
    float psum[2] = {0.0f, 0.0f};
    h8_t pf[2][2];
#pragma unroll
    for (int tk = 0; tk < 2; tk++)
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[tk][r], a.scale_log2, -mxs));
        psum[tk] += p;
        pf[tk][r / 8][r % 8] = (_Float16)p;
      }
    l_run += psum[0] + psum[1];

    // O^T += V^T . P^T : k-slot s' of lane half lg in step (tk, hs) is key tk*32 + hs*16 + 8*(s'/4) + 4*lg + s'%4
    const unsigned char *const vt = lds + buf * BUF + TILE;
#pragma unroll
    for (int tk = 0; tk < 2; tk++)
#pragma unroll
      for (int hs = 0; hs < 2; hs++)
#pragma unroll
        for (int td = 0; td < NT; td++) {
          s4_t v[2];
#pragma unroll
          for (int e = 0; e < 2; e++) {
            const int r = tk * 32 + hs * 16 + 8 * e + vrow, c = td * 64 + vcol;
            v[e] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4_t *)(vt + r * ROWB + v_at(r, c >> 4) * 16 + (c & 15)));
          }
          const h8_t vf = __builtin_bit_cast(h8_t, __builtin_shufflevector(v[0], v[1], 0, 1, 2, 3, 4, 5, 6, 7));
          o_acc[td] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, pf[tk][hs], o_acc[td], 0, 0, 0);
        }
  }

  if (a.parts > 1) {
    // Sums cross compute units on different XCDs: device-scope stores and loads (cache policy 16), counted once they are
    // acknowledged (the offset in the vector register, see sum_parts in gemm_tile.hip).
    constexpr int VALS = (HD / 2 + 4) * 64;                   // floats of one wavefront: O^T, then (m, l)
    const uint32_t slot = (uint32_t)VALS * 4;
    const __amdgpu_buffer_rsrc_t rw = wave_buffer(a.ws + ((size_t)blk * a.parts * 4 + wave) * VALS, (a.parts - 1) * 4u * slot + slot);
    const uint32_t mine = (uint32_t)part * 4 * slot + lane * 16;
#pragma unroll
    for (int td = 0; td < NT; td++)
#pragma unroll
      for (int r4 = 0; r4 < 4; r4++) {
        const f4_t v = {o_acc[td][r4 * 4], o_acc[td][r4 * 4 + 1], o_acc[td][r4 * 4 + 2], o_acc[td][r4 * 4 + 3]};
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4_t, v), rw, mine + (td * 4 + r4) * 1024, 0, 16);
      }
    const f4_t ml = {m_run, l_run, 0.0f, 0.0f};
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4_t, ml), rw, mine + NT * 4 * 1024, 0, 16);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    int old = 0;
    if (lane == 0) old = __hip_atomic_fetch_add(&a.counters[blk * 4 + wave], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    old = __builtin_amdgcn_readfirstlane(old);
    if (old != a.parts - 1) return;
    if (lane == 0) __hip_atomic_store(&a.counters[blk * 4 + wave], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // for the next launch
    // two parts per round trip; past the last part the last one again, with weight zero
    m_run = -1e30f;
    l_run = 0.0f;
#pragma unroll
    for (int td = 0; td < NT; td++)
#pragma unroll
      for (int r = 0; r < 16; r++) o_acc[td][r] = 0.0f;
    for (int p0 = 0; p0 < a.parts; p0 += 2) {
      f4_t w[2], v[2][NT * 4];
#pragma unroll
      for (int u = 0; u < 2; u++) {
        const uint32_t from = (uint32_t)min(p0 + u, a.parts - 1) * 4 * slot + lane * 16;
        w[u] = __builtin_bit_cast(f4_t, __builtin_amdgcn_raw_buffer_load_b128(rw, from + NT * 4 * 1024, 0, 16));
#pragma unroll
        for (int i = 0; i < NT * 4; i++) v[u][i] = __builtin_bit_cast(f4_t, __builtin_amdgcn_raw_buffer_load_b128(rw, from + i * 1024, 0, 16));
      }
      const float m = fmaxf(m_run, fmaxf(w[0][0], w[1][0]));
      const float f = __builtin_amdgcn_exp2f((m_run - m) * a.scale_log2);
      const float f0 = __builtin_amdgcn_exp2f((w[0][0] - m) * a.scale_log2);   // a part without a visible key: 0
      const float f1 = p0 + 1 < a.parts ? __builtin_amdgcn_exp2f((w[1][0] - m) * a.scale_log2) : 0.0f;
      m_run = m;
      l_run = l_run * f + (w[0][1] * f0 + w[1][1] * f1);
#pragma unroll
      for (int i = 0; i < NT * 4; i++)
#pragma unroll
        for (int e = 0; e < 4; e++) o_acc[i / 4][(i % 4) * 4 + e] = o_acc[i / 4][(i % 4) * 4 + e] * f + (v[0][i][e] * f0 + v[1][i][e] * f1);
    }
  }

  const float inv = 1.0f / add_xor32(l_run);
  {
    _Float16 *op = a.out + q_off;
#pragma unroll
    for (int td = 0; td < NT; td++)
#pragma unroll
      for (int j = 0; j < 2; j++) {
        // a lane half holds four of every eight neighbouring features; the halves exchange, so that each has all eight of every other
        // group: one store instruction of 16 bytes a lane instead of two of 8 (57 positions, 24 heads of 128: 6.5 -> 5.6 us, 16 x 128
        // positions, 32 heads: 14.0 -> 12.7)
        uint32_t g[2][2];
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
          for (int e = 0; e < 2; e++) {
            const h2_t h = {(_Float16)(o_acc[td][(2 * j + u) * 4 + 2 * e] * inv), (_Float16)(o_acc[td][(2 * j + u) * 4 + 2 * e + 1] * inv)};
            g[u][e] = __builtin_bit_cast(uint32_t, h);
          }
        const auto lo = __builtin_amdgcn_permlane32_swap(g[0][0], g[1][0], false, false);
        const auto hi = __builtin_amdgcn_permlane32_swap(g[0][1], g[1][1], false, false);
        const u4_t v = {lo[0], hi[0], lo[1], hi[1]};
        if (q_valid) *(u4_t *)(op + td * 32 + 16 * j + 8 * lg) = v;
      }
  }
}

// ---------------------------------------------------------------- row-wise companions

// Embedding.call / Int8Embedding.call (nn/index.ts:607-619, llama3.ts:71-77) for `rows` token ids.  VEC: rows of whole pieces of eight elements,
// a piece of 16 bytes per thread and store; element by element a wavefront's request was 128 bytes (us, that | this: 5 rows of 2048 2.7 | 2.3, 16 of 4096 3.6 | 2.25, int8 4.1 | 2.35, 4096 of 4096 15.6 | 11.1, 32768 of 4096 196 | 97).
template <bool VEC> __global__ __launch_bounds__(256) void embed_rows_kernel(int kind, const void *table, const _Float16 *scale, const int32_t *tokens, _Float16 *out, int dim, int vocab) {
  int tok = tokens[blockIdx.x];
  tok = tok < 0 ? 0 : (tok >= vocab ? vocab - 1 : tok);
  _Float16 *o = out + (size_t)blockIdx.x * dim;
  if (kind == JSGRAD_W_F16) {
    const _Float16 *src = (const _Float16 *)table + (size_t)tok * dim;
    if constexpr (VEC) {
      for (int i = threadIdx.x * 8; i < dim; i += 256 * 8) *(h8_t *)(o + i) = *(const h8_t *)(src + i);
    } else {
      for (int i = threadIdx.x; i < dim; i += 256) o[i] = src[i];
    }
  } else {
    const int8_t *src = (const int8_t *)table + (size_t)tok * dim;
    const float s = (float)scale[tok];
    if constexpr (VEC) {
      for (int i = threadIdx.x * 8; i < dim; i += 256 * 8) {
        const uint2 c = *(const uint2 *)(src + i);
        h8_t v;
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = mul_rn16((float)(int8_t)((e < 4 ? c.x : c.y) >> (8 * (e & 3))), s);
        *(h8_t *)(o + i) = v;
      }
    } else {
      for (int i = threadIdx.x; i < dim; i += 256) o[i] = mul_rn16((float)src[i], s);
    }
  }
}

// RMSNorm.call (nn/index.ts:586-588), one block per row.  A thread keeps its 16-byte chunks of the row (and of the weight)
// in registers between the sum of squares and the scaling: one round of loads.  CHUNKS 0: longer rows, in two passes.
template <int THREADS, int CHUNKS>
__global__ __launch_bounds__(THREADS) void rmsnorm_rows_kernel(const _Float16 *x, const _Float16 *w, _Float16 *y, int d, float eps, float inv_d) {
  constexpr int NW = THREADS / 64;
  __shared__ float red[NW];
  auto total = [&](float ss) {
    ss = wave_sum(ss);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    float t[NW];
#pragma unroll
    for (int i = 0; i < NW; i++) t[i] = red[i];
#pragma unroll
    for (int n = NW / 2; n > 0; n /= 2)
#pragma unroll
      for (int i = 0; i < n; i++) t[i] = t[2 * i] + t[2 * i + 1];
    return t[0];
  };
  const _Float16 *xr = x + (size_t)blockIdx.x * d;
  _Float16 *yr = y + (size_t)blockIdx.x * d;
  float ss = 0.0f;
  if constexpr (CHUNKS > 0) {
    h8_t xv[CHUNKS] = {}, wv[CHUNKS] = {};
#pragma unroll
    for (int c = 0; c < CHUNKS; c++) {
      const int i = (threadIdx.x + c * THREADS) * 8;
      if (i < d) { xv[c] = *(const h8_t *)(xr + i); wv[c] = *(const h8_t *)(w + i); }
    }
#pragma unroll
    for (int c = 0; c < CHUNKS; c++)
#pragma unroll
      for (int e = 0; e < 8; e++) { const float f = (float)xv[c][e]; ss = fmaf(f, f, ss); }
    const float r = __fsqrt_rn(__fdiv_rn(1.0f, __fadd_rn(__fmul_rn(total(ss), inv_d), eps)));
#pragma unroll
    for (int c = 0; c < CHUNKS; c++) {
      const int i = (threadIdx.x + c * THREADS) * 8;
      if (i < d) {
        h8_t o;
#pragma unroll
        for (int e = 0; e < 8; e++) o[e] = (_Float16)__fmul_rn(rn16(__fmul_rn((float)xv[c][e], r)), (float)wv[c][e]);
        *(h8_t *)(yr + i) = o;
      }
    }
  } else {
    for (int i = threadIdx.x; i < d; i += THREADS) { const float f = (float)xr[i]; ss = fmaf(f, f, ss); }
    const float r = __fsqrt_rn(__fdiv_rn(1.0f, __fadd_rn(__fmul_rn(total(ss), inv_d), eps)));
    for (int i = threadIdx.x; i < d; i += THREADS) {
      const float v = rn16(__fmul_rn((float)xr[i], r));
      yr[i] = (_Float16)__fmul_rn(v, (float)w[i]);
    }
  }
}

// Tensor.argmax (tensor.ts:2314-2320) of every row: lowest index among the maxima.  One block per row.  VEC: rows of whole
// 16-byte pieces; a thread asks for eight pieces at once, keeps the first whose maximum is the largest and looks for the element in it
// at the end.
template <bool VEC> __global__ __launch_bounds__(1024) void argmax_rows_kernel(const _Float16 *x, int n, int32_t *out) {
  __shared__ float vmax[16];
  __shared__ int imax[16];
  const _Float16 *xr = x + (size_t)blockIdx.x * n;
  float best = -INFINITY;
  int bi = 0x7fffffff;
  auto merge = [&](float ov, int oi) { if (ov > best || (ov == best && oi < bi)) { best = ov; bi = oi; } };
  if constexpr (VEC) {
    constexpr int U = 8;
    const int pieces = n / 8;
    h8_t bv = {};
    int bp = -1;                                              // the first piece whose maximum is the best so far, and its elements
    for (int p0 = threadIdx.x; p0 < pieces; p0 += U * 1024) {
      h8_t v[U];
#pragma unroll
      for (int u = 0; u < U; u++) v[u] = *(const h8_t *)(xr + (size_t)min(p0 + u * 1024, pieces - 1) * 8);   // the last piece again changes nothing
#pragma unroll
      for (int u = 0; u < U; u++) {
        float m = (float)v[u][0];
#pragma unroll
        for (int e = 1; e < 8; e++) m = fmaxf(m, (float)v[u][e]);
        if (m > best || (bp < 0 && m == best)) { best = m; bv = v[u]; bp = min(p0 + u * 1024, pieces - 1); }
      }
    }
    if (bp >= 0)
#pragma unroll
      for (int e = 7; e >= 0; e--)
        if ((float)bv[e] == best) bi = bp * 8 + e;
  } else {
    for (int i = threadIdx.x; i < n; i += 1024) merge((float)xr[i], i);
  }
  for (int off = 32; off > 0; off >>= 1) merge(__shfl_xor(best, off), __shfl_xor(bi, off));
  if ((threadIdx.x & 63) == 0) { vmax[threadIdx.x >> 6] = best; imax[threadIdx.x >> 6] = bi; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 16; w++) merge(vmax[w], imax[w]);
    out[blockIdx.x] = bi == 0x7fffffff ? n : bi;
  }
}

}  // namespace jsg

using namespace jsg;

extern "C" {

int jsgrad_hip_attn_prefill(const void *q, const void *cache_k, const void *cache_v, void *out, int batch, int seq_len, int start_pos, int n_heads,
                            int n_kv_heads, int head_dim, int max_context) {
  JSG_READY();
  JSG_REQUIRE(q && cache_k && cache_v && out, "jsgrad_hip_attn_prefill: null pointer argument");
  JSG_REQUIRE(batch > 0 && batch <= 65535 && seq_len > 0, "jsgrad_hip_attn_prefill: batch %d, seq_len %d", batch, seq_len);
  JSG_REQUIRE(n_heads > 0 && n_heads <= 65535 && n_kv_heads > 0 && n_heads % n_kv_heads == 0, "jsgrad_hip_attn_prefill: n_heads %d / n_kv_heads %d", n_heads, n_kv_heads);
  JSG_REQUIRE(head_dim == 64 || head_dim == 128, "jsgrad_hip_attn_prefill: head_dim %d (64 and 128 are built)", head_dim);
  JSG_REQUIRE(start_pos >= 0 && start_pos + seq_len <= max_context, "jsgrad_hip_attn_prefill: positions [%d, %d) outside the cache of %d", start_pos,
              start_pos + seq_len, max_context);
  PrefillAttnArgs a = {};
  a.q = (const _Float16 *)q; a.cache_k = (const _Float16 *)cache_k; a.cache_v = (const _Float16 *)cache_v; a.out = (_Float16 *)out;
  a.S = seq_len; a.start_pos = start_pos; a.max_context = max_context;
  const int n_rep = n_heads / n_kv_heads;
  a.n_rep = divisor(n_rep); a.n_kv_heads = divisor(n_kv_heads);
  JSG_REQUIRE((size_t)seq_len * n_rep < (size_t)1 << 30, "jsgrad_hip_attn_prefill: seq_len %d", seq_len);
  a.scale_log2 = (float)(1.0 / sqrt((double)head_dim)) * 1.4426950408889634f;
  a.tiles = (seq_len * n_rep + PF_QROWS - 1) / PF_QROWS;
  a.tile_div = divisor(a.tiles);
  a.pairs = batch * n_kv_heads;
  a.parts = 1;
  // Fewer blocks than half of what the chip holds (two per CU): the keys are cut into parts.  Not during a graph capture,
  // where nothing can be allocated.
  const size_t blocks = (size_t)a.tiles * a.pairs;
  Workspace sums;
  if (!state().capturing && blocks * 2 <= (size_t)2 * state().cu_count && blocks * 4 <= PF_COUNTERS) {
    // A tile takes 0.7-0.9 us and folding a part about as long, one after the other: least at about sqrt(tiles) parts, and nothing
    // to gain below eight.  (57 positions behind 1024, 24 heads of 128: 24.6 / 18.6 / 15.5 / 17.1 us in 1 / 2 / 4 / 8 parts;
    // 371 positions of 32 heads of 64: 9.3 / 9.1 / 12.2 in 1 / 2 / 4.)
    const int fill = (int)((size_t)2 * state().cu_count / blocks), mean_tiles = (start_pos + seq_len / 2) / PF_KEYS + 1;
    if (mean_tiles >= 8) a.parts = fill < (int)sqrtf((float)mean_tiles) ? fill : (int)sqrtf((float)mean_tiles);
  }
  if (a.parts > 1 && !sums.get(blocks * a.parts * 4 * (head_dim / 2 + 4) * 64 * sizeof(float))) a.parts = 1;
  if (a.parts > 1) {
    static int *counters = nullptr;
    if (!counters) JSG_HIP(hipGetSymbolAddress((void **)&counters, HIP_SYMBOL(pf_counters)));
    a.ws = (float *)sums.p;
    a.counters = counters;
  }
  const dim3 grid((unsigned)(blocks * a.parts)), block(PF_THREADS);
  if (head_dim == 64) JSG_LAUNCH(PROF_ATTN_PREFILL, attn_prefill_kernel<64>, grid, block, 0, a);
  else JSG_LAUNCH(PROF_ATTN_PREFILL, attn_prefill_kernel<128>, grid, block, 0, a);
  return 0;
}

int jsgrad_hip_embed_rows(int kind, const void *table, const void *scale, const int32_t *tokens, int rows, void *out, int dim, int vocab) {
  JSG_READY();
  JSG_REQUIRE(table && tokens && out, "jsgrad_hip_embed_rows: null pointer argument");
  JSG_REQUIRE(kind == JSGRAD_W_F16 || (kind == JSGRAD_W_I8 && scale), "jsgrad_hip_embed_rows: table kind %d (fp16, or int8 with row scales)", kind);
  JSG_REQUIRE(rows > 0 && dim > 0 && vocab > 0, "jsgrad_hip_embed_rows: rows %d, dim %d, vocab %d", rows, dim, vocab);
  const bool vec = dim % 8 == 0 && (uintptr_t)table % (kind == JSGRAD_W_F16 ? 16 : 8) == 0 && (uintptr_t)out % 16 == 0;
  if (vec) JSG_LAUNCH(PROF_EMBED, embed_rows_kernel<true>, dim3(rows), dim3(256), 0, kind, table, (const _Float16 *)scale, tokens, (_Float16 *)out, dim, vocab);
  else JSG_LAUNCH(PROF_EMBED, embed_rows_kernel<false>, dim3(rows), dim3(256), 0, kind, table, (const _Float16 *)scale, tokens, (_Float16 *)out, dim, vocab);
  return 0;
}

int jsgrad_hip_rmsnorm_rows(const void *x, const void *w, void *y, int rows, int d, float eps) {
  JSG_READY();
  JSG_REQUIRE(x && w && y && rows > 0 && d > 0, "jsgrad_hip_rmsnorm_rows: bad argument");
  const float inv_d = (float)(1.0 / (double)d);
  // A few rows are one latency chain, shortest with one chunk per thread; thousands of rows fill the chip either way, and larger blocks leave gaps.
  // us, 256 threads of up to four chunks | one chunk each: 16 x 3072 2.12 | 1.84, 16 x 4096 2.19 | 1.90, 32768 x 3072 69.8 | 73.7, 16 x 8192 2.78 | 2.14, 371 x 8192
  // 4.55 | 4.15, 4096 x 8192 24.3 | 26.5; a step of 16 sequences of the 8B int8 shape (65 norms) 3127 | 3106.
#define JSG_NORM(THREADS, CHUNKS)                                                                                       \
  JSG_LAUNCH(PROF_RMSNORM, (rmsnorm_rows_kernel<THREADS, CHUNKS>), dim3(rows), dim3(THREADS), 0, (const _Float16 *)x,    \
             (const _Float16 *)w, (_Float16 *)y, d, eps, inv_d)
  if (d % 8 == 0 && d <= 2048) JSG_NORM(256, 1);
  else if (d % 8 == 0 && d <= 8192 && rows > 1024) JSG_NORM(256, 4);
  else if (d % 8 == 0 && d <= 4096) JSG_NORM(512, 1);
  else if (d % 8 == 0 && d <= 8192) JSG_NORM(1024, 1);
  else JSG_NORM(256, 0);
#undef JSG_NORM
  return 0;
}

int jsgrad_hip_argmax_rows(const void *logits, int rows, int n, int32_t *tokens_out) {
  JSG_READY();
  JSG_REQUIRE(logits && tokens_out && rows > 0 && n > 0, "jsgrad_hip_argmax_rows: bad argument");
  // 16 rows, us, element by element | in pieces: 512 3.9 | 4.1, 4096 4.2 | 4.5, 8192 4.9 | 5.4, 16384 6.2 | 5.4, 32000 8.7 | 5.4, 128256 24.4 | 6.9
  if (n > 8192 && n % 8 == 0 && (uintptr_t)logits % 16 == 0) JSG_LAUNCH(PROF_ARGMAX, argmax_rows_kernel<true>, dim3(rows), dim3(1024), 0, (const _Float16 *)logits, n, tokens_out);
  else JSG_LAUNCH(PROF_ARGMAX, argmax_rows_kernel<false>, dim3(rows), dim3(1024), 0, (const _Float16 *)logits, n, tokens_out);
  return 0;
}

}  // extern "C"
