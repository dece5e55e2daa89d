// Decode-time grouped-query attention for MANY sequences at once (jsgrad_hip_attn_decode_batch): the streaming form of the
// work item of attention_core.h.
//
// With one sequence a launch has a few dozen items and waits for the chain of dependent steps inside each, so an item there
// is worked on by 16 wavefronts that request all their rows up front (attention_core.h).  With 16 sequences a launch moves over
// a hundred megabytes: what counts is that every CU keeps requests in flight all the time, that the arithmetic behind them stays small, and that
// little comes behind the last row.  Here the four wavefronts of a block walk their own tiles of rows, each with a running maximum per 16 lanes,
// and meet once, at the end: a tile's K rows are asked for as soon as the last tile's scores are made, its V rows as soon as those are used.
// Scores come from the matrix unit (products of halves, float sums, as the packed dot product has them); the weights stay float and multiply V in
// the vector unit.  The last block of a kv head to finish (an agent-scope counter) merges the blocks.  The arithmetic is that of attention_core.h
// (float scores, the reference's polynomial exp2, float P.V) in another order and against running maxima, so the float sums differ in their last bits.
// Against chunks that were scored, weighted and summed in three steps between barriers, five blocks to a CU (dot products and lane folds in the
// vector unit: half of a SIMD's time), us: 8 kv heads of 128, 4 query heads each, 16 sequences at 2050 positions 34.3 -> 29.0 (134 MB, which blocks that
// only read take 24.5 for), at 300 12.0 -> 9.3, 32 at 1000 34.7 -> 27.6, 5 at 300 9.8 -> 7.5; heads of 64, 16 at 2050 23.4 -> 19.2, 5 at 300
// 8.2 -> 6.8.  Two tiles on their way instead of one: 30.5 -> 31.5; 8 wavefronts: 5 sequences at 300 7.5 -> 8.5.
#pragma once
#include <type_traits>

#include "attention_core.h"

namespace jsg {

constexpr int ATT_STREAM_BLOCKS = 64;   // of a (sequence, kv head) pair: what the workspace has room for, and the merge a lane for each

// Blocks for T visible positions of a (sequence, kv head) pair, of at most `most`.  One block takes the pair in `rounds` round trips of 0.8 us, n
// blocks in an n-th of them, and a merge: 2 us, and more with n.  So n blocks are worth it where they save three rounds, and n^2 = 6 rounds is the most.
// us, 1 | 2 | 3 | 4 | 6 | 8 | 12 | 16 blocks, head_dim 128: 2 sequences 2048 positions 30.4 | 19.2 | 15.4 | 13.1 | 11.3 | 10.5 | 10.4 | 11.5, 5 sequences
// 90 5.8 | 6.7 | 6.9 | 6.9 | 7.1 | 7.6 | 7.7 | 8.5, 300 8.4 | 8.3 | 7.9 | 7.8 | 7.6 | 7.9 | 8.3 | 8.7, 1000 17.8 | 12.8 | 11.5 | 10.2 | 9.7 | 10.9 | 11.1 | 11.9;
// head_dim 64: 5 sequences 300 6.7 | 7.3 | 6.7 | 6.8 | 6.9 | 7.1 | 7.2 | 7.4, 600 8.2 | 8.3 | 7.6 | 7.6 | 7.3 | 7.3 | 7.4 | 7.6.
// split_from: there are about as many pairs as compute units (attention.hip), so that parts of a pair wait for each other's loads, not only for their
// own: only from that many rounds on, and n^2 = 3 rounds.
template <int HD, int NW> __device__ __forceinline__ int att_stream_blocks(int T, int most, int split_from) {
  constexpr int ROUND = NW * (HD == 64 ? 32 : 16);
  const int rounds = (T + ROUND - 1) / ROUND;
  if (rounds < split_from) return 1;
  const int n = min(min(most, rounds), (int)__builtin_amdgcn_sqrtf((split_from ? 3.0f : 6.0f) * (float)rounds));
  return rounds - (rounds + n - 1) / n >= 3 ? n : 1;
}
template <int I, int N, typename F> __device__ __forceinline__ void static_for(F &&f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>());
    static_for<I + 1, N>(f);
  }
}
// lane N of every 16-lane row to all lanes of the row; upper: to the row's upper eight lanes only, the others keep `keep`
template <int N> __device__ __forceinline__ float row_bcast(float v) { return dpp_f<0x150 + N>(v); }
template <int N> __device__ __forceinline__ float row_bcast_upper(float keep, float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(keep), __float_as_int(v), 0x150 + N, 0xf, 0xc, false));
}

template <int HD, int NREP, int NW> struct AttnStream {
  static constexpr int G = HD / 8;             // lanes per V row: 16 bytes each
  static constexpr int HALVES = 16 / G;        // V rows under a 16-lane row: 1 or 2
  static constexpr int TILE = 16 * HALVES;     // rows of a wavefront's tile
  static constexpr int KS = HD / 32;           // matrix instructions per 16 rows
  // Column c of the scores is head c % HP: every lane has the scores of four rows of one head, and with up to four heads four lanes have the same
  // ones, so that each takes the exponential of one of them (row `slot`): row r's weight for head j lies in lane j + HP * (r % SLOTS), value r / SLOTS.
  static constexpr int HP = NREP == 3 ? 4 : NREP;
  static constexpr int SLOTS = HP == 8 ? 2 : 4, EX = 4 / SLOTS;
  static constexpr int NV = NREP * 8;          // sums of a lane
  static_assert(HD == 64 || HD == 128, "one or two V rows per 16 lanes");
  static_assert(HP == 1 || HP == 2 || HP == 4 || HP == 8, "heads divide the columns");
  struct Smem {
    float sc[NREP][ATT_STREAM_BLOCKS];         // the merge's weights
    float o_part[NW][NREP * HD];
    float m[NREP][NW], l[NREP][NW], w[NREP][NW];
    float m_sh[NREP], l_sh[NREP];
    int is_last;
  };

  // Item `split` of n_active(T) of kv head g: the tiles split * NW + wavefront, + n * NW, ..
  // Must be called by every thread of the block (it contains barriers).
  template <typename Blocks> __device__ static void item(const AttnArgs &a, Smem &sm, int g, int split, Blocks blocks) {
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr int nthreads = NW * 64;
    const int l16 = lane & 15, lq = lane >> 4, sub = l16 % G, half = l16 / G, slot = l16 / HP % SLOTS;
    const size_t row_stride = (size_t)a.n_kv_heads * HD;
    const _Float16 *const kbase = (const _Float16 *)a.cache_k + (size_t)g * HD + lq * 8;
    const _Float16 *const vbase = (const _Float16 *)a.cache_v + (size_t)g * HD + sub * 8;

    h8_t qf[KS];
    {
      const _Float16 *const qp = (const _Float16 *)a.q + (size_t)(g * NREP + min(l16 % HP, NREP - 1)) * HD + lq * 8;
#pragma unroll
      for (int s = 0; s < KS; s++) qf[s] = *(const h8_t *)(qp + s * 32);
    }
    // The tile on its way.  Rows past `last` are that one again: every load is asked for, so that the compiler can count the later ones
    // when it waits for one (behind a branch it would wait for all of them).
    h8_t kf[HALVES][KS];
    u4_t vf[4];
    auto load_k = [&](int tb, int last) {
#pragma unroll
      for (int h = 0; h < HALVES; h++) {
        const _Float16 *const from = kbase + (size_t)min(tb + h * 16 + l16, last) * row_stride;
#pragma unroll
        for (int s = 0; s < KS; s++) kf[h][s] = *(const h8_t *)(from + s * 32);
      }
    };
    auto load_v = [&](int tb, int last) {
#pragma unroll
      for (int r = 0; r < 4; r++) vf[r] = *(const u4_t *)(vbase + (size_t)min(tb + half * 16 + lq * 4 + r, last) * row_stride);
    };
    // the first one before the position has arrived: what lies behind it is masked.  Not where blocks that may have nothing to do come on top of a full
    // chip (33 sequences at 60 of 4000 positions, us: 9.5, without their loads 5.7; one block per pair 5.5)
    if (split != 0 && a.split_from && split >= blocks(a.st[1] + 1)) return;
    int tb = (split * NW + wave) * TILE;
    load_k(tb, a.max_context - 1);
    load_v(tb, a.max_context - 1);
    const int pos = __builtin_amdgcn_readfirstlane(a.st[1]);
    if (pos < 0 || pos >= a.max_context) return;
    const int T = pos + 1, n_active = blocks(T), stride = n_active * NW * TILE;
    if (split >= n_active) return;

    float o[NREP][8], m = -INFINITY, l = 0.0f;                // m, l: of head l16 % HP over the rows of this lane quarter; l: of its slots
#pragma unroll
    for (int j = 0; j < NREP; j++)
#pragma unroll
      for (int e = 0; e < 8; e++) o[j][e] = 0.0f;
    for (; tb < T; tb += stride) {
      float s[HALVES][4];
#pragma unroll
      for (int h = 0; h < HALVES; h++) {
        // Summed as a tree, like a tile's weighted rows below: results that are not the nearest half of the float64 ones, 16 sequences of 2050 positions,
        // heads of 128: as one chain each 0.26 %, the chunked form 0.20 %, so 0.18 %; 16 of 2000, heads of 64, 0.22 | 0.19 | 0.18 %.
        f4_t acc[KS];
#pragma unroll
        for (int k = 0; k < KS; k++) acc[k] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[h][k], qf[k], f4_t{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
        for (int w = KS / 2; w > 0; w /= 2)
#pragma unroll
          for (int k = 0; k < w; k++) acc[k] += acc[k + w];
#pragma unroll
        for (int r = 0; r < 4; r++) s[h][r] = acc[0][r] * a.scale;
      }
      load_k(tb + stride, T - 1);
      if (tb + TILE > T) {                                   // rows past the end: no weight, and nothing that a weight of zero could meet
#pragma unroll
        for (int r = 0; r < 4; r++) {
#pragma unroll
          for (int h = 0; h < HALVES; h++)
            if (tb + h * 16 + lq * 4 + r >= T) s[h][r] = -INFINITY;
          if (tb + half * 16 + lq * 4 + r >= T) vf[r] = u4_t{0, 0, 0, 0};
        }
      }
      float mx = m;
#pragma unroll
      for (int h = 0; h < HALVES; h++) mx = fmaxf(fmaxf(fmaxf(mx, s[h][0]), fmaxf(s[h][1], s[h][2])), s[h][3]);
      if (__builtin_amdgcn_ballot_w64(mx != m) != 0) {        // rare behind the first tiles
        const float f = m == -INFINITY ? 0.0f : exp_f32(m - mx);
        l *= f;
        static_for<0, NREP>([&](auto I) {
          constexpr int j = decltype(I)::value;
          const float fj = row_bcast<j>(f);
#pragma unroll
          for (int e = 0; e < 8; e++) o[j][e] *= fj;
        });
        m = mx;
      }
      const float base = m == -INFINITY ? 0.0f : m;           // no row yet: weights of zero
      float p[HALVES][EX];
#pragma unroll
      for (int h = 0; h < HALVES; h++)
#pragma unroll
        for (int x = 0; x < EX; x++) {
          float mine = s[h][x * SLOTS];
#pragma unroll
          for (int i = 1; i < SLOTS; i++) mine = slot == i ? s[h][x * SLOTS + i] : mine;
          p[h][x] = exp_f32(mine - base);
          l += p[h][x];
        }
      static_for<0, NREP>([&](auto I) {
        constexpr int j = decltype(I)::value;
        float pj[4];
        static_for<0, 4>([&](auto R) {
          constexpr int r = decltype(R)::value, from = j + HP * (r % SLOTS);
          pj[r] = row_bcast<from>(p[0][r / SLOTS]);
          if constexpr (HALVES == 2) pj[r] = row_bcast_upper<from>(pj[r], p[1][r / SLOTS]);
        });
#pragma unroll
        for (int e = 0; e < 8; e++) {
          float sum = pj[0] * (float)as_h2(vf[0][e / 2])[e % 2];
#pragma unroll
          for (int r = 1; r < 4; r++) sum = fmaf(pj[r], (float)as_h2(vf[r][e / 2])[e % 2], sum);
          o[j][e] += sum;
        }
      });
      load_v(tb + stride, T - 1);
    }

    // The wavefront's partial sums per head, against its maximum.  Lane quarters trade halves: a sum of what both hold costs one exchange for two
    // values, and in the end quarter lq has values [lq * NV / 4, + NV / 4) of the lane group's NV.
    {
      const float M = max_xor32(max_xor16(m)), f = m == -INFINITY ? 0.0f : exp_f32(m - M);
      l = add_xor32(add_xor16(l * f));
      if constexpr (HP * SLOTS == 16) l += dpp_f<0x128>(l);   // row_ror: the slots of a head repeat after HP * SLOTS lanes
      if constexpr (HP * SLOTS == 8 || HP == 4) l += dpp_f<0x124>(l);
      if constexpr (HP <= 2) l += dpp_f<0x122>(l);
      if constexpr (HP == 1) l += dpp_f<0x121>(l);
      if (lane < NREP) { sm.m[lane][wave] = M; sm.l[lane][wave] = l; }
      float v[NV / 2], u[NV / 4];
      static_for<0, NREP>([&](auto I) {
        constexpr int j = decltype(I)::value;
        const float fj = row_bcast<j>(f);
#pragma unroll
        for (int e = 0; e < 8; e++) o[j][e] *= fj;
      });
#pragma unroll
      for (int i = 0; i < NV / 2; i++) {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(o[i / 8][i % 8]), __float_as_uint(o[(i + NV / 2) / 8][(i + NV / 2) % 8]), false, false);
        v[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
      }
#pragma unroll
      for (int i = 0; i < NV / 4; i++) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[i]), __float_as_uint(v[i + NV / 4]), false, false);
        u[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
        if constexpr (HALVES == 2) u[i] += dpp_f<0x128>(u[i]);
      }
      if (half == 0)
#pragma unroll
        for (int i = 0; i < NV / 4; i++) sm.o_part[wave][(lq * (NV / 4) + i) * G + sub] = u[i];
    }
    lds_barrier();
    // the block's wavefronts against its maximum
    if (tid < NREP * NW) {
      const int j = tid / NW;
      float M = sm.m[j][0];
#pragma unroll
      for (int w = 1; w < NW; w++) M = fmaxf(M, sm.m[j][w]);
      const float mw = sm.m[j][tid % NW];
      sm.w[j][tid % NW] = mw == -INFINITY ? 0.0f : exp_f32(mw - M);
      sm.m_sh[j] = M;
    }
    lds_barrier();
    // Value i of the kv head's NREP * HD, in the order they are kept in here: head i / G / 8, element i % G * 8 + i / G % 8
    auto part_sum = [&](int i) {
      float v = 0.0f;
#pragma unroll
      for (int w = 0; w < NW; w++) v = fmaf(sm.o_part[w][i], sm.w[i / G / 8][w], v);
      return v;
    };
    auto weight_sum = [&](int j) {
      float L = 0.0f;
#pragma unroll
      for (int w = 0; w < NW; w++) L = fmaf(sm.l[j][w], sm.w[j][w], L);
      return L;
    };
    // P.V sum times 1 / (sum of the weights), softmax's e * (1 / sum) (tensor.ts:2211-2214)
    auto store_out = [&](int i, float O, float inv) {
      ((_Float16 *)a.out)[(size_t)g * NREP * HD + i / G / 8 * HD + i % G * 8 + i / G % 8] = Act<_Float16>::rn(O * inv);   // the cast of the P.V result
    };
    if (n_active == 1) {                                      // nothing to merge
      for (int i = tid; i < NREP * HD; i += nthreads) store_out(i, part_sum(i), 1.0f / weight_sum(i / G / 8));
      return;
    }
    float *const base = a.partial + (size_t)g * a.nsplit * NREP * (HD + 2), *const mine = base + (size_t)split * NREP * (HD + 2);
    for (int i = tid; i < NREP * HD; i += nthreads) st_coherent(&mine[i], part_sum(i));
    if (tid < NREP) {
      st_coherent(&mine[NREP * HD + tid], sm.m_sh[tid]);
      st_coherent(&mine[NREP * (HD + 1) + tid], weight_sum(tid));
    }

    // ---- publish, and let the last block of this kv head merge
    __syncthreads();  // every coherent store of the block has been acknowledged
    if (tid == 0) {
      int old = __hip_atomic_fetch_add(&a.counters[g], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      sm.is_last = (old == n_active - 1);
    }
    __syncthreads();
    if (!sm.is_last) return;
    // A value's partial results are asked for together with the (m, l) that their weights are made of, MB blocks at a time: one round trip.
    // One wavefront per query head makes the weights; block lane < n_active <= ATT_STREAM_BLOCKS.
    auto part = [&](int i, int s) { return ld_coherent(base + (size_t)min(s, n_active - 1) * NREP * (HD + 2) + i); };
    constexpr int PER = (NREP * HD + nthreads - 1) / nthreads;
    auto merge = [&](auto I) {
      constexpr int MB = decltype(I)::value;
      float p[PER][MB], O[PER];
      auto ask = [&](int s0) {
#pragma unroll
        for (int q = 0; q < PER; q++)
#pragma unroll
          for (int u = 0; u < MB; u++) p[q][u] = part(min(tid + q * nthreads, NREP * HD - 1), s0 + u);
      };
      ask(0);
      for (int j = wave; j < NREP; j += NW) {
        const float ms = part(NREP * HD + j, lane), ls = part(NREP * (HD + 1) + j, lane);
        const float M = wave_max(lane < n_active ? ms : -INFINITY), w = lane < n_active ? exp_f32(ms - M) : 0.0f;
        const float L = wave_sum(lane < n_active ? ls * w : 0.0f);
        sm.sc[j][lane] = w;
        if (lane == 0) sm.l_sh[j] = 1.0f / L;
      }
      lds_barrier();
#pragma unroll
      for (int q = 0; q < PER; q++) O[q] = 0.0f;
      for (int s0 = 0; s0 < n_active; s0 += MB) {
        if (s0) ask(s0);
#pragma unroll
        for (int q = 0; q < PER; q++)
#pragma unroll
          for (int u = 0; u < MB; u++)
            if (s0 + u < n_active) O[q] = fmaf(p[q][u], sm.sc[min(tid + q * nthreads, NREP * HD - 1) / G / 8][s0 + u], O[q]);
      }
#pragma unroll
      for (int q = 0; q < PER; q++)
        if (tid + q * nthreads < NREP * HD) store_out(tid + q * nthreads, O[q], sm.l_sh[(tid + q * nthreads) / G / 8]);
    };
    if (n_active <= 2) merge(std::integral_constant<int, 2>());
    else if (n_active <= 4) merge(std::integral_constant<int, 4>());
    else merge(std::integral_constant<int, 8>());
    if (tid == 0) __hip_atomic_store(&a.counters[g], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
};

}  // namespace jsg
