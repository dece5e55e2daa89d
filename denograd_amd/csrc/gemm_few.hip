// At most 16 rows of fp16 activations (batched decode), fp16 or int8 weights: y[M][N] = x[M][K] . W[N][K]^T, float accumulation, fp16
// out; what the reference computes is in gemm.hip.
//
// The launch is bound by reading W once.  A block of eight wavefronts stays on its compute unit and walks tiles of 16 weight rows;
// the wavefronts split K, and a wavefront's share of x (16 rows of K / 8 elements, at most 128 registers) is in operand layout in
// its registers for the whole launch, so x costs one read per block, and no barrier stands between a wavefront and its weights.
// Those come by direct global-to-LDS loads into a ring that belongs to the wavefront (16 KiB: 128 KiB of every compute unit's LDS
// are on their way), 256 to 512 contiguous bytes of a row at a time: asked for in operand layout (64 bytes of each of 16 rows per
// load) the same bytes take a quarter longer.  Where the ring has room for it, x comes through its last slots.  Per tile the eight
// partial sums are added through LDS in wavefront order.
// Tiles that are left after whole rounds over the compute units are dealt as halves of eight rows where that is enough for
// everybody (w1|w3 of 14336 rows: 896 tiles on 256 units are 3.5 rounds instead of 4).
#include <type_traits>

#include "gemm.h"

namespace jsg {

constexpr int FW_WAVES = 8, FW_THREADS = FW_WAVES * 64;

template <int KIND, int EPI, int SB> struct FwShape {
  static constexpr int SLOT = 16 * SB;                        // bytes of a step: 16 rows x SB bytes
  static constexpr int LOADS = SB / 64;                       // direct loads of 1 KiB per step
  static constexpr int SCALE = KIND == JSGRAD_W_I8 ? 256 : 0; // a slot of row scales (a 4-byte load of all lanes fills 256 bytes)
  static constexpr int RED = (EPI == GEPI_SWIGLU ? 2 : 1) * FW_WAVES * 1024;   // the wavefronts' sums
  static constexpr int FIT = (160 * 1024 - RED) / (FW_WAVES * (SLOT + SCALE));
  static constexpr int NS = FIT < 4 ? FIT : 4;                // steps on their way
  static constexpr int RING = NS * (SLOT + SCALE);            // per wavefront
  static constexpr int LDS = FW_WAVES * RING + RED;
  static_assert(NS >= 2, "one step arrives while another is used");
};

// K = 8 wavefronts x PARTS steps x SB bytes of a weight row.  NORM as a kernel of its own: with the question asked inside the one without a norm was slower as
// well (us, w1|w3 of 2 / 12 rows x 8192 x 2048 15.9 / 16.5, now 15.0 / 15.1).
template <int KIND, int EPI, int SB, int PARTS, bool LONG, bool NORM> __global__ __launch_bounds__(FW_THREADS, 2) void few_rows_kernel(GemmArgs a, int tiles) {
  typedef FwShape<KIND, EPI, SB> S;
  constexpr int NMAT = EPI == GEPI_SWIGLU ? 2 : 1, LOADS = S::LOADS, NS = S::NS;
  constexpr int KB = KIND == JSGRAD_W_F16 ? 2 : 1;            // bytes of a weight
  constexpr int NFR = SB / 64;                                // 16-byte fragment reads of a lane per step
  constexpr int MPR = KIND == JSGRAD_W_F16 ? 1 : 2;           // matrix instructions per fragment read
  constexpr int NF = PARTS * NFR * MPR;                       // x fragments
  static_assert(NF <= (NORM ? 16 : 32), "x fits 128 registers; with the norm's weights it takes twice as many");
  extern __shared__ __align__(16) unsigned char few_lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, lq = lane >> 4;
  const int G = gridDim.x;
  const uint32_t row_bytes = (uint32_t)a.K * KB, k_first = (uint32_t)wave * PARTS * SB;

  // Units of this block: whole tiles blockIdx.x, + G, ..; what is left after whole rounds as halves, if they go round
  const int whole = tiles / G, left = tiles - whole * G;
  const bool halves = 2 * left <= G;
  const bool more = (int)blockIdx.x < (halves ? 2 * left : left);
  const int units = whole + (more ? 1 : 0), n_steps = units * NMAT * PARTS;
  auto is_half = [&](int u) { return halves && u == whole; };
  auto first_row = [&](int u) { return u < whole || !halves ? ((int)blockIdx.x + u * G) * 16 : whole * G * 16 + (int)blockIdx.x * 8; };
  auto place = [&](int n, int q, const void *&w, const _Float16 *&s, int &row) {   // a tile never straddles two matrices
    if constexpr (EPI == GEPI_SWIGLU) { w = q ? a.w1 : a.w0; s = q ? a.s1 : a.s0; row = n; }
    else if constexpr (EPI == GEPI_ROPE_KV) {
      const int which = n < a.n0 ? 0 : (n < a.n0 + a.n1 ? 1 : 2);
      w = which == 0 ? a.w0 : (which == 1 ? a.w1 : a.w2);
      s = which == 0 ? a.s0 : (which == 1 ? a.s1 : a.s2);
      row = which == 0 ? n : (which == 1 ? n - a.n0 : n - a.n0 - a.n1);
    } else { w = a.w0; s = a.s0; row = n; }
  };

  // A step's bytes lie in its slot row by row; 16-byte piece p of row r is kept at position p ^ swizzle(r), so that the 16
  // rows of a fragment read hit different banks.  Row 8 begins with load LOADS / 2: a half unit issues that many.
  auto swizzle = [](int r) { return SB % 256 == 0 ? r & 15 : (r >> 1) & 7; };
  uint32_t vo[LOADS];
#pragma unroll
  for (int j = 0; j < LOADS; j++) {
    const int o = j * 1024 + lane * 16, r = o / SB, p = (o % SB) / 16;
    vo[j] = (uint32_t)r * row_bytes + (uint32_t)(p ^ swizzle(r)) * 16;
  }
  unsigned char *const ring = few_lds + wave * S::RING;
  const uint32_t ring0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)ring;
  auto issue = [&](int s) {
    const int u = s / (NMAT * PARTS), q = s / PARTS % NMAT, part = s % PARTS;
    const void *w; const _Float16 *sc; int row;
    place(first_row(u), q, w, sc, row);
    const i4_t rw = dma_rsrc((const unsigned char *)w + (size_t)row * row_bytes);
    const uint32_t to = ring0 + (uint32_t)(s % NS) * (S::SLOT + S::SCALE), so = k_first + part * SB;
    const bool half = is_half(u);
#pragma unroll
    for (int j = 0; j < LOADS; j++)
      if (j < LOADS / 2 || !half) dma16_stream(rw, vo[j], so, to + j * 1024);
    if constexpr (KIND == JSGRAD_W_I8) dma4(dma_rsrc(sc + row), (uint32_t)(lane & (half ? 3 : 7)) * 4, 0, to + S::SLOT);
  };
  constexpr int FULL = LOADS + (KIND == JSGRAD_W_I8 ? 1 : 0), HALF = LOADS / 2 + (KIND == JSGRAD_W_I8 ? 1 : 0);
  // Wait until what was issued in front of the `steps` steps from s on has landed; those may stay in flight, and so may a store that went out behind
  // them (memory operations of a wavefront are counted in the order they were issued).
  auto arrived = [&](int s, auto steps, bool store) {
    constexpr int N = decltype(steps)::value;
    int behind = 0;
#pragma unroll
    for (int i = 0; i < N; i++)
      if (s + i < n_steps) behind += is_half((s + i) / (NMAT * PARTS)) ? HALF : FULL;
    if (N > 0 && behind >= N * FULL && store) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N * FULL + 1) : "memory");
    else if (N > 0 && behind >= N * FULL) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N * FULL) : "memory");
    else if (N > 1 && behind >= FULL) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(FULL) : "memory");
    else if (N > 0 && behind >= HALF) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(HALF) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  };

  // x first: fragment f of read i holds the K elements that a lane finds in its 16 bytes of the weight row
  float *const red = (float *)(few_lds + FW_WAVES * S::RING);  // [matrix][wavefront][16 x rows][16 weight rows]
  h8_t xf[NF];
  constexpr int XS = PARTS * MPR;                              // slots that the wavefront's share of x would fill
  auto norm_x = [&](const h8_t (&wf)[NORM ? NF : 1]) {         // in registers: sums over a wavefront's share, the eight shares through LDS in order
    float ss = 0.0f;
#pragma unroll
    for (int f = 0; f < NF; f++) ss = square_sum(xf[f], ss);
    ss = add_xor32(add_xor16(ss));
    if (lq == 0) red[wave * 256 + l16] = ss;
    lds_barrier();
    float tot = red[l16];
#pragma unroll
    for (int w = 1; w < FW_WAVES; w++) tot += red[w * 256 + l16];
    const float r = norm_factor(a, tot);
#pragma unroll
    for (int f = 0; f < NF; f++) xf[f] = norm_piece(xf[f], r, wf[f]);
    lds_barrier();                                            // the sums have been read
  };
  if constexpr (XS <= NS && !(LONG && NORM)) {
    // Through the last slots of the ring, which are free until their steps are asked for.  The compiler does not count direct loads: a load of x
    // to registers would be waited for with every step asked for behind it, and nothing would be on its way until they are used.
    const i4_t rx = dma_rsrc(a.x);
#pragma unroll
    for (int i = 0; i < XS; i++)
#pragma unroll
      for (int j = 0; j < LOADS; j++) {
        const int o = j * 1024 + lane * 16, r = o / SB, p = (o % SB) / 16;
        // Rows past the end: the last one again, or what the slot held, and never stored.  Steps of 256 bytes: a load is four rows, the last one of nobody's up
        // to 12 (us, 9 / 12 rows, with it | without: int8 4096 x 2048 4.6 / 4.6 | 4.4 / 4.4, wq|wk|wv of 3072 x 2048 4.4 / 4.5 | 4.2 / 4.3)
        if (j < LOADS / 2 || a.M > (SB == 256 && j == LOADS - 1 ? 12 : 8))
          dma16(rx, (uint32_t)min(r, a.M - 1) * (uint32_t)a.K * 2 + (uint32_t)(p ^ swizzle(r)) * 16, k_first * MPR + i * SB, ring0 + (NS - XS + i) * (S::SLOT + S::SCALE) + j * 1024);
      }
    // the norm's weights of the wavefront's share into its part of the sums' space: at most 1 KiB
    unsigned char *const nw = (unsigned char *)red + wave * 1024;
    if constexpr (NORM) dma16(dma_rsrc(a.norm_w), min((uint32_t)lane * 16, (uint32_t)(XS * SB) - 16), k_first * MPR, (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)nw);
#pragma unroll
    for (int i = 0; i < NS - XS; i++)
      if (i < n_steps) issue(i);
    arrived(0, std::integral_constant<int, NS - XS>(), false);
#pragma unroll
    for (int f = 0; f < NF; f++) {
      const int at = f / MPR * (64 * MPR) + f % MPR * 16;     // byte of the wavefront's share of a row, without the lane quarter's
      xf[f] = *(const h8_t *)(ring + (NS - XS + at / SB) * (S::SLOT + S::SCALE) + l16 * SB + ((at % SB / 16 + lq * MPR) ^ swizzle(l16)) * 16);
    }
    h8_t wf[NORM ? NF : 1];
    if constexpr (NORM)
#pragma unroll
      for (int f = 0; f < NF; f++) wf[f] = *(const h8_t *)(nw + f / MPR * (64 * MPR) + f % MPR * 16 + lq * (MPR * 16));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");        // x is in registers: its slots are filled
#pragma unroll
    for (int i = NS - XS; i < NS; i++)
      if (i < n_steps) issue(i);
    if constexpr (NORM) norm_x(wf);
  } else {
    const _Float16 *xr = a.x + (size_t)min(l16, a.M - 1) * a.K + k_first / KB + lq * (16 / KB);   // rows past the end: never stored
#pragma unroll
    for (int f = 0; f < NF; f++) xf[f] = *(const h8_t *)(xr + (f / MPR) * (64 / KB) + (f % MPR) * 8);
    if constexpr (NORM) {
      // using x waits for all loads before it and behind it: the first step goes out ahead of that and the others behind
      h8_t wf[NF];
      const _Float16 *wr = a.norm_w + k_first / KB + lq * (16 / KB);
#pragma unroll
      for (int f = 0; f < NF; f++) wf[f] = *(const h8_t *)(wr + (f / MPR) * (64 / KB) + (f % MPR) * 8);
      if (n_steps > 0) issue(0);
      norm_x(wf);
    }
#pragma unroll
    for (int i = NORM ? 1 : 0; i < NS; i++)
      if (i < n_steps) issue(i);
    // Waited for here, or the compiler, which does not count the direct loads, would wait for all of them at the first use of x in
    // every turn of the loop below.  Where there is hardly a second turn the steps behind the first need not have landed yet.
    if constexpr (LONG)
#pragma unroll
      for (int f = 0; f < NF; f++) asm volatile("" : "+v"(xf[f]));
  }

  // whether this wavefront stores sums of a unit.  Not asked for one int8 matrix, whose units are over in a step or two: the longer code costs more than
  // it saves (us, 5 rows, without | with: int8 4096 x 4096 6.1 | 6.3; fp16 w1|w3 of 8192 x 3072 16.8 | 16.4, 16 rows 17.7 | 16.9).
  const bool stores = (KIND == JSGRAD_W_F16 || EPI == GEPI_SWIGLU) && wave * 4 < a.M;
  int s = 0;
  for (int u = 0; u < units; u++) {
#pragma unroll
    for (int q = 0; q < NMAT; q++) {
      f4_t acc = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int part = 0; part < PARTS; part++, s++) {
        arrived(s + 1, std::integral_constant<int, NS - 1>(), stores && u > 0 && q * PARTS + part < NS);
        const unsigned char *const from = ring + (s % NS) * (S::SLOT + S::SCALE);
        u4_t raw[NFR];
#pragma unroll
        for (int i = 0; i < NFR; i++) raw[i] = *(const u4_t *)(from + l16 * SB + ((i * 4 + lq) ^ swizzle(l16)) * 16);
        h2_t scale = {};
        if constexpr (KIND == JSGRAD_W_I8) {
          const _Float16 v = *(const _Float16 *)(from + S::SLOT + l16 * 2);
          scale = h2_t{v, v};
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");    // the slot is in registers: it is filled again
        if (s + NS < n_steps) issue(s + NS);
#pragma unroll
        for (int i = 0; i < NFR; i++) {
          if constexpr (KIND == JSGRAD_W_F16) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, raw[i]), xf[part * NFR + i], acc, 0, 0, 0);
          else {
#pragma unroll
            for (int h = 0; h < 2; h++) {
              u4_t o;
              uint32_t lo, hi;
              i8x4_to_h2x2(raw[i][2 * h], lo, hi); o.x = pk_mul_h2(lo, scale); o.y = pk_mul_h2(hi, scale);
              i8x4_to_h2x2(raw[i][2 * h + 1], lo, hi); o.z = pk_mul_h2(lo, scale); o.w = pk_mul_h2(hi, scale);
              acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, o), xf[(part * NFR + i) * 2 + h], acc, 0, 0, 0);
            }
          }
        }
      }
      // lane: x row l16, weight rows 4 lq .. + 3
      *(f4_t *)&red[(q * FW_WAVES + wave) * 256 + l16 * 16 + lq * 4] = acc;
    }
    lds_barrier();
    if (tid < 256) {                                          // whole wavefronts
      const int m = tid >> 4, c = tid & 15, n = first_row(u) + c;
      float tot[NMAT];
#pragma unroll
      for (int q = 0; q < NMAT; q++) {
        tot[q] = red[q * FW_WAVES * 256 + tid];
#pragma unroll
        for (int w = 1; w < FW_WAVES; w++) tot[q] += red[(q * FW_WAVES + w) * 256 + tid];
      }
      const bool mine = m < a.M && (c < 8 || !is_half(u));
      const float own = rn16(tot[0]);
      if constexpr (EPI == GEPI_SWIGLU) {
        if (mine) a.y[(size_t)m * a.N + n] = (_Float16)(silu_act<_Float16>(own) * rn16(tot[NMAT - 1]));
      } else if constexpr (EPI == GEPI_STORE) {
        if (mine) a.y[(size_t)m * a.N + n] = (_Float16)(a.residual ? (float)a.residual[(size_t)m * a.N + n] + own : own);
      } else {
        const float other = dpp_f<0xB1>(own);                 // the neighbouring column: the other half of the rotary pair
        if (mine) {
          const int which = n < a.n0 ? 0 : (n < a.n0 + a.n1 ? 1 : 2);
          const int nl = which == 0 ? n : (which == 1 ? n - a.n0 : n - a.n0 - a.n1);
          const int b = m / a.seq_len, pos = a.start_pos + m % a.seq_len;
          float v = own;
          if (which < 2) {
            const h2_t cs = *(const h2_t *)(a.rope_table + ((size_t)pos * (a.head_dim / 2) + ((nl % a.head_dim) >> 1)) * 2);
            const float cc = (float)cs.x, dd = (float)cs.y;
            v = nl & 1 ? other * dd + own * cc : own * cc - other * dd;
          }
          if (which == 0) a.y[(size_t)m * a.n0 + nl] = (_Float16)v;
          else (which == 1 ? a.cache_k : a.cache_v)[((size_t)b * a.max_context + pos) * a.n1 + nl] = (_Float16)v;
        }
      }
    }
    if (u + 1 < units) lds_barrier();                         // the sums have been read
  }
}

template <int KIND, int EPI, int SB, int PARTS, bool LONG, bool NORM> static int launch_few_as(const GemmArgs &a, int tiles, int grid, int prof_kind) {
  constexpr int lds = FwShape<KIND, EPI, SB>::LDS;
  static bool raised = false;
  if (!raised) {
    JSG_HIP(hipFuncSetAttribute((const void *)few_rows_kernel<KIND, EPI, SB, PARTS, LONG, NORM>, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    raised = true;
  }
  JSG_LAUNCH(prof_kind, (few_rows_kernel<KIND, EPI, SB, PARTS, LONG, NORM>), dim3(grid), dim3(FW_THREADS), lds, a, tiles);
  return 0;
}
// LONG, where x does not come through the ring: two weight tiles or more per block (us, with and without: fp16 16384 x 2048 16.3 | 17.1, 2048 x 8192 9.2 | 8.7).
// With a norm: int8 rows of 4096, whose x fills the ring, so that no weights are asked for until it is in registers.  Up to seven rows, and from seven quarters of a
// step per block on (w1|w3 six), x goes to registers straight, the first step of weights beside it.  us, 1 / 5 / 8 rows, ring | registers: 6656 x 4096 11.2 / 11.4 / 11.5
// | 10.8 / 11.2 / 11.7, 7168 11.6 / 11.8 / 11.8 | 11.1 / 11.6 / 12.1, 8192 12.5 / 12.7 / 12.7 | 11.6 / 12.2 / 12.7, w1|w3 of 2560 10.1 / 10.2 / 10.2 | 9.7 / 10.1 / 10.6,
// 3072 10.8 / 10.9 / 11.0 | 10.2 / 10.6 / 11.2, 4096 12.4 / 12.4 / 12.5 | 11.5 / 12.0 / 12.6; less per block: 4096 8.1 / 8.0 / 8.0 | 8.6 / 8.7 / 9.2.
template <int KIND, int EPI, int SB, int PARTS> static int launch_few(const GemmArgs &a, int prof_kind) {
  constexpr int MPR = KIND == JSGRAD_W_F16 ? 1 : 2;
  const int tiles = a.N / 16, cus = state().cu_count, grid = 2 * tiles < cus ? 2 * tiles : cus;
  if constexpr (PARTS * SB * MPR <= 1024)                     // rows of at most 4096: what gemm_few takes with a norm
    if (a.norm_w) {
      if constexpr (KIND == JSGRAD_W_I8 && SB == 512)
        if (a.M <= 7 && (EPI == GEPI_SWIGLU ? 2 * tiles >= grid + grid / 2 : tiles >= grid + grid * 3 / 4)) return launch_few_as<KIND, EPI, SB, PARTS, true, true>(a, tiles, grid, prof_kind);
      return launch_few_as<KIND, EPI, SB, PARTS, false, true>(a, tiles, grid, prof_kind);
    }
  if constexpr (PARTS * MPR > FwShape<KIND, EPI, SB>::NS)
    if (tiles * (EPI == GEPI_SWIGLU ? 2 : 1) >= 2 * grid) return launch_few_as<KIND, EPI, SB, PARTS, true, false>(a, tiles, grid, prof_kind);
  return launch_few_as<KIND, EPI, SB, PARTS, false, false>(a, tiles, grid, prof_kind);
}

// A wavefront's share of a weight row, in steps of 512, 384 or 256 bytes: long steps ask for long stretches of a row, the number
// of steps is bounded by the registers x takes.
template <int KIND, int EPI> static int gemm_few_kind(const GemmArgs &a, int prof_kind, bool *taken) {
  constexpr bool F16 = KIND == JSGRAD_W_F16;
  *taken = true;
  const int share = a.K % (FW_WAVES * 64) ? 0 : a.K * (F16 ? 2 : 1) / FW_WAVES;
  switch (share) {
    case 256: return launch_few<KIND, EPI, 256, 1>(a, prof_kind);
    case 384: return launch_few<KIND, EPI, 384, 1>(a, prof_kind);
    case 512: return launch_few<KIND, EPI, 512, 1>(a, prof_kind);
    case 2 * 384: return launch_few<KIND, EPI, 384, 2>(a, prof_kind);
    case 2 * 512: return launch_few<KIND, EPI, 512, 2>(a, prof_kind);
    case 3 * 512: if constexpr (F16) return launch_few<KIND, EPI, 512, 3>(a, prof_kind); else break;
    case 4 * 512: if constexpr (F16) return launch_few<KIND, EPI, 512, 4>(a, prof_kind); else break;
  }
  *taken = false;
  return 0;
}
template <int EPI> static int gemm_few_epi(int kind, const GemmArgs &a, int prof_kind, bool *taken) {
  if (kind == JSGRAD_W_F16) return gemm_few_kind<JSGRAD_W_F16, EPI>(a, prof_kind, taken);
  if (kind == JSGRAD_W_I8) return gemm_few_kind<JSGRAD_W_I8, EPI>(a, prof_kind, taken);
  return 0;
}

int gemm_few(int epi, int kind, const GemmArgs &a, int prof_kind, bool *taken) {
  *taken = false;
  if (a.M > 16 || a.N % 16 || ((uintptr_t)a.s0 | (uintptr_t)a.s1 | (uintptr_t)a.s2) & 3) return 0;
  // int8: the codes of a tile are half the bytes behind the same x, and a tile is over in a step or two; gemm_group.hip keeps its ring full
  // over wide matrices.  us, 8 / 16 rows, that one | this one: 2048 x 8192 9.1 / 9.4 | 9.2 / 12.0, 3072 x 8192 9.9 / 10.1 | 10.4 / 12.5, 4096 x 6144
  // 10.3 / 10.4 | 9.3 / 12.3; with x through the ring 3072 x 4096 - / 8.0 | 5.6 / 5.9, 4096 x 4096 - / 8.6 | 6.1 / 6.7, 6144 x 4096 - / 9.6 | 9.2 / 9.8, 8192 x 4096
  // - / 9.7 | 10.3 / 10.8, 16384 x 3072 11.7 / 11.7 | 11.6 / 12.1, 28672 x 4096 21.4 / 21.5 | 25.2 / 25.9, 128256 x 2048 45 / 47 | 53 / 59.  With a norm in
  // front, which there is a launch of its own: one matrix level (16384 x 3072 13.5 / 13.6 | 13.6 / 14.4, 24576 x 2048 13.9 / 14.2 | 13.8 / 14.3), w1|w3 of
  // rows of 2048 and 3072 faster here at any number (9216 x 2048 13.5 / 13.8 | 12.6 / 13.1, 14336 15.6 / 15.8 | 15.1 / 15.8, 20480 21.6 / 21.9 | 18.1 / 18.9, 28672
  // 27.2 / 27.6 | 22.5 / 23.4; 8192 x 3072 14.2 / 14.3 | 12.7 / 13.4, 14336 20.8 / 21.1 | 19.2 / 19.8, 20480 28.0 / 28.7 | 23.6 / 24.2, 28672 36.4 / 37.0 | 30.5 / 31.5),
  // of rows of 4096 slower (6144 x 4096 15.0 / 15.5 | 15.7 / 16.4).
  // fp16, skinny_gemm_kernel | this one, 2 / 8 / 16 rows: 2048 x 2048 6.2 / 6.3 / 6.3 | 4.5 / 4.5 / 5.1, 2048 x 8192 14.1 / 14.9 / 15.9 |
  // 8.8 / 9.5 / 12.4, 16384 x 2048 23.6 / 23.7 / 24.4 | 16.3 / 17.2 / 18.2, 128256 x 2048 147 / 153 / 162 | 88 / 92 / 94 (6.0 TB/s).
  // fp16 rows of more than 4096 elements (6144 and 8192 come here): the more rows of x a block reads for its few tiles, the nearer gemm_group.hip, which reads x from LDS, comes.  us,
  // 9 / 12 / 16 rows, that one | this one: 1024 x 6144 9.9 / 10.0 / 10.1 | 7.5 / 8.3 / 9.3, 2048 x 6144 10.5 / 10.6 / 10.8 | 8.4 / 9.0 / 10.1, 4096 x 6144
  // 13.2 / 13.2 / 13.3 | 12.1 / 12.8 / 13.9, 8192 x 6144 19.2 / 19.4 / 19.4 | 19.4 / 20.0 / 20.9, 20480 x 6144 58.0 / 58.5 / 58.7 | 40.6 / 41.5 / 42.6;
  // 2048 x 8192 11.0 / 11.1 / 11.3 | 9.8 / 11.2 / 12.7, 3072 x 8192 12.9 / 12.9 / 13.0 | 12.6 / 13.9 / 15.3, 4096 x 8192 17.3 / 17.3 / 17.3 | 14.7 / 16.0 /
  // 17.5, 8192 x 8192 26.5 / 26.7 / 26.7 | 25.1 / 25.9 / 27.0, 12032 x 8192 38.5 / 38.7 / 38.8 | 34.2 / 35.0 / 36.4.
  const int rows = a.N * (epi == GEPI_SWIGLU ? 2 : 1);
  const size_t elements = (size_t)rows * a.K;
  if (kind == JSGRAD_W_F16 && a.K > 4096 &&
      (a.K > 6144 ? rows > 1024 && rows <= 3072 && a.M > (rows <= 2048 ? 12 : 9) : rows > 2048 && elements < (size_t)80 << 20 && a.M > (rows <= 6144 ? 13 : 8)))
    return 0;
  // A norm in front is done in registers, x and the norm's weights at once: rows of half the length at most.  us per decode step, norms as launches of
  // their own (33 of the 1B shape) | here: 1B shape 2 rows 897 | 832, 5 rows 903 | 846, 12 rows 968 | 908, 16 rows 1006 | 944; int8 14 layers of the 3B shape
  // with 6 rows 830 | 810, of the 8B shape with 4 rows 1131 | 1113.  In gemm_group.hip, whose blocks read all of x for it and norm every fragment, it
  // costs more than the launches: 8B int8 16 rows 3321 | 3403, 8B NF4 16 layers 8 rows 1403 | 1467.
  // The norm's weights are read here in 16-byte pieces; from any other address in memory first.
  if (a.norm_w && (a.K > 4096 || (uintptr_t)a.norm_w & 15)) return 0;
  const size_t most = a.norm_w && epi == GEPI_SWIGLU && a.K <= 3072 ? SIZE_MAX : (size_t)36 << 20;
  // int8 rows of 4096 behind 9 to 16 rows: up to 4096 weight rows.  us, 9 / 16 rows, the kernels below | this one: 512 weight rows 6.5 / 6.9 | 4.6 / 4.7, 1024 6.7 /
  // 7.0 | 4.8 / 4.8, 2048 7.0 / 7.3 | 5.1 / 5.2, 3072 7.3 / 7.6 | 5.8 / 5.8, 4096 7.8 / 8.1 | 6.6 / 6.6; behind the line 5120 8.8 / 8.8 | 8.5 / 8.5, 6144 9.2 / 9.3 |
  // 9.1 / 9.2, 8192 9.7 / 9.7 | 10.7 / 10.6; w1|w3 of 1024 9.8 / 10.0 | 6.3 / 6.3, of 2048 10.5 / 10.7 | 6.9 / 7.1.
  if (kind == JSGRAD_W_I8 && (elements > most || (a.M > 8 && (a.K > 4096 || (a.K > 3072 && rows > 4096))))) return 0;
  if (pin_env(a, "JSG_GEMM_NO_SKINNY") || pin_env(a, "JSG_GEMM_SKINNY_TILES")) return 0;   // tests that want one of the other kernels
  if (epi == GEPI_STORE) return gemm_few_epi<GEPI_STORE>(kind, a, prof_kind, taken);
  if (epi == GEPI_ROPE_KV) return gemm_few_epi<GEPI_ROPE_KV>(kind, a, prof_kind, taken);
  return gemm_few_epi<GEPI_SWIGLU>(kind, a, prof_kind, taken);
}

}  // namespace jsg
