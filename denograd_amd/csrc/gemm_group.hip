// Several-row linear layers of up to some dozens of rows, any weight format: y[M][N] = x[M][K] . W[N][K]^T; what the reference computes is
// in gemm_tile.hip.
//
// The launch should be bound by reading W once.  With few rows a tile has little arithmetic, and what a compute unit can draw is the
// bytes it has on their way over the time they take (2 us under load): so one block of eight wavefronts owns nearly all of a unit's
// LDS (int8 in 16x64 tiles: two blocks half each) as a ring of ST turns.  A turn is G neighbouring K stages of the tile (G x 64 elements, nf4 G x 128), one per K group; the WN
// wavefronts of a group split the tile's columns, so a weight is dequantised once per block and a piece of x is read by WN wavefronts.
// Fragments are read a turn ahead of the matrix instructions that use them, one barrier per turn.  The groups' sums are
// added in LDS in group order; K parts over blocks as in gemm_tile.hip, in part order.
// Measured (weights from memory, us, the kernels it took the sizes from | this one): 16 rows, int8 28672 x 4096 27.0 | 21.9 (5.4 TB/s), 4096 x 14336 17.8 |
// 15.1; 24 rows, int8 16384 x 3072 22.8 | 15.0, 128256 x 3072 213 | 77; fp16 16384 x 2048 23.8 | 14.7, 128256 x 3072 265 | 126 (6.2 TB/s), 4096 x 14336
// 36 | 23; nf4 28672 x 4096 46 | 25, with 8 rows 36.7 | 21.7.  From 33 rows on LDS reads and matrix instructions of a turn take as long as its bytes to
// arrive, and it is ahead by less: 57 rows, 16384 x 3072 int8 19.5 | 17.5, nf4 21.4 | 18.4, 128256 x 3072 int8 112 | 104.
#include <type_traits>

#include "gemm_tile.h"

namespace jsg {

constexpr int GROUP_THREADS = 512;

// A stage of a group: WB bytes (64 or 128) of every weight row, as 16-byte pieces; a lane's piece is the operands of STEPS matrix instructions, and
// x is read in the order of K that this makes: lane quarter lq, step s of piece group p: elements (p * 4 + lq) * 8 * STEPS + 8 s .. + 7.
template <int KIND, int WB> struct GFmt {
  static constexpr int STEPS = KIND == JSGRAD_W_F16 ? 1 : (KIND == JSGRAD_W_I8 ? 2 : 4);
  static constexpr int PG = WB / 64;                          // piece groups: four pieces, one per lane quarter
  static constexpr int KF = PG * STEPS, KS = KF * 32;         // steps and K elements of a stage
};
template <int KIND, int WB, int BM, int BN, int WN, int ST> struct GShape {
  typedef GFmt<KIND, WB> F;
  static constexpr int G = 8 / WN;                            // K groups
  static constexpr int X = BM * F::KS * 2, W = BN * WB;       // bytes of a group's stage
  static constexpr int SCALES = KIND == JSGRAD_W_NF4 ? 256 * F::PG : 0;   // per wavefront
  static constexpr int TURN = G * (X + W) + 8 * SCALES;
  static constexpr int TABLE = KIND == JSGRAD_W_NF4 ? 16384 : (KIND == JSGRAD_W_I8 ? 2048 : 0);   // nf4: 16 copies of the table of code pairs; int8: row scales
  static constexpr int RED = G * BM * (BN + 4) * 4;
  static constexpr int LDS = (TURN * ST > RED ? TURN * ST : RED) + TABLE;
  static_assert(LDS + 64 <= 160 * 1024, "LDS of one compute unit");
};

template <int KIND, int EPI, int WB, int BM, int BN, int WN, int ST> __global__ __launch_bounds__(GROUP_THREADS, 2) void group_kernel(TileArgs t) {
  typedef GFmt<KIND, WB> F;
  typedef GShape<KIND, WB, BM, BN, WN, ST> S;
  const GemmArgs &a = t.g;
  extern __shared__ __align__(16) unsigned char group_lds[];
  constexpr int G = S::G, KS = F::KS, KF = F::KF, PG = F::PG, STEPS = F::STEPS, TM = BM / 16, TN = BN / 16 / WN;
  constexpr int XI = S::X / 1024, WI = S::W / 1024;           // direct loads of 1 KiB per group and turn: eight x rows, or 1024 / WB weight rows
  constexpr int NX = G * XI / 8, NW = G * WI / 8;             // ... and per wavefront
  static_assert(NX * 8 == G * XI && NW * 8 == G * WI && TN >= 1, "every wavefront issues the same loads");
  constexpr int NLD = NX + NW + (KIND == JSGRAD_W_NF4 ? PG : 0);
  constexpr int CW = EPI == GEPI_SWIGLU ? BN / 2 : BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, lq = lane >> 4;
  const int kg = wave / WN, wn = wave % WN;
  const TileId id = tile_id<BM, CW>(t);
  const int m0 = id.m0;
  uint32_t *const table = (uint32_t *)(group_lds + (S::LDS - S::TABLE));
  if constexpr (KIND == JSGRAD_W_NF4)                         // entry e, copy c at word 16 e + c; read after a barrier
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int e = (i * 512 + tid) >> 4;
      table[i * 512 + tid] = nf4_code_bits(e >> 4) | (nf4_code_bits(e & 15) << 16);
    }

  // ---- loads: wavefront w issues NX and NW consecutive ones of the turn's G * XI and G * WI
  const uint32_t x_bytes = (uint32_t)a.K * 2, w_bytes = KIND == JSGRAD_W_F16 ? a.K * 2 : (KIND == JSGRAD_W_I8 ? a.K : a.K / 2);
  const int nst = a.K / KS, k0 = (int)((long long)id.part * nst / t.split), ns = (int)((long long)(id.part + 1) * nst / t.split) - k0;
  const int turns = (ns + G - 1) / G;
  // Weight rows whose distance is a multiple of 4 KiB: blocks start their walk through K at different turns and wrap around, so that they
  // don't queue at the same offset of such rows for the same memory channels (28672 x 4096, us: int8, 8 rows 30.1 -> 26.4, 24 rows 33.9 ->
  // 32.2; fp16, 24 rows in 32x64 tiles 46.3 -> 41.9, but in 32x128 47 -> 55 and 57 rows 49.3 -> 56.7; other distances and K parts: 1 % slower).
  // int8 in 16x64 tiles: a turn is 256 bytes of a row, neighbours start two of them apart (14336 x 8192, one | two | four: 28.3 | 22.4 | 22.0, w1|w3 of
  // 8192 x 8192 25.8 | 23.5 | 35.2).
  constexpr unsigned APART = KIND == JSGRAD_W_I8 && BM == 16 && BN == 64 ? 2 : 1;
  const int first = BM <= 32 && (KIND != JSGRAD_W_F16 || BM * BN < 4096) && t.split == 1 && w_bytes % 4096 == 0 ? (int)((unsigned)(id.col / CW) * APART % (unsigned)turns) : 0;
  auto turn_of = [&](int turn) { const int r = turn + first; return r >= turns ? r - turns : r; };
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)group_lds;
  const i4_t ra = dma_rsrc(a.x + (size_t)m0 * a.K);
  uint32_t va[NX], la[NX];
  int ga[NX];
#pragma unroll
  for (int i = 0; i < NX; i++) {
    const int idx = wave * NX + i, in = idx % XI, sl = in / (BM / 8), r8 = in % (BM / 8) * 8;
    ga[i] = idx / XI;
    va[i] = (uint32_t)min(r8 + (lane >> 3), a.M - 1 - m0) * x_bytes + (uint32_t)((lane & 7) ^ (lane >> 3)) * 16 + sl * 128;   // rows past the end are computed and never stored
    la[i] = lds0 + ga[i] * (S::X + S::W) + in * 1024;
  }
  constexpr int RPL = 1024 / WB;                           // weight rows of a load
  i4_t rb[NW];
  uint32_t lb[NW];
  int gb[NW];
#pragma unroll
  for (int i = 0; i < NW; i++) {
    const int idx = wave * NW + i;
    gb[i] = idx / WI;
    rb[i] = dma_rsrc(weight_ptr<EPI, BN>(t, id.col, idx % WI * RPL, w_bytes));
    lb[i] = lds0 + gb[i] * (S::X + S::W) + S::X + idx % WI * 1024;
  }
  const uint32_t vb = WB == 128 ? (uint32_t)(lane >> 3) * w_bytes + (uint32_t)((lane & 7) ^ (lane >> 3)) * 16
                                   : (uint32_t)(lane >> 2) * w_bytes + (uint32_t)((lane & 3) ^ ((lane >> 3) & 3)) * 16;
  // scales of this wavefront's rows (one matrix: a wavefront's columns never straddle two)
  const int my_row = wn * TN * 16;
  const WeightRow sr = weight_row<EPI, BN>(t, id.col, my_row);
  i4_t rs;
  uint32_t odd = 0;                                           // int8 scales between two words: loaded from the word they begin in, and lying a half further on
  if constexpr (KIND != JSGRAD_W_F16) {
    const _Float16 *const from = pick(t.s, sr.mat) + (size_t)sr.row * (KIND == JSGRAD_W_I8 ? 1 : a.K / 64);
    if constexpr (KIND == JSGRAD_W_I8) odd = (uint32_t)((uintptr_t)from >> 1) & 1;
    rs = dma_rsrc(from - odd);
  }
  const uint32_t vs = KIND == JSGRAD_W_I8 ? min((uint32_t)lane, TN * 8 - 1 + odd) * 4 : (uint32_t)(lane & (TN * 16 - 1)) * (a.K / 32);
  auto load = [&](int at, int buf) {
    const int turn = turn_of(at);
    const uint32_t base = (uint32_t)buf * S::TURN;
#pragma unroll
    for (int i = 0; i < NX; i++) dma16(ra, va[i], (uint32_t)(k0 + min(turn * G + ga[i], ns - 1)) * (KS * 2), base + la[i]);
#pragma unroll
    for (int i = 0; i < NW; i++) dma16_stream(rb[i], vb, (uint32_t)(k0 + min(turn * G + gb[i], ns - 1)) * WB, base + lb[i]);
    if constexpr (KIND == JSGRAD_W_NF4)
#pragma unroll
      for (int p = 0; p < PG; p++) dma4(rs, vs, (uint32_t)((k0 + min(turn * G + kg, ns - 1)) * PG + p) * 4, lds0 + base + G * (S::X + S::W) + wave * S::SCALES + p * 256);
  };

  f4_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++) acc[i][j] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
  struct Frags {
    h8_t x[KF][TM];
    u4_t w[PG][TN];
    h2_t s[PG][TN];                                           // nf4: the scales of the piece group's two blocks
  };
  Frags fr[2];
  auto read = [&](int buf, Frags &f) {
    const unsigned char *px = group_lds + buf * S::TURN + kg * (S::X + S::W) + l16 * 128;
    const unsigned char *pw = group_lds + buf * S::TURN + kg * (S::X + S::W) + S::X + (my_row + l16) * WB;
#pragma unroll
    for (int p = 0; p < PG; p++) {
#pragma unroll
      for (int s = 0; s < STEPS; s++) {
        const int piece = (p * 4 + lq) * STEPS + s;
        const unsigned char *from = px + (piece >> 3) * (BM * 128) + ((piece & 7) ^ (l16 & 7)) * 16;
#pragma unroll
        for (int i = 0; i < TM; i++) f.x[p * STEPS + s][i] = *(const h8_t *)(from + i * 2048);
      }
      const uint32_t at = (WB == 128 ? (p * 4 + lq) ^ (l16 & 7) : lq ^ ((l16 >> 1) & 3)) * 16;
#pragma unroll
      for (int j = 0; j < TN; j++) {
        f.w[p][j] = *(const u4_t *)(pw + j * 16 * WB + at);
        if constexpr (KIND == JSGRAD_W_NF4) f.s[p][j] = *(const h2_t *)(group_lds + buf * S::TURN + G * (S::X + S::W) + wave * S::SCALES + p * 256 + (j * 16 + l16) * 4);
      }
    }
  };
  h2_t scale[TN];
  const uint32_t *const tab = table + l16;
  auto compute = [&](int turn, const Frags &f) {
    if (turn_of(turn) * G + kg >= ns) return;                 // the last turn may not have a stage for every group
#pragma unroll
    for (int p = 0; p < PG; p++)
#pragma unroll
      for (int j = 0; j < TN; j++) {
        const u4_t raw = f.w[p][j];
        const uint32_t wds[4] = {raw.x, raw.y, raw.z, raw.w};
        const _Float16 s1 = lq < 2 ? f.s[p][j].x : f.s[p][j].y;
        const h2_t sv = {s1, s1};
#pragma unroll
        for (int s = 0; s < STEPS; s++) {
          u4_t o;
          if constexpr (KIND == JSGRAD_W_F16) o = raw;
          else if constexpr (KIND == JSGRAD_W_I8) {
            uint32_t lo, hi;
            i8x4_to_h2x2(wds[2 * s], lo, hi); o.x = pk_mul_h2(lo, scale[j]); o.y = pk_mul_h2(hi, scale[j]);
            i8x4_to_h2x2(wds[2 * s + 1], lo, hi); o.z = pk_mul_h2(lo, scale[j]); o.w = pk_mul_h2(hi, scale[j]);
          } else {
            const uint32_t c = wds[s];
            o.x = pk_mul_h2(tab[(c & 0xffu) * 16], sv);
            o.y = pk_mul_h2(tab[((c >> 8) & 0xffu) * 16], sv);
            o.z = pk_mul_h2(tab[((c >> 16) & 0xffu) * 16], sv);
            o.w = pk_mul_h2(tab[(c >> 24) * 16], sv);
          }
          const h8_t b = __builtin_bit_cast(h8_t, o);
#pragma unroll
          for (int i = 0; i < TM; i++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b, f.x[p * STEPS + s][i], acc[i][j], 0, 0, 0);
        }
      }
  };

  // int8: one scale per row, through LDS in front of everything (a load to a register would be waited for with all later ones)
  if constexpr (KIND == JSGRAD_W_I8) dma4(rs, vs, 0, lds0 + (S::LDS - S::TABLE) + wave * 256);
#pragma unroll
  for (int i = 0; i < ST - 1; i++)
    if (i < turns) load(i, i);
  int buf = 0, into = ST - 1;
  // turn t: its loads have landed (those of the turns behind it may be on their way), everybody has read the turn before it,
  // whose buffer is refilled
  auto step = [&](int turn, int cur) {
    const int behind = min(turns - 1 - turn, ST - 2);
    static_assert(ST >= 2 && ST <= 6 && (ST - 2) * NLD <= 63, "what the counter of outstanding loads holds");
    if (ST == 6 && behind == 4) wait_loads<4 * NLD>();
    else if (ST >= 5 && behind == 3) wait_loads<3 * NLD>();
    else if (ST >= 4 && behind == 2) wait_loads<2 * NLD>();
    else if (ST >= 3 && behind == 1) wait_loads<NLD>();
    else wait_loads<0>();
    turn_barrier_lds();
    if (turn + ST - 1 < turns) load(turn + ST - 1, into);
    read(buf, fr[cur]);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (KIND == JSGRAD_W_I8)
      if (turn == 0)
#pragma unroll
        for (int j = 0; j < TN; j++) {
          const _Float16 v = *(const _Float16 *)(group_lds + (S::LDS - S::TABLE) + wave * 256 + (j * 16 + l16 + odd) * 2);
          scale[j] = h2_t{v, v};
        }
    buf = buf + 1 == ST ? 0 : buf + 1;
    into = into + 1 == ST ? 0 : into + 1;
  };
  step(0, 0);
  int turn = 1;
  for (; turn + 1 < turns; turn += 2) {
    step(turn, 1);
    compute(turn - 1, fr[0]);
    __builtin_amdgcn_sched_barrier(0);
    step(turn + 1, 0);
    compute(turn, fr[1]);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (turn < turns) {
    step(turn, 1);
    compute(turn - 1, fr[0]);
    compute(turn, fr[1]);
  } else compute(turn - 1, fr[0]);

  // ---- the groups' sums through LDS (every load has landed and been read)
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  turn_barrier();
  constexpr int RS = BN + 4;
  float *const red = (float *)group_lds;
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++) *(f4_t *)&red[(kg * BM + i * 16 + l16) * RS + my_row + j * 16 + lq * 4] = acc[i][j];
  lds_barrier();

  // a piece: eight neighbouring columns of a row of the tile (SWIGLU: of w1 and of w3); pieces are dealt to the threads
  struct Eight { f4_t lo, hi; };
  auto summed = [&](int row, int col) {
    Eight e;
#pragma unroll
    for (int g = 0; g < G; g++) {
      const float *p = &red[(g * BM + row) * RS + col];
      const f4_t lo = *(const f4_t *)p, hi = *(const f4_t *)(p + 4);
      if (g == 0) e = Eight{lo, hi};
      else { e.lo += lo; e.hi += hi; }
    }
    return e;
  };
  constexpr int RAW = BM * BN / 8, PPR = BN / 8;              // pieces of the tile, per row
  __amdgpu_buffer_rsrc_t rw;
  const int split = t.split;
  if (split > 1) {
    __shared__ int last;
    rw = wave_buffer(t.ws + (size_t)id.tile * split * (BM * BN), (uint32_t)split * (BM * BN) * 4u);
    for (int p = tid; p < RAW; p += GROUP_THREADS) {
      const Eight e = summed(p / PPR, p % PPR * 8);
      const uint32_t o = (uint32_t)id.part * (BM * BN * 4) + (uint32_t)p * 32;
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4_t, e.lo), rw, o, 0, 16);
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4_t, e.hi), rw, o + 16, 0, 16);
    }
    wait_loads<0>();
    turn_barrier();
    if (tid == 0) {
      const int old = __hip_atomic_fetch_add(&t.counters[id.tile], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      last = old == split - 1;
      if (last) __hip_atomic_store(&t.counters[id.tile], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // for the next launch
    }
    __syncthreads();
    if (!last) return;
  }
  auto total = [&](int row, int col) {
    if (split == 1) return summed(row, col);
    const uint32_t o = (uint32_t)(row * PPR + col / 8) * 32;
    Eight e;
    e.lo = __builtin_bit_cast(f4_t, __builtin_amdgcn_raw_buffer_load_b128(rw, o, 0, 16));
    e.hi = __builtin_bit_cast(f4_t, __builtin_amdgcn_raw_buffer_load_b128(rw, o + 16, 0, 16));
#pragma unroll 4
    for (int p = 1; p < split; p++) {
      e.lo += __builtin_bit_cast(f4_t, __builtin_amdgcn_raw_buffer_load_b128(rw, o + (uint32_t)p * (BM * BN * 4), 0, 16));
      e.hi += __builtin_bit_cast(f4_t, __builtin_amdgcn_raw_buffer_load_b128(rw, o + (uint32_t)p * (BM * BN * 4) + 16, 0, 16));
    }
    return e;
  };
  constexpr int OUT = BM * CW / 8, OPR = CW / 8;
  for (int p = tid; p < OUT; p += GROUP_THREADS) {
    const int row = p / OPR, c8 = p % OPR * 8, m = m0 + row, n = id.col + c8;
    if (m >= a.M) continue;
    h8_t res = {};
    if constexpr (EPI == GEPI_STORE)
      if (a.residual) res = *(const h8_t *)&a.residual[(size_t)m * a.N + n];
    const Eight e = total(row, c8);
    h8_t v;
    if constexpr (EPI == GEPI_SWIGLU) {
      const Eight u = total(row, c8 + BN / 2);
#pragma unroll
      for (int c = 0; c < 4; c++) { v[c] = (_Float16)swiglu(e.lo[c], u.lo[c]); v[c + 4] = (_Float16)swiglu(e.hi[c], u.hi[c]); }
    } else {
#pragma unroll
      for (int c = 0; c < 4; c++) { v[c] = (_Float16)e.lo[c]; v[c + 4] = (_Float16)e.hi[c]; }
    }
    store_piece<EPI>(a, m, n, v, res);
  }
}

template <int KIND, int EPI, int WB, int BM, int BN, int WN, int ST> static int launch_group_as(const TileArgs &t, int prof_kind) {
  constexpr int lds = GShape<KIND, WB, BM, BN, WN, ST>::LDS;
  static bool raised = false;
  if (!raised) {
    JSG_HIP(hipFuncSetAttribute((const void *)group_kernel<KIND, EPI, WB, BM, BN, WN, ST>, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    raised = true;
  }
  const int tiles = ((t.g.M + BM - 1) / BM) * (t.g.N / (EPI == GEPI_SWIGLU ? BN / 2 : BN));
  JSG_LAUNCH(prof_kind, (group_kernel<KIND, EPI, WB, BM, BN, WN, ST>), dim3(tiles * t.split), dim3(GROUP_THREADS), lds, t);
  return 0;
}

// Turns in LDS: as many as fit.  Stages have 128 bytes of a weight row, whole cache lines for eight rows per load: with 64 bytes of sixteen rows int8
// codes came at three quarters of the rate (us, 64 | 128: 16384 x 3072, 16 rows 16.7 | 13.2, 28672 x 4096 27.4 | 22.1, 24 rows 32.7 | 26.6, 128256 x 3072 101 |
// 77; nf4 28672 x 4096, 24 rows 29 | 25).  int8 in 16x64 tiles: two K groups and 74 KB, so that two blocks share a unit and one's first loads and sums run
// beside the other's turns (four groups and 146 KB | two: 41984 x 2560 31 | 21.7, 128256 x 1024 42.3 | 27.8, 28672 x 4096 26.5 | 22.5, 4096 x 14336 15.5 |
// 14.7).  nf4 behind 64 rows of x, where that many K elements of x leave no room for a third turn, keeps 64.
template <int KIND, int EPI> static int launch_group_kind(int bm, int bn, const TileArgs &t, int prof_kind) {
  constexpr bool NF4 = KIND == JSGRAD_W_NF4, F16 = KIND == JSGRAD_W_F16;
  if (bm == 16 && bn == 64) return launch_group_as<KIND, EPI, 128, 16, 64, F16 ? 2 : 4, 3>(t, prof_kind);
  if (bm == 16 && bn == 128) return launch_group_as<KIND, EPI, 128, 16, 128, F16 ? 2 : 4, F16 || NF4 ? 2 : 3>(t, prof_kind);
  if (bm == 32 && bn == 64) return launch_group_as<KIND, EPI, 128, 32, 64, F16 ? 2 : 4, F16 ? 3 : (NF4 ? 2 : 4)>(t, prof_kind);
  if (bm == 32 && bn == 128) return launch_group_as<KIND, EPI, 128, 32, 128, 4, NF4 ? 2 : 3>(t, prof_kind);
  if (bm == 64 && bn == 64) return launch_group_as<KIND, EPI, NF4 ? 64 : 128, 64, 64, F16 ? 2 : 4, F16 ? 2 : 3>(t, prof_kind);
  if (bm == 64 && bn == 128) return launch_group_as<KIND, EPI, NF4 ? 64 : 128, 64, 128, 4, F16 ? 3 : 2>(t, prof_kind);
  return fail("jsgrad_hip_gemm: no tile shape");
}

static int launch_group(int epi, int kind, int bm, int bn, const TileArgs &t, int prof_kind) {
  auto with = [&](auto k) {
    constexpr int KIND = decltype(k)::value;
    if (epi == GEPI_STORE) return launch_group_kind<KIND, GEPI_STORE>(bm, bn, t, prof_kind);
    if (epi == GEPI_ROPE_KV) return launch_group_kind<KIND, GEPI_ROPE_KV>(bm, bn, t, prof_kind);
    return launch_group_kind<KIND, GEPI_SWIGLU>(bm, bn, t, prof_kind);
  };
  if (kind == JSGRAD_W_F16) return with(std::integral_constant<int, JSGRAD_W_F16>());
  if (kind == JSGRAD_W_I8) return with(std::integral_constant<int, JSGRAD_W_I8>());
  return with(std::integral_constant<int, JSGRAD_W_NF4>());
}

// The shapes with their K groups, and what a block's time is made of (us): a turn when every block has a compute unit to itself, what is
// added to it when all units have one, a turn when there are several rounds of blocks, and a round's end.  Fitted to 8 to 57 rows over the matrices
// of the 1B, 3B and 8B models in the three formats, weights from memory, each under every shape and number of K parts that could
// matter; the choice is 2 % slower than the best shape on average.  (int8 16x64, two blocks to a unit: for the choice rather than for the single time.)
struct GroupShape { int bm, bn, stage, groups; float step, fill, round_step, end; };   // stage: K elements
constexpr int N_GROUP = 6;
static const GroupShape GROUP_SHAPES[3][N_GROUP] = {   // fp16, int8, nf4
  {{16, 64, 64, 4, 0.44f, 0.43f, 0.91f, 1.3f}, {16, 128, 64, 4, 1.19f, 0.89f, 2.06f, 1.1f}, {32, 64, 64, 4, 0.52f, 0.51f, 1.07f, 1.5f}, {32, 128, 64, 2, 0.46f, 0.60f, 0.98f, 1.6f}, {64, 64, 64, 4, 1.06f, 0.54f, 1.64f, 1.6f}, {64, 128, 64, 2, 0.54f, 0.88f, 1.27f, 2.4f}},
  {{16, 64, 128, 2, 0.325f, 0.168f, 0.456f, 0.91f}, {16, 128, 128, 2, 0.54f, 0.42f, 1.03f, 1.8f}, {32, 64, 128, 2, 0.39f, 0.29f, 0.77f, 1.7f}, {32, 128, 128, 2, 0.64f, 0.60f, 1.23f, 2.4f}, {64, 64, 128, 2, 0.53f, 0.45f, 1.03f, 2.4f}, {64, 128, 128, 2, 0.82f, 1.11f, 1.70f, 3.6f}},
  {{16, 64, 256, 2, 0.87f, 0.26f, 1.33f, 1.6f}, {16, 128, 256, 2, 1.69f, 0.45f, 2.27f, 1.9f}, {32, 64, 256, 2, 1.25f, 0.30f, 1.77f, 1.9f}, {32, 128, 256, 2, 1.94f, 0.63f, 2.56f, 2.5f}, {64, 64, 128, 2, 0.83f, 0.26f, 1.18f, 2.5f}, {64, 128, 128, 2, 1.06f, 0.81f, 1.70f, 3.8f}},
};
// The K parts' sums of a launch lie in memory that belongs to the library: they are also there in a graph capture and on a full device, and
// one in-order stream serves every launch.
constexpr int GROUP_COUNTERS = 4096;
constexpr size_t GROUP_SUMS = (size_t)8 << 20;
static __device__ __align__(256) unsigned char group_sums[GROUP_SUMS];
static __device__ int group_counters[GROUP_COUNTERS];

static size_t group_bytes(const GroupShape &s, int M, int weight_rows, int split) {
  return split < 2 ? 0 : (size_t)((M + s.bm - 1) / s.bm) * (weight_rows / s.bn) * split * s.bm * s.bn * 4;
}
// JSG_GEMM_TILE, for tests and measurements: "g64x128", or "g64x128/3" with K parts
static bool group_pin(const GemmArgs &a, int &bm, int &bn, int &split) {
  const char *e = pin_env(a, "JSG_GEMM_TILE");
  split = 1;
  return e && *e == 'g' && sscanf(e + 1, "%dx%d/%d", &bm, &bn, &split) >= 2;
}
GroupChoice choose_group(int epi, int kind, const GemmArgs &a) {
  GroupChoice best;
  int bm = 0, bn = 0, split = 0;
  const bool pin = group_pin(a, bm, bn, split);
  // Scales come by direct loads of four bytes: int8's, once per block, from any even address (us with scales at an odd multiple of two bytes, the
  // kernels below | here: 9 x 128256 x 1024 85.8 | 32.8, 7 x w1|w3 of 14336 x 3072 37.0 | 18.8); nf4's, every turn, from whole words only.
  // With more rows than a tile has the weights would be read twice.
  if (((uintptr_t)a.s0 | (uintptr_t)a.s1 | (uintptr_t)a.s2) & (kind == JSGRAD_W_I8 ? 1 : 3) || (!pin && a.M > 64)) return best;
  const int cus = state().cu_count, weight_rows = a.N * (epi == GEPI_SWIGLU ? 2 : 1);
  for (int i = 0; i < N_GROUP; i++) {
    const GroupShape &s = GROUP_SHAPES[kind - JSGRAD_W_F16][i];
    const int stages = a.K / s.stage;
    if (weight_rows % s.bn || a.K % s.stage || (pin && (s.bm != bm || s.bn != bn))) continue;
    const int tiles = ((a.M + s.bm - 1) / s.bm) * (weight_rows / s.bn);
    for (int d = 1; d <= 16 && d <= stages; d++) {
      if (pin && d != (split < stages ? split : stages)) continue;
      const int blocks = tiles * d, turns = ((stages + d - 1) / d + s.groups - 1) / s.groups;
      // parts of at least two turns (int8 behind 16 rows, whose turns are short: four; 16 x 1024 x 6144 in 12 parts of two 9.7 us, in six of four 8.5),
      // and not more than two blocks for every unit
      if (d > 1 && (tiles > GROUP_COUNTERS || group_bytes(s, a.M, weight_rows, d) > GROUP_SUMS || (!pin && (turns < (kind == JSGRAD_W_I8 && s.bm == 16 ? 4 : 2) || blocks > 2 * cus)))) break;
      const float fill = (float)blocks / cus;
      float us = 3.5f + (fill <= 1.0f ? (s.step + s.fill * fill) * turns + s.end : ((blocks + cus - 1) / cus) * (s.round_step * turns + s.end));
      if (d > 1) us += 1.7f + (float)d * s.bm * s.bn * 4 / 83e3f * (fill > 1.0f ? fill : 1.0f);
      // int8 in two row tiles of 16, whole rows: the weights come twice, and half the bytes in tiles of 32 with K parts are the faster by what the estimates
      // are apart (24 x 6144 x 4096: 11.1 us, 32x64 in two parts 10.8; in parts they are not, 24 x 2048 x 8192: 10.1 | 10.8)
      else if (kind == JSGRAD_W_I8 && s.bm == 16 && a.M > 16 && a.M <= 32) us += 0.5f;
      if (best.shape < 0 || us < best.us) { best.us = us; best.shape = i; best.split = d; }
    }
  }
  return best;
}

int run_group(int epi, int kind, const GemmArgs &a, const GroupChoice &c, int prof_kind) {
  static int *counters = nullptr;
  static float *sums = nullptr;
  if (!sums) {
    JSG_HIP(hipGetSymbolAddress((void **)&counters, HIP_SYMBOL(group_counters)));
    JSG_HIP(hipGetSymbolAddress((void **)&sums, HIP_SYMBOL(group_sums)));
  }
  const GroupShape &s = GROUP_SHAPES[kind - JSGRAD_W_F16][c.shape];
  TileArgs t = tile_args(epi, a, counters);
  t.split = c.split;
  t.ws = sums;
  return launch_group(epi, kind, s.bm, s.bn, t, prof_kind);
}

int gemm_group(int epi, int kind, const GemmArgs &a, int prof_kind, bool *taken) {
  *taken = false;
  int bm, bn, split;
  const bool pin = group_pin(a, bm, bn, split);
  if (!pin) {
    if (a.M > 32 || pin_env(a, "JSG_GEMM_TILE") || pin_env(a, "JSG_GEMM_NO_SKINNY") || pin_env(a, "JSG_GEMM_SKINNY_TILES")) return 0;   // tests that want one of the other kernels
    // One round of skinny_gemm_kernel's blocks over short rows: no K parts whose sums have to travel.  us, that | this one: 24 rows, fp16
    // 2048 x 2048 7.5 | 7.5, 3072 x 2048 8.1 | 8.1, 3072 x 3072 9.9 | 9.3, 4096 x 3072 9.9 | 10.5, 4096 x 3584 11.3 | 11.1, 2048 x 8192 18.7 | 11.5; int8
    // 1024 x 4096 8.7 | 8.2, 2048 x 4096 8.9 | 9.6, 4096 x 3584 9.2 | 10.2, 4096 x 4096 10.2 | 10.3, 4096 x 4608 11.0 | 10.8, 6144 x 4096 17.5 | 11.4, 28672 x 4096 50 | 27; nf4
    // 4096 x 4096 9.3 | 10.9, 4096 x 5120 12.0 | 12.4, 4096 x 6144 12.8 | 12.6, 3072 x 8192 14.8 | 12.9, 28672 x 4096 46 | 25; 16 / 2 rows, int8 4096 x 4096
    // 8.9 / 8.4 | 9.0 / 8.8, 2560 x 5120 10.0 / 8.7 | 8.4 / 8.2, 3840 x 5120 10.0 / 8.9 | 9.8 / 9.5 (w1|w3 of 2048 x 5120 14.2 / 13.2 | 11.3 / 11.3), 4096 x 5632
    // 10.3 / 9.0 | 10.2 / 9.8, 6144 x 4096 13.3 / 11.6 | 9.8 / 9.7; 16 rows, nf4 4096 x 6144 10.3 | 10.9, 4096 x 8192
    // 11.9 | 12.1, 4096 x 10240 14.8 | 13.4; 8 rows, nf4 4096 x 4096 7.8 | 9.4, 3072 x 8192 10.7 | 11.5, 6144 x 4096 11.3 | 10.7, 28672 x 4096 36.7 | 21.7.
    // Where this one finds four or five parts for a unit each (up to 3072 weight rows) the line lies lower.
    const int rows = a.N * (epi == GEPI_SWIGLU ? 2 : 1), round = 16 * state().cu_count;
    const bool wide = rows > 3072;
    const int longest = kind == JSGRAD_W_F16 ? (wide ? 3072 : 2048)
                      : kind == JSGRAD_W_I8 ? (a.M <= 16 ? (wide && epi != GEPI_SWIGLU ? 5632 : 4096) : (rows > 1024 ? 4096 : 3072))
                                            : (a.M <= (wide ? 16 : 8) ? 8192 : (wide ? 5120 : 4096));
    if (a.K % 512 || a.K < 1024 || (rows <= round && a.K <= longest)) return 0;
    // ... whose blocks have w1 and w3 at once: nf4, us, 2 / 16 / 32 rows, 4096 x 2048 10.4 / 10.4 / 11.9 | 9.8 / 9.6 / 9.9, x 3072 10.8 / 10.9 / 12.5 | 10.7 / 10.7 /
    // 12.3, x 3584 10.1 / 10.3 / 12.2 | 11.1 / 11.2 / 12.8, x 4096 10.7 / 11.1 / 13.0 | 11.8 / 11.8 / 14.0, x 5120 15.3 / 16.1 / 18.7 | 12.9 / 13.4 / 16.0
    if (kind == JSGRAD_W_NF4 && epi == GEPI_SWIGLU && a.N <= round && a.K > 3072 && a.K <= 4096) return 0;
  }
  const GroupChoice c = choose_group(epi, kind, a);
  if (c.shape < 0) return pin ? fail("jsgrad_hip_gemm: no tile shape") : 0;
  if (!pin && kind == JSGRAD_W_NF4 && a.N <= 16 * state().cu_count && epi != GEPI_SWIGLU) {
    // nf4, one round of that kernel's blocks.  9 to 16 rows: its time is nearly a line in K, this one's has the steps of its turns; us, 12 / 16 rows, that | this
    // one: 3072 x 5120 9.4 / 9.5 | 9.0 / 9.1, x 6144 9.7 / 10.1 | 10.2 / 10.3, x 7168 10.2 / 10.8 | 9.8 / 9.9, x 8192 10.6 /
    // 11.2 | 11.3 / 11.4, 2560 x 8192 10.6 / 11.1 | 9.9 / 10.1.  At most 8 rows: 4096 x 10240 12.7 | 12.7, x 11264 12.7 | 13.4, x 12288 13.0 | 13.8, x 14336 15.2 | 14.9.
    if (a.M > 8 && a.M <= 16 && a.K > 5120 && a.K <= 8192 && c.us > 7.05f + 0.00047f * a.K) return 0;
    if (a.M <= 8 && a.N > 3072 && a.K > 10240 && a.K <= 12288) return 0;
  }
  *taken = true;
  return run_group(epi, kind, a, c, prof_kind);
}

}  // namespace jsg
