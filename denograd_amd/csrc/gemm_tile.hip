// Several-row linear layers with more rows than the weight-streaming kernels take (gemm.hip): y[M][N] = x[M][K] . W[N][K]^T on
// the gfx950 matrix cores, fp16 operands, float accumulation, fp16 out.
//
// What the reference computes (/root/reference/jsgrad/tensor.ts:2593-2605 `dot`, :3800 `linear`; Int8Linear.call
// /root/reference/jsgrad/models/llama3.ts:35; NF4Linear.call :91-97): with more than one input row the weight operand is
// expanded over the rows, so a quantised weight is first realised in fp16, W = RN16(code * scale), and the products of
// two fp16 values are then summed in float.  So it is here.  With many rows `realise_kernel` writes that matrix once per call
// (int8 8B w1|w3: 117 MB in, 235 MB out, ~60 us, where the product takes 5.4 ms at 32768 rows) and the fp16 kernels serve the
// three formats.  With some hundred rows or fewer the writing and reading of the realised matrix would be most of the
// time; `qtile_kernel` keeps the codes in LDS and dequantises a fragment as it is read.  In between, and without memory, the kernel of
// gemm_staged.hip has sizes where it comes first.
//
// Both operands are K-contiguous in memory (x rows, W rows), so an operand fragment of v_mfma_f32_16x16x32_f16 (8 K elements
// of one row per lane) is one 16-byte LDS read.  The 16x16 instruction is used because the chip is power-limited under this
// load: registers only, random data, it sustains 1.87 PFLOP/s at 1.90 GHz, the 32x32 one 1.62 at 1.68 GHz.
// K tiles of 64: a row of a tile is one 128-byte line.  Tiles come by direct global-to-LDS loads: a wavefront's load fills
// 1 KiB of LDS in lane order, i.e. eight rows, and the lanes pick their 16-byte piece of the row so that piece p of row r
// lands at position p ^ (r & 7): fragment reads of 16 rows then hit different banks without padding, which such a load
// could not produce.  The loads are written as assembly, because the compiler, which sees LDS written, would drain them
// before every LDS read.
//
// Eight wavefronts, two per SIMD, as two groups that take turns (half a phase apart, a barrier per turn): while one group's
// matrix instructions run, the other reads its next fragments and asks for tiles further on.
#include <algorithm>

#include "gemm_tile.h"

namespace jsg {

// ---- epilogue of one wavefront: R16 x C16 tiles of 16x16 outputs.  The weight fragment is the first MFMA operand, so a lane
// holds output row lane % 16 and the four neighbouring columns 4 * (lane / 16) + 0..3 of a tile.  Stored from there an
// instruction would touch 16 rows with 32 bytes each (4 % on a K = 4096 product); the wavefront turns RB row tiles at a time through
// its own piece of LDS and reads them back as 16-byte pieces along the rows, so stores, residual and rope table move whole
// lines.  val(i, j, c): accumulator c of row tile i, column tile j as a float.
template <int EPI, int R16, int C16, int RB, typename F>
__device__ __forceinline__ void tile_epilogue(const GemmArgs &a, _Float16 *ep, int mrow, int ncol, const F &val) {
  constexpr int CW = C16 * 16, RS = CW + 8, CPR = CW / 8, PASS = RB * 16 * CPR / 64;
  static_assert(R16 % RB == 0 && PASS >= 1 && 64 % CPR == 0, "whole passes of 64 lanes");
  const int lane = threadIdx.x & 63, l16 = lane & 15, lq = lane >> 4;
#pragma unroll
  for (int i0 = 0; i0 < R16; i0 += RB) {
    // the residual of these rows is requested before they are turned
    h8_t res[EPI == GEPI_STORE ? PASS : 1];
    if constexpr (EPI == GEPI_STORE) {
      if (a.residual) {
#pragma unroll
        for (int p = 0; p < PASS; p++) {
          const int q = p * 64 + lane, m = min(mrow + i0 * 16 + q / CPR, a.M - 1);
          res[p] = *(const h8_t *)&a.residual[(size_t)m * a.N + ncol + (q % CPR) * 8];
        }
      }
    }
#pragma unroll
    for (int i = 0; i < RB; i++)
#pragma unroll
      for (int j = 0; j < C16; j++) {
        h4_t o;
#pragma unroll
        for (int c = 0; c < 4; c++) o[c] = (_Float16)val(i0 + i, j, c);
        *(h4_t *)&ep[(i * 16 + l16) * RS + j * 16 + lq * 4] = o;
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the wavefront's own writes, before its own reads
#pragma unroll
    for (int p = 0; p < PASS; p++) {
      const int q = p * 64 + lane, row = q / CPR, piece = q % CPR;
      const int m = mrow + i0 * 16 + row, n = ncol + piece * 8;
      const h8_t v = *(const h8_t *)&ep[row * RS + piece * 8];
      if (m >= a.M) continue;
      store_piece<EPI>(a, m, n, v, res[EPI == GEPI_STORE ? p : 0]);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the reads, before the next rows overwrite the piece
  }
}

// ---- K parts: every part leaves its sums in the workspace, the last of a tile's parts to arrive adds them in K order, so the
// result does not depend on who is last.  False: this block was not the last.
// Parts run on different XCDs: stores and loads go to the point all of them share (cache policy 16: device scope), and the
// count goes up once the block's stores are acknowledged.  The part is in the vector offset: behind a 16-byte store with its
// offset in a scalar register the compiler overwrites the first data register too early (sums came out with every fourth
// value zero).
// RB: rows of accumulators fetched at a time, where there are no registers for all of a part
template <int TM, int TN, int SUMS, int RB = TM> __device__ __forceinline__ bool sum_parts(const TileArgs &t, const TileId &id, int wave, f4_t (&acc)[TM][TN]) {
  __shared__ int last;
  const __amdgpu_buffer_rsrc_t rw = wave_buffer(t.ws + (size_t)id.tile * t.split * SUMS, (uint32_t)t.split * SUMS * 4u);
  const uint32_t o0 = ((uint32_t)wave * TM * TN * 64 + (threadIdx.x & 63)) * 16;
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4_t, acc[i][j]), rw, o0 + (uint32_t)id.part * SUMS * 4u + (i * TN + j) * 1024, 0, 16);
  wait_loads<0>();
  turn_barrier();
  if (threadIdx.x == 0) {
    const int old = __hip_atomic_fetch_add(&t.counters[id.tile], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    last = old == t.split - 1;
    if (last) __hip_atomic_store(&t.counters[id.tile], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // for the next launch
  }
  __syncthreads();
  if (!last) return false;
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++) acc[i][j] = __builtin_bit_cast(f4_t, __builtin_amdgcn_raw_buffer_load_b128(rw, o0 + (i * TN + j) * 1024, 0, 16));
  for (int p = 1; p < t.split; p++) {
#pragma unroll
    for (int i0 = 0; i0 < TM; i0 += RB) {
      f4_t u[RB][TN];
#pragma unroll
      for (int i = 0; i < RB; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
          u[i][j] = __builtin_bit_cast(f4_t, __builtin_amdgcn_raw_buffer_load_b128(rw, o0 + (uint32_t)p * SUMS * 4u + ((i0 + i) * TN + j) * 1024, 0, 16));
#pragma unroll
      for (int i = 0; i < RB; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i0 + i][j] += u[i][j];
    }
  }
  return true;
}

// ---------------------------------------------------------------- 256 x 256
//
// Wavefront (g, wn) owns rows 128 g .. +127 and columns 64 wn .. +63 as four quadrants of 64 x 32; a phase of a K tile is one
// quadrant (16 matrix instructions, ~270 cycles): A0 B0 | A0 B1 | A1 B1 | A1 B0, so a tile costs 24 fragment reads and
// fits 210 registers.  Time runs in slots separated by barriers; group 0 reads in slot 2p and computes in slot 2p + 1 of
// phase p, group 1 one slot later.  Two LDS buffers of 64 KiB: the part of a buffer that both groups have read is refilled
// at once with the tile after next (A0 read in slots 0 and 1, refilled in slots 2 and 3; B0 in 4 and 5; B1, read in 2 and
// 3, in 6 and 7; A1, read in 4 and 5, in 8 and 9), so every load has 11 slots (3000 cycles) to arrive and five pairs of a
// wavefront's loads may be outstanding when a phase needs the sixth.
// Tiles behind the last whole round of blocks may come in K parts (t.whole, t.split), so that the last round is a short one: us, as chosen without |
// with, launches one after the other, 1200 x 4096 x 14336 162 | 135, w1|w3 of 14336 x 4096 behind 1600 rows 390 | 358, 3300 x 6144 x 4096 160 | 148, 4099 x 4096 x
// 14336 449 | 391, 8192 x 3072 x 8192 332 | 314.  ms of prompts, 8 layers of the 8B shape, nf4: 1200 6.06 | 5.51, 1600 7.26 | 6.84, 4099 15.4 | 14.7, 6000
// 21.6 | 20.8 (two runs differ by 0.5 %).
// Measured (fp16): 32768 x 28672 x 4096 1420, 32768 x 4096 x 14336 1430-1450, 4096^3 1410 TFLOP/s (1050-1110 for the kernel
// with 32x32 instructions and tiles through registers it replaces; the same loop without its epilogue 1500).
constexpr int T256_OPERAND = 256 * 128;                       // bytes of one operand tile
template <int EPI> __global__ __launch_bounds__(TILE_THREADS, 2) void tile256_kernel(TileArgs t) {
  const GemmArgs &a = t.g;
  extern __shared__ __align__(16) unsigned char tile_lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, lq = lane >> 4;
  const int g = wave >> 2, wn = wave & 3;
  constexpr int CW = EPI == GEPI_SWIGLU ? 128 : 256;
  const TileId id = tile_id<256, CW>(t, t.whole);
  const int m0 = id.m0;

  // Loads: half h of an operand is 128 rows = 16 loads of eight rows, two per wavefront.  The tile's rows are ordered by
  // who reads them: LDS row = 128 g + 64 h + .. for x, 64 wn + 32 h + .. for the weights.
  const uint32_t row_bytes = (uint32_t)a.K * 2;
  const i4_t ra = dma_rsrc(a.x + (size_t)m0 * a.K);
  const int lr = lane >> 3, lp = lane & 7;
  const uint32_t piece = (uint32_t)(lp ^ lr) * 16;            // rows of a load start at a multiple of 8
  uint32_t va[2][2], la[2][2], lb[2][2];
  i4_t rb[2][2];
#pragma unroll
  for (int h = 0; h < 2; h++)
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int idx = 2 * wave + i;
      const int ar = (idx >> 3) * 128 + h * 64 + (idx & 7) * 8, br = (idx >> 2) * 64 + h * 32 + (idx & 3) * 8;
      va[h][i] = (uint32_t)min(ar + lr, a.M - 1 - m0) * row_bytes + piece;   // rows past the end are computed and never stored
      const int src = EPI == GEPI_SWIGLU ? h * 128 + (idx >> 2) * 32 + (idx & 3) * 8 : br;   // half 0: w1 rows, half 1: w3 rows
      rb[h][i] = dma_rsrc(weight_ptr<EPI, 256>(t, id.col, src, row_bytes));
      la[h][i] = ar * 128;
      lb[h][i] = T256_OPERAND + br * 128;
    }
  const uint32_t vb = (uint32_t)lr * row_bytes + piece;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)tile_lds;
  const int nkt = a.K / TILE_BK, parts = id.tile < t.whole ? 1 : t.split, k0 = id.part * nkt / parts, nk = (id.part + 1) * nkt / parts - k0;
  // past the last tile the last one is asked for again, into a buffer nobody computes from any more
  auto load_a = [&](int kt, int h) {
    const uint32_t so = (uint32_t)(k0 + min(kt, nk - 1)) * 128, base = lds0 + (kt & 1) * 2 * T256_OPERAND;
    dma16(ra, va[h][0], so, base + la[h][0]);
    dma16(ra, va[h][1], so, base + la[h][1]);
  };
  auto load_b = [&](int kt, int h) {
    const uint32_t so = (uint32_t)(k0 + min(kt, nk - 1)) * 128, base = lds0 + (kt & 1) * 2 * T256_OPERAND;
    dma16(rb[h][0], vb, so, base + lb[h][0]);
    dma16(rb[h][1], vb, so, base + lb[h][1]);
  };

  f4_t acc[8][4];                                             // [x half, row tile][weight half, column tile]
#pragma unroll
  for (int i = 0; i < 8; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) acc[i][j] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
  h8_t af[4][2], bf[2][2][2];
  const uint32_t sw0 = (uint32_t)(lq ^ (l16 & 7)) * 16, sw1 = sw0 ^ 64;   // position of K pieces lq and lq + 4 in rows congruent to l16
  auto read_a = [&](int cur, int h) {
    const unsigned char *p = tile_lds + cur * 2 * T256_OPERAND + (g * 128 + h * 64 + l16) * 128;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      af[i][0] = *(const h8_t *)(p + i * 2048 + sw0);
      af[i][1] = *(const h8_t *)(p + i * 2048 + sw1);
    }
  };
  auto read_b = [&](int cur, int h) {
    const unsigned char *p = tile_lds + cur * 2 * T256_OPERAND + T256_OPERAND + (wn * 64 + h * 32 + l16) * 128;
#pragma unroll
    for (int j = 0; j < 2; j++) {
      bf[h][j][0] = *(const h8_t *)(p + j * 2048 + sw0);
      bf[h][j][1] = *(const h8_t *)(p + j * 2048 + sw1);
    }
  };
  auto compute = [&](int ah, int bh) {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[ah * 4 + i][bh * 2 + j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bf[bh][j][k], af[i][k], acc[ah * 4 + i][bh * 2 + j], 0, 0, 0);
    __builtin_amdgcn_s_setprio(0);
  };

  load_a(0, 0); load_b(0, 0); load_b(0, 1); load_a(0, 1);
  load_a(1, 0); load_b(1, 0); load_b(1, 1);
  wait_loads<10>();
  turn_barrier();                                             // A0 and B0 of tile 0 are there
  if (g == 1) turn_barrier();                                 // group 1 is a slot behind
  for (int kt = 0; kt < nk; kt++) {
    const int cur = kt & 1;
    read_a(cur, 0); read_b(cur, 0); load_a(kt + 1, 1);
    wait_loads<10>(); turn_barrier_lds();                     // B1 of this tile has landed
    compute(0, 0); turn_barrier();
    read_b(cur, 1); load_a(kt + 2, 0);
    wait_loads<10>(); turn_barrier_lds();                     // A1 of this tile
    compute(0, 1); turn_barrier();
    read_a(cur, 1); load_b(kt + 2, 0);
    turn_barrier_lds();
    compute(1, 1); turn_barrier();
    load_b(kt + 2, 1);
    wait_loads<10>(); turn_barrier();                         // A0 and B0 of the next tile
    compute(1, 0); turn_barrier();
  }
  if (g == 0) turn_barrier();
  wait_loads<0>();
  turn_barrier();                                             // nobody reads or fills the tiles any more

  if (parts > 1) {
    TileId in_parts = id;
    in_parts.tile -= t.whole;
    if (!sum_parts<8, 4, 65536, 2>(t, in_parts, wave, acc)) return;
  }

  constexpr int C16 = EPI == GEPI_SWIGLU ? 2 : 4;
  _Float16 *ep = (_Float16 *)tile_lds + wave * 64 * (C16 * 16 + 8);
  tile_epilogue<EPI, 8, C16, 4>(a, ep, m0 + g * 128, id.col + wn * C16 * 16, [&](int i, int j, int c) {
    if constexpr (EPI == GEPI_SWIGLU) return swiglu(acc[i][j][c], acc[i][2 + j][c]);
    else return acc[i][j][c];
  });
}

// ---------------------------------------------------------------- smaller tiles, K parts
//
// The same eight wavefronts over a BM x BN tile, each group (half the rows) as WR x 4 / WR, a phase per K tile (two groups half a phase apart as
// above), ST tiles in LDS, of which ST - 1 are on their way or being read.  Tiles of 192 and 256 rows: WR 2, i.e. 48 or 64 rows x 64
// columns to a wavefront, since a group's turn is its fragment reads: 14 or 16 of them for 24 or 32 matrix instructions, 20 with 128 x 32 (256 rows: 1-3 %).  For inputs of some dozens to some hundred rows, where 256 x 256
// tiles would leave most of the chip idle.  What bounds it, from builds with parts of the loop left out (128 x 128, 64 K
// tiles, us): nothing but barriers 3, matrix instructions 15, direct loads 18 (the 64 bytes a clock of a CU's L1), fragment
// reads 21 (each group reads alone and waits), all of it 30.  192 rows: 371 x 16384 x 2048 31.7 us, with 256 35.3 (36 % of its rows past the end);
// 700 x 6144 x 4096 45.1 | 50.2, 1100 x 16384 x 2048 85 | 96, 320 x 4096 x 14336 in parts 54.8, with 128 rows 67.8.
template <int EPI, int BM, int BN, int ST> constexpr size_t tile_lds_bytes() { return (size_t)(BM + BN) * 128 * ST; }
template <int EPI, int BM, int BN, int ST, int WR> __global__ __launch_bounds__(TILE_THREADS, 2) void tile_kernel(TileArgs t) {
  const GemmArgs &a = t.g;
  extern __shared__ __align__(16) unsigned char tile_lds[];
  constexpr int TM = BM / 32 / WR, TN = BN / 64 * WR, NLD = (BM + BN) / 64, BUF = (BM + BN) * 128;
  static_assert(EPI != GEPI_SWIGLU || TN % 2 == 0, "a wavefront holds the w1 and the w3 tile of the same columns");
  constexpr int CW = EPI == GEPI_SWIGLU ? BN / 2 : BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, lq = lane >> 4;
  const int g = wave >> 2, wr = (wave & 3) / (4 / WR), wn = (wave & 3) % (4 / WR);
  const int my_row = (g * WR + wr) * TM * 16;                 // first row of this wavefront in the tile
  const TileId id = tile_id<BM, CW>(t);
  const int m0 = id.m0;

  const uint32_t row_bytes = (uint32_t)a.K * 2;
  const i4_t ra = dma_rsrc(a.x + (size_t)m0 * a.K);
  const int lr = lane >> 3, lp = lane & 7;
  const uint32_t piece = (uint32_t)(lp ^ lr) * 16;
  constexpr int NA = BM / 64, NB = BN / 64;                   // a wavefront's loads per tile: eight rows each, 64 rows apart
  uint32_t va[NA];
  i4_t rb[NB];
#pragma unroll
  for (int i = 0; i < NA; i++) va[i] = (uint32_t)min(wave * 8 + i * 64 + lr, a.M - 1 - m0) * row_bytes + piece;
#pragma unroll
  for (int i = 0; i < NB; i++) rb[i] = dma_rsrc(weight_ptr<EPI, BN>(t, id.col, wave * 8 + i * 64, row_bytes));
  const uint32_t vb = (uint32_t)lr * row_bytes + piece;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)tile_lds + wave * 1024;
  const int nkt = a.K / TILE_BK, k0 = (int)((long long)id.part * nkt / t.split), nk = (int)((long long)(id.part + 1) * nkt / t.split) - k0;
  auto load = [&](int kt, int buf) {
    const uint32_t so = (uint32_t)(k0 + min(kt, nk - 1)) * 128, base = lds0 + buf * BUF;
#pragma unroll
    for (int i = 0; i < NA; i++) dma16(ra, va[i], so, base + i * 8192);
#pragma unroll
    for (int i = 0; i < NB; i++) dma16(rb[i], vb, so, base + BM * 128 + i * 8192);
  };

  f4_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++) acc[i][j] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
  h8_t af[2][TM], bf[2][TN];
  const uint32_t sw0 = (uint32_t)(lq ^ (l16 & 7)) * 16, sw1 = sw0 ^ 64;
  auto read = [&](int buf) {
    const unsigned char *pa = tile_lds + buf * BUF + (my_row + l16) * 128, *pb = tile_lds + buf * BUF + BM * 128 + l16 * 128;
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const uint32_t sw = k ? sw1 : sw0;
#pragma unroll
      for (int i = 0; i < TM; i++) af[k][i] = *(const h8_t *)(pa + i * 2048 + sw);
#pragma unroll
      for (int j = 0; j < TN; j++) {
        const int row = EPI == GEPI_SWIGLU ? (j < TN / 2 ? 0 : BN / 2) + (wn * (TN / 2) + j % (TN / 2 > 0 ? TN / 2 : 1)) * 16 : (wn * TN + j) * 16;
        bf[k][j] = *(const h8_t *)(pb + row * 128 + sw);
      }
    }
  };

#pragma unroll
  for (int i = 0; i < ST - 1; i++) load(i, i);
  wait_loads<(ST - 2) * NLD>();
  turn_barrier();
  if (g == 1) turn_barrier();
  int buf = 0, into = ST - 1;
  for (int kt = 0; kt < nk; kt++) {
    read(buf);
    load(kt + ST - 1, into);                                  // the buffer of tile kt - 1, which both groups have read
    wait_loads<(ST - 2) * NLD>();                             // tile kt + 1 has landed
    turn_barrier_lds();
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bf[k][j], af[k][i], acc[i][j], 0, 0, 0);
    __builtin_amdgcn_s_setprio(0);
    turn_barrier();
    buf = buf + 1 == ST ? 0 : buf + 1;
    into = into + 1 == ST ? 0 : into + 1;
  }
  if (g == 0) turn_barrier();
  wait_loads<0>();
  turn_barrier();

  if (t.split > 1 && !sum_parts<TM, TN, BM * BN>(t, id, wave, acc)) return;

  constexpr int C16 = EPI == GEPI_SWIGLU ? TN / 2 : TN, RB = TM < 4 ? TM : 4;
  _Float16 *ep = (_Float16 *)tile_lds + wave * RB * 16 * (C16 * 16 + 8);
  static_assert((size_t)8 * RB * 16 * (C16 * 16 + 8) * 2 <= tile_lds_bytes<EPI, BM, BN, ST>(), "the turning pieces fit the tiles' LDS");
  tile_epilogue<EPI, TM, C16, RB>(a, ep, m0 + my_row, id.col + wn * C16 * 16, [&](int i, int j, int c) {
    if constexpr (EPI == GEPI_SWIGLU) return swiglu(acc[i][j][c], acc[i][j + TN / 2][c]);
    else return acc[i][j][c];
  });
}

// ---------------------------------------------------------------- quantised weights, dequantised as they are read
//
// Four wavefronts side by side over a BM x BN tile, each with all BM rows of its BN / 4 columns, so that a weight is dequantised
// once per block: RN16(code * scale) of the eight codes of a fragment, then BM / 16 matrix instructions that use it.  x tiles as
// above; of the weights the codes go to LDS (a stage is 64 K elements of int8, 128 of nf4: 64 bytes of a row, four rows per 256
// bytes, piece p of row r at position p ^ (r / 4 & 3)), for nf4 with the two block scales of every row behind them.
// Fragments are read one step ahead of the matrix instructions; two or three blocks share a CU.
// Against realising first (us, int8, that | this): 57 x 5120 x 3072 15.7 + 11.3 | 11.4, 57 x 16384 x 3072 42 + 22 | 18.7,
// 371 x 16384 x 2048 27 + 34 | 40, 700 x 28672 x 4096 78 + 178 | 222, 1500 x 4096 x 4096 14 + 55 | 75.
template <int KIND> struct QFmt {
  static constexpr int KS = KIND == JSGRAD_W_I8 ? 64 : 128;   // K elements per stage: 64 bytes of codes per row
  static constexpr int SCALES = KIND == JSGRAD_W_NF4 ? 16 : 0;   // LDS bytes of scales per weight row and stage (a load brings 16 rows four times)
};
constexpr int QT_THREADS = 256;
template <int KIND, int BM, int BN> constexpr int qtile_stage() { return BM * QFmt<KIND>::KS * 2 + BN * (64 + QFmt<KIND>::SCALES); }
template <int KIND, int EPI, int BM, int BN, int ST> __global__ __launch_bounds__(QT_THREADS, 2) void qtile_kernel(TileArgs t) {
  const GemmArgs &a = t.g;
  extern __shared__ __align__(16) unsigned char tile_lds[];
  __shared__ uint32_t pairs[KIND == JSGRAD_W_NF4 ? 256 : 1];  // nf4: the two code values of a byte (element 2j is the high nibble, llama3.ts:92-94)
  constexpr int KS = QFmt<KIND>::KS, KF = KS / 32, SLABS = KS / 64;
  constexpr int TM = BM / 16, TN = BN / 64, NA = BM / 32 * SLABS, NB = BN / 64, NLD = NA + NB + (KIND == JSGRAD_W_NF4 ? TN : 0), BUF = qtile_stage<KIND, BM, BN>();
  static_assert(EPI != GEPI_SWIGLU || TN == 2, "a wavefront holds the w1 and the w3 tile of the same columns");
  constexpr int CW = EPI == GEPI_SWIGLU ? BN / 2 : BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, lq = lane >> 4;
  const TileId id = tile_id<BM, CW>(t);
  const int m0 = id.m0;
  if constexpr (KIND == JSGRAD_W_NF4) pairs[tid] = nf4_code_bits(tid >> 4) | (nf4_code_bits(tid & 15) << 16);   // read after the barrier below

  const uint32_t x_bytes = (uint32_t)a.K * 2, w_bytes = KIND == JSGRAD_W_I8 ? a.K : a.K / 2;
  const i4_t ra = dma_rsrc(a.x + (size_t)m0 * a.K);
  const uint32_t piece = (uint32_t)((lane & 7) ^ (lane >> 3)) * 16;
  constexpr int NA1 = NA / SLABS;
  uint32_t va[NA1];
#pragma unroll
  for (int i = 0; i < NA1; i++) va[i] = (uint32_t)min((wave * NA1 + i) * 8 + (lane >> 3), a.M - 1 - m0) * x_bytes + piece;
  i4_t rb[NB];
#pragma unroll
  for (int i = 0; i < NB; i++) rb[i] = dma_rsrc(weight_ptr<EPI, BN>(t, id.col, (wave * NB + i) * 16, w_bytes));
  const uint32_t vb = (uint32_t)(lane >> 2) * w_bytes + (uint32_t)((lane & 3) ^ (lane >> 4)) * 16;   // rows of a load start at a multiple of 16
  // the tile's weight row of fragment row l16 of this wavefront's column tile j
  auto frag_row = [&](int j) { return EPI == GEPI_SWIGLU ? j * (BN / 2) + wave * 16 : (wave * TN + j) * 16; };
  i4_t rs[TN];                                                // scales.  nf4: one per block of 64, a dword has those of a stage
  const uint32_t vs = (uint32_t)l16 * (a.K / 32);
#pragma unroll
  for (int j = 0; j < TN; j++) {
    const WeightRow w = weight_row<EPI, BN>(t, id.col, frag_row(j));
    rs[j] = dma_rsrc(pick(t.s, w.mat) + (size_t)w.row * (KIND == JSGRAD_W_I8 ? 1 : a.K / 64));
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)tile_lds;
  const int nst = a.K / KS, k0 = (int)((long long)id.part * nst / t.split), nk = (int)((long long)(id.part + 1) * nst / t.split) - k0;
  auto load = [&](int kt, int buf) {
    const uint32_t k = (uint32_t)(k0 + min(kt, nk - 1)), base = lds0 + buf * BUF;
#pragma unroll
    for (int sl = 0; sl < SLABS; sl++)
#pragma unroll
      for (int i = 0; i < NA1; i++) dma16(ra, va[i], k * (KS * 2) + sl * 128, base + sl * BM * 128 + (wave * NA1 + i) * 1024);
#pragma unroll
    for (int i = 0; i < NB; i++) dma16(rb[i], vb, k * 64, base + BM * KS * 2 + (wave * NB + i) * 1024);
    if constexpr (KIND == JSGRAD_W_NF4)
#pragma unroll
      for (int j = 0; j < TN; j++) dma4(rs[j], vs, k * 4, base + BM * KS * 2 + BN * 64 + (wave * TN + j) * 256);
  };

  f4_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++) acc[i][j] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
  h8_t af[2][TM];
  uint2 bq[2][TN];                                            // eight codes (nf4: in the first word)
  h2_t bs[2][TN];                                             // nf4: the scales of the stage's two blocks
  auto read = [&](int buf, int f) {
    const unsigned char *pa = tile_lds + buf * BUF + (f / 2) * BM * 128 + l16 * 128, *pb = tile_lds + buf * BUF + BM * KS * 2;
    const uint32_t sw = (uint32_t)(((f & 1) * 4 + lq) ^ (l16 & 7)) * 16;
#pragma unroll
    for (int i = 0; i < TM; i++) af[f & 1][i] = *(const h8_t *)(pa + i * 2048 + sw);
#pragma unroll
    for (int j = 0; j < TN; j++) {
      const unsigned char *pr = pb + (frag_row(j) + l16) * 64;
      if constexpr (KIND == JSGRAD_W_I8) bq[f & 1][j] = *(const uint2 *)(pr + (uint32_t)((f * 2 + (lq >> 1)) ^ (l16 >> 2)) * 16 + (lq & 1) * 8);
      else {
        bq[f & 1][j].x = *(const uint32_t *)(pr + (uint32_t)(f ^ (l16 >> 2)) * 16 + lq * 4);
        bs[f & 1][j] = *(const h2_t *)(pb + BN * 64 + (wave * TN + j) * 256 + l16 * 4);
      }
    }
  };
  // int8: one scale per row.  They come through LDS as well, in front of everything: a load to a register would be waited for
  // with all later loads, which the compiler does not count.
  h2_t scale[TN];
  if constexpr (KIND == JSGRAD_W_I8)
#pragma unroll
    for (int j = 0; j < TN; j++) dma4(rs[j], (uint32_t)(lane & 7) * 4, 0, lds0 + ST * BUF + (wave * TN + j) * 256);
#pragma unroll
  for (int i = 0; i < ST; i++) load(i, i);
  wait_loads<(ST - 1) * NLD>();
  turn_barrier_lds();
  if constexpr (KIND == JSGRAD_W_I8)
#pragma unroll
    for (int j = 0; j < TN; j++) {
      const _Float16 v = *(const _Float16 *)(tile_lds + ST * BUF + (wave * TN + j) * 256 + l16 * 2);
      scale[j] = h2_t{v, v};
    }
  auto compute = [&](int f) {
#pragma unroll
    for (int j = 0; j < TN; j++) {
      u4_t o;
      if constexpr (KIND == JSGRAD_W_I8) {
        uint32_t lo, hi;
        i8x4_to_h2x2(bq[f & 1][j].x, lo, hi); o.x = pk_mul_h2(lo, scale[j]); o.y = pk_mul_h2(hi, scale[j]);
        i8x4_to_h2x2(bq[f & 1][j].y, lo, hi); o.z = pk_mul_h2(lo, scale[j]); o.w = pk_mul_h2(hi, scale[j]);
      } else {
        const _Float16 s1 = f / 2 ? bs[f & 1][j].y : bs[f & 1][j].x;
        const h2_t s = {s1, s1};
        const uint32_t c = bq[f & 1][j].x;
        o.x = pk_mul_h2(pairs[c & 0xffu], s);
        o.y = pk_mul_h2(pairs[(c >> 8) & 0xffu], s);
        o.z = pk_mul_h2(pairs[(c >> 16) & 0xffu], s);
        o.w = pk_mul_h2(pairs[c >> 24], s);
      }
      const h8_t b = __builtin_bit_cast(h8_t, o);
#pragma unroll
      for (int i = 0; i < TM; i++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b, af[f & 1][i], acc[i][j], 0, 0, 0);
    }
  };

  read(0, 0);
  int buf = 0;
  for (int kt = 0; kt < nk; kt++) {
#pragma unroll
    for (int f = 0; f < KF; f++) {
      if (f < KF - 1) read(buf, f + 1);
      else {
        // every fragment of this stage is in registers: its buffer is refilled, the next stage has landed
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        wait_loads<(ST - 2) * NLD>();
        turn_barrier();
        load(kt + ST, buf);
        buf = buf + 1 == ST ? 0 : buf + 1;
        read(buf, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      compute(f);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  wait_loads<0>();
  turn_barrier();
  if (t.split > 1 && !sum_parts<TM, TN, BM * BN>(t, id, wave, acc)) return;

  constexpr int C16 = EPI == GEPI_SWIGLU ? 1 : TN, RB = 4;
  _Float16 *ep = (_Float16 *)tile_lds + wave * RB * 16 * (C16 * 16 + 8);
  static_assert((size_t)4 * RB * 16 * (C16 * 16 + 8) * 2 <= (size_t)ST * BUF, "the turning pieces fit the stages' LDS");
  tile_epilogue<EPI, TM, C16, RB>(a, ep, m0, id.col + wave * C16 * 16, [&](int i, int j, int c) {
    if constexpr (EPI == GEPI_SWIGLU) return swiglu(acc[i][0][c], acc[i][1][c]);
    else return acc[i][j][c];
  });
}

// ---------------------------------------------------------------- quantised weights, realised in fp16
//
// One matrix to out[rows][K].  A thread makes eight elements at a time, so a wavefront's store is 1 KiB
// without gaps (nf4 with 64 bytes per thread: 3.0 TB/s of codes in and halves out), and has four such pieces in flight.
template <int KIND> __global__ __launch_bounds__(256) void realise_kernel(const unsigned char *w, const _Float16 *scale, _Float16 *out, size_t pieces, int ppr) {
  __shared__ uint32_t pairs[KIND == JSGRAD_W_NF4 ? 256 : 1];
  if constexpr (KIND == JSGRAD_W_NF4) {
    pairs[threadIdx.x] = nf4_code_bits(threadIdx.x >> 4) | (nf4_code_bits(threadIdx.x & 15) << 16);
    __syncthreads();
  }
  constexpr int U = 4;
  for (size_t i0 = (size_t)blockIdx.x * (256 * U) + threadIdx.x; i0 < pieces; i0 += (size_t)gridDim.x * (256 * U)) {
    uint2 q[U];
    _Float16 s1[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const size_t i = i0 + u * 256 < pieces ? i0 + u * 256 : pieces - 1;
      if constexpr (KIND == JSGRAD_W_I8) {
        q[u] = *(const uint2 *)(w + i * 8);
        s1[u] = scale[(uint32_t)i / (uint32_t)ppr];
      } else {
        q[u].x = *(const uint32_t *)(w + i * 4);
        s1[u] = scale[i >> 3];                      // a block of 64 is eight pieces
      }
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const size_t i = i0 + u * 256;
      if (i >= pieces) break;
      const h2_t s = {s1[u], s1[u]};
      u4_t o;
      if constexpr (KIND == JSGRAD_W_I8) {
        uint32_t lo, hi;
        i8x4_to_h2x2(q[u].x, lo, hi); o.x = pk_mul_h2(lo, s); o.y = pk_mul_h2(hi, s);
        i8x4_to_h2x2(q[u].y, lo, hi); o.z = pk_mul_h2(lo, s); o.w = pk_mul_h2(hi, s);
      } else {
#pragma unroll
        for (int b = 0; b < 4; b++) o[b] = pk_mul_h2(pairs[(q[u].x >> (8 * b)) & 0xffu], s);
      }
      *(u4_t *)(out + i * 8) = o;
    }
  }
}

static int realise(int kind, const void *w, const _Float16 *scale, int rows, int K, _Float16 *out, int prof_kind) {
  const int ppr = K / 8;                                      // pieces per row
  const size_t pieces = (size_t)rows * ppr;
  JSG_REQUIRE(pieces < (size_t)1 << 32, "jsgrad_hip_gemm: a matrix of %d x %d is too large", rows, K);
  const size_t want = (pieces + 1023) / 1024;
  const int grid = (int)(want < (size_t)16 * state().cu_count ? want : (size_t)16 * state().cu_count);
  if (kind == JSGRAD_W_I8) JSG_LAUNCH(prof_kind, realise_kernel<JSGRAD_W_I8>, dim3(grid), dim3(256), 0, (const unsigned char *)w, scale, out, pieces, ppr);
  else JSG_LAUNCH(prof_kind, realise_kernel<JSGRAD_W_NF4>, dim3(grid), dim3(256), 0, (const unsigned char *)w, scale, out, pieces, ppr);
  return 0;
}

// ---------------------------------------------------------------- host side

constexpr int TILE_COUNTERS = 4096;
// What one call asks of the workspace at most: K parts' sums, and a realised matrix (w1|w3 of the 8B shape 235 MB, its lm_head 1 GB)
constexpr size_t SUMS_LIMIT = (size_t)256 << 20, REALISED_LIMIT = (size_t)2 << 30;
static __device__ int tile_counters[TILE_COUNTERS];

// 256 x 256 with K parts: only the tiles behind the last whole round of blocks come in parts
static int whole_tiles(int tiles) { return tiles / state().cu_count * state().cu_count; }
template <int EPI> static int launch_tile256(const TileArgs &t, int prof_kind) {
  constexpr int lds = 4 * T256_OPERAND;
  static bool raised = false;   // one process, one device, one thread: set once per instantiation
  if (!raised) {
    JSG_HIP(hipFuncSetAttribute((const void *)tile256_kernel<EPI>, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    raised = true;
  }
  const int tiles = ((t.g.M + 255) / 256) * (t.g.N / (EPI == GEPI_SWIGLU ? 128 : 256));
  TileArgs u = t;
  u.whole = t.split > 1 ? whole_tiles(tiles) : tiles;
  JSG_LAUNCH(prof_kind, (tile256_kernel<EPI>), dim3(u.whole + (tiles - u.whole) * t.split), dim3(TILE_THREADS), lds, u);
  return 0;
}
template <int EPI, int BM, int BN, int ST, int WR = 1> static int launch_tile(const TileArgs &t, int prof_kind) {
  constexpr int lds = (int)tile_lds_bytes<EPI, BM, BN, ST>();
  static_assert(lds + 64 <= 160 * 1024, "LDS of one compute unit");
  static bool raised = false;
  if (!raised) {
    JSG_HIP(hipFuncSetAttribute((const void *)tile_kernel<EPI, BM, BN, ST, WR>, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    raised = true;
  }
  const int tiles = ((t.g.M + BM - 1) / BM) * (t.g.N / (EPI == GEPI_SWIGLU ? BN / 2 : BN));
  JSG_LAUNCH(prof_kind, (tile_kernel<EPI, BM, BN, ST, WR>), dim3(tiles * t.split), dim3(TILE_THREADS), lds, t);
  return 0;
}

template <int KIND, int EPI, int BM, int BN, int ST> static int launch_qtile(const TileArgs &t, int prof_kind) {
  constexpr int lds = qtile_stage<KIND, BM, BN>() * ST + (KIND == JSGRAD_W_I8 ? BN * 16 : 0);
  static_assert(lds + 1100 <= 160 * 1024, "LDS of one compute unit");
  static bool raised = false;
  if (!raised) {
    JSG_HIP(hipFuncSetAttribute((const void *)qtile_kernel<KIND, EPI, BM, BN, ST>, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    raised = true;
  }
  const int tiles = ((t.g.M + BM - 1) / BM) * (t.g.N / (EPI == GEPI_SWIGLU ? BN / 2 : BN));
  JSG_LAUNCH(prof_kind, (qtile_kernel<KIND, EPI, BM, BN, ST>), dim3(tiles * t.split), dim3(QT_THREADS), lds, t);
  return 0;
}

// The shapes, with the K elements of a step and four times: us of a step of blocks that have a compute unit each, what fill adds to it
// when every unit has one (they share memory and power), us of a step of a round when there are several, and of a round's end.
// Fitted to 33 to 4096 rows over the matrices of the 1B, 3B and 8B models, each under every shape that could matter, weights in memory
// and in the last level cache, for the choice rather than for the single time (an estimate is off by 5-10 % r.m.s.).
struct TileShape { int bm, bn, bk; float step, fill, round_step, end; bool pairs = true; };   // pairs: w1|w3 as well
static const TileShape TILE_SHAPES[] = {
  {64, 64, 64, 0.19f, 0.03f, 0.22f, 0.0f, false},
  {64, 128, 64, 0.27f, 0.064f, 0.37f, 0.0f},
  {128, 128, 64, 0.38f, 0.13f, 0.63f, 0.3f},
  {192, 128, 64, 0.51f, 0.26f, 0.73f, 1.5f},
  {256, 128, 64, 0.55f, 0.32f, 0.85f, 1.0f},
  {256, 256, 64, 0.82f, 0.39f, 1.3f, 3.0f},
};
static const TileShape QTILE_SHAPES_I8[] = {{64, 64, 64, 0.25f, 0.024f, 0.18f, 0.03f, false}, {64, 128, 64, 0.35f, 0.03f, 0.36f, 0.57f}, {128, 128, 64, 0.52f, 0.087f, 0.50f, 1.2f}};
static const TileShape QTILE_SHAPES_NF4[] = {{64, 64, 128, 0.51f, 0.062f, 0.43f, 0.3f, false}, {64, 128, 128, 0.86f, 0.075f, 0.70f, 0.74f}, {128, 128, 128, 1.6f, 0.13f, 1.4f, 3.2f}};
// gemm_staged.hip
static const TileShape STAGED_SHAPES_I8[] = {{32, 128, 64, 0.48f, 0.1f, 0.36f, 0.5f, false}, {128, 128, 64, 0.88f, 0.09f, 0.61f, 1.2f}, {256, 128, 64, 1.13f, 0.16f, 1.04f, 2.5f}, {256, 256, 64, 1.1f, 0.43f, 1.7f, 6.0f}};
static const TileShape STAGED_SHAPES_NF4[] = {{32, 128, 64, 0.53f, 0.17f, 0.29f, 0.5f, false}, {128, 128, 64, 0.92f, 0.09f, 0.71f, 0.7f}, {256, 128, 64, 1.2f, 0.17f, 1.03f, 2.0f}, {256, 256, 64, 1.4f, 0.29f, 1.9f, 7.8f}};
constexpr int N_SHAPES = sizeof(TILE_SHAPES) / sizeof(TILE_SHAPES[0]), N_QSHAPES = sizeof(QTILE_SHAPES_I8) / sizeof(QTILE_SHAPES_I8[0]), N_STAGED = sizeof(STAGED_SHAPES_I8) / sizeof(STAGED_SHAPES_I8[0]);

// Which shape and how many K parts: the least of an estimate of the launch's time (4.5 us for start and first tiles; for K parts 1.7 us
// and the sums' way through memory; 256 x 256, whose blocks wait for each other's 256 KB and share the chip's power, 20 us: with less it is taken where it
// loses, 2048 x 4096 x 4096 64 | 72, 1200 x 6144 x 4096 61 | 68).  Over the measured sizes the choice is 0.9 % slower than the best shape on average.  Examples, us with weights from memory, this choice | others: 371 x 2048 x 8192 128x128 in 5 parts 26.3 | in 3 parts
// 32.2, 64x128 in 2 32.9, 256x128 in 7 34.4; 371 x 2048 x 2048 64x64 12.7 | 64x128 in 2 parts 12.4, in one 15.5; 700 x 28672 x 4096
// 256x128 185 | 256x256 188, 128x128 223; 2048 x 6144 x 4096 256x256 90 | 128x128 111, 256x128 112; int8 codes, 57 x 5120 x 3072 64x64 in
// 3 parts 11.2 | 64x128 in 5 12.4, 64x64 in 6 12.9.
struct Choice { float us; int shape, split; };
// JSG_GEMM_TILE, for tests and measurements: rows x columns of a tile, optionally with K parts, of the fp16 kernels ("128x128",
// "64x128/3"; quantised weights are then realised), of qtile_kernel ("q64x64/3") or of the staged kernel ("s256x256"); "small", "tall",
// "wide" and "db" name fp16 tiles from 64x64 (w1|w3: 64x128) to 256x256.  A tile that the output width does not allow is not taken.
struct Pin { char family = 0; int bm = 0, bn = 0, split = 1; };   // family: 't', 'q' or 's'; 0: no pin
static Pin read_pin(int epi, const GemmArgs &a) {
  Pin p;
  const char *e = pin_env(a, "JSG_GEMM_TILE");
  if (!e) return p;
  p.family = *e == 'q' || (*e == 's' && e[1] != 'm') ? *e : 't';
  const struct { const char *name; int bm, bn; } names[] = {{"small", 64, epi == GEPI_SWIGLU ? 128 : 64}, {"tall", 128, 128}, {"wide", 256, 128}, {"db", 256, 256}};
  for (const auto &n : names)
    if (!strcmp(e, n.name)) { p.bm = n.bm; p.bn = n.bn; return p; }
  sscanf(e + (p.family != 't'), "%dx%d/%d", &p.bm, &p.bn, &p.split);
  return p;
}
// tail: 256 x 256 tiles may have K parts too (tile256_kernel)
static Choice choose_tile(const TileShape *shapes, int n_shapes, int epi, int M, int weight_rows, int K, size_t ws_limit, const Pin &pin) {
  const bool tail = shapes == TILE_SHAPES;
  const int cus = state().cu_count;
  Choice best = {0.0f, -1, 1};
  for (int s = 0; s < n_shapes; s++) {
    const TileShape &c = shapes[s];
    if (weight_rows % c.bn || K % c.bk || (epi == GEPI_SWIGLU && !c.pairs)) continue;
    const int tiles = ((M + c.bm - 1) / c.bm) * (weight_rows / c.bn), nk = K / c.bk;
    for (int d = 1; d <= 16; d++) {
      const bool big = c.bm * c.bn == 65536;
      const int whole = big ? whole_tiles(tiles) : 0, in_parts = tiles - whole;
      if (d > 1 && ((big && !tail) || in_parts == 0 || nk < d || in_parts > TILE_COUNTERS || (size_t)in_parts * d * c.bm * c.bn * 4 > ws_limit)) break;
      if (d > 1 && (pin.family ? d > pin.split : nk / d * c.bk < (big ? 512 : 256) || in_parts * d > (big ? 1 : 2) * cus)) break;
      const int blocks = tiles * d, steps = (nk + d - 1) / d;
      const float fill = (float)blocks / cus;
      float us = 4.5f + (fill <= 1.0f ? (c.step + c.fill * fill) * steps + c.end : ((blocks + cus - 1) / cus) * (c.round_step * steps + c.end));
      if (d > 1 && big) us = 4.5f + (float)(whole / cus) * (c.round_step * nk + c.end) + c.round_step * steps + c.end;
      if (d > 1) us += (big ? 20.0f : 1.7f) + (float)d * c.bm * c.bn * 4 / 83e3f * (fill > 1.0f && !big ? fill : 1.0f);
      if (pin.bm == c.bm && pin.bn == c.bn && d == pin.split) us = 0.0f;   // taken
      // Parts behind whole rounds instead of a smaller tile: only where the estimate is 6 % lower.  Alone they keep what it says (4096 x 6144 x 4096 176 | 168), but
      // between the other launches of a prompt, where the chip is at its power limit, a last round that leaves units idle runs faster.  us there, smaller tile | parts, with
      // estimates that are 2 to 5.6 % lower: 3000 x 6144 x 4096 147 | 155, 4096 182 | 184 (189 | 196 on another card), 4200 x 5120 x 3072 138 | 147, 7000 x 3072 x 3072 127 |
      // 130; 7 % int8 6400 x 3072 x 3072 135 | 121, 16 % 3300 x 6144 x 4096 175 | 165, 5000 x 4096 x 4096 166 | 157.
      const bool sure = d == 1 || whole == 0 || (best.shape >= 0 && shapes[best.shape].bm == c.bm && shapes[best.shape].bn == c.bn);
      if (best.shape < 0 || us * (sure ? 1.0f : 1.06f) < best.us) best = {us, s, d};
    }
  }
  return best;
}

static size_t sums_bytes(const TileShape *shapes, const Choice &c, int M, int weight_rows) {
  if (c.split < 2) return 0;
  const int bm = shapes[c.shape].bm, bn = shapes[c.shape].bn, tiles = ((M + bm - 1) / bm) * (weight_rows / bn);
  return (size_t)(tiles - (bm * bn == 65536 ? whole_tiles(tiles) : 0)) * c.split * bm * bn * 4;
}

template <int KIND, int EPI> static int launch_qshape(int s, const TileArgs &t, int prof_kind) {
  constexpr bool I8 = KIND == JSGRAD_W_I8;
  switch (s) {
    case 0: if constexpr (EPI != GEPI_SWIGLU) return launch_qtile<KIND, EPI, 64, 64, I8 ? 4 : 3>(t, prof_kind); else break;
    case 1: return launch_qtile<KIND, EPI, 64, 128, I8 ? 4 : 3>(t, prof_kind);
    case 2: return launch_qtile<KIND, EPI, 128, 128, I8 ? 3 : 2>(t, prof_kind);
  }
  return fail("jsgrad_hip_gemm: no tile shape");
}
template <int EPI> static int launch_shape(int s, const TileArgs &t, int prof_kind) {
  switch (s) {
    case 0: if constexpr (EPI != GEPI_SWIGLU) return launch_tile<EPI, 64, 64, 4>(t, prof_kind); else break;
    case 1: return launch_tile<EPI, 64, 128, 4>(t, prof_kind);
    case 2: return launch_tile<EPI, 128, 128, 4>(t, prof_kind);
    case 3: return launch_tile<EPI, 192, 128, 3, 2>(t, prof_kind);
    case 4: return launch_tile<EPI, 256, 128, 3, 2>(t, prof_kind);
    case 5: return launch_tile256<EPI>(t, prof_kind);
  }
  return fail("jsgrad_hip_gemm: no tile shape");
}

template <int EPI> static int gemm_tiled_epi(int kind, const GemmArgs &a, int prof_kind) {
  constexpr int NMAT = EPI == GEPI_SWIGLU ? 2 : 1;            // weight rows per output column
  const void *const w[3] = {a.w0, a.w1, a.w2};
  const _Float16 *const sc[3] = {a.s0, a.s1, a.s2};
  const int n[3] = {EPI == GEPI_ROPE_KV ? a.n0 : a.N, EPI == GEPI_ROPE_KV ? a.n1 : 0, EPI == GEPI_ROPE_KV ? a.n2 : 0};   // rows on top of each other
  static int *counters = nullptr;
  if (!counters) JSG_HIP(hipGetSymbolAddress((void **)&counters, HIP_SYMBOL(tile_counters)));
  TileArgs t = tile_args(EPI, a, counters);

  const Pin pin = read_pin(EPI, a), none;
  auto pinned = [&](char family) -> const Pin & { return pin.family == family ? pin : none; };
  const size_t ws_limit = state().capturing ? 0 : SUMS_LIMIT;
  const int wrows = a.N * NMAT;
  auto run = [&](const Choice &c, float *sums, auto launch) -> int {
    JSG_REQUIRE(c.shape >= 0, "jsgrad_hip_gemm: no tile shape for %d columns", a.N);
    t.split = c.split;
    t.ws = sums;
    return launch(c.shape, t, prof_kind);
  };
  Workspace ws;
  // the K parts' sums, if there are parts, in the workspace
  auto run_whole = [&](const TileShape *shapes, int n_shapes, Choice c, const Pin &p, auto launch) -> int {
    const size_t sums = sums_bytes(shapes, c, a.M, wrows);
    if (sums && !ws.get(sums)) c = choose_tile(shapes, n_shapes, EPI, a.M, wrows, a.K, 0, p);
    return run(c, (float *)ws.p, launch);
  };

  Choice f = choose_tile(TILE_SHAPES, N_SHAPES, EPI, a.M, wrows, a.K, ws_limit, pinned('t'));
  // At most 64 rows: the group kernel, where its estimate is the least.  The estimates of the tiled kernels are without the rate at which
  // they can draw weights with so few rows (57 rows, from 12 MB on: fp16 4.6 TB/s, codes 3.9, and for codes a seventh too low below that): us,
  // theirs measured | the group kernel: fp16 16384 x 3072 25.5 | 24.2, 28672 x 4096 52.5 | 49.4; int8 16384 x 2048 15.3 | 13.6, 16384 x 3072
  // 18.8 | 17.5, 128256 x 3072 112 | 104; nf4 16384 x 3072 20.9 | 18.4, 28672 x 4096 34.5 | 31.6; with K parts level, 3072 x 8192 int8 14.9 | 15.4;
  // nf4 of 13 MB (10240 x 2560) 14.1 | 15.7, of 17 (w1|w3 of 8192 x 2048) 17.0 | 14.0.
  const GroupChoice g = pin.family ? GroupChoice() : choose_group(EPI, kind, a);
  auto group_first = [&](float us) {
    if (g.shape < 0) return false;
    const float mb = (float)((double)wrows * a.K * (kind == JSGRAD_W_F16 ? 2.0 : (kind == JSGRAD_W_I8 ? 1.0 : 0.5)) * 1e-6);
    if (g.split == 1 && mb > (kind == JSGRAD_W_NF4 ? 14.0f : 12.0f)) us = kind == JSGRAD_W_F16 ? std::max(us, 3.8f + mb / 4.6f) : std::max(us * 1.15f, 3.8f + mb / 3.9f);
    return g.us < us;
  };
  if (kind == JSGRAD_W_F16) {
    if (group_first(f.us)) return run_group(EPI, kind, a, g, prof_kind);
    return run_whole(TILE_SHAPES, N_SHAPES, f, pinned('t'), launch_shape<EPI>);
  }

  // Quantised: dequantised as read (qtile_kernel), dequantised on the way into LDS (gemm_staged.hip), or realised first, whichever is
  // estimated to be done first; without memory for the realised matrix (a capture, a full device) one of the first two.  Realising:
  // codes in and halves out at 8.5 TB/s, slower where the last level cache cannot hold them until they are read (w1|w3 of the 8B
  // shape, 352 MB: 60 us), a launch per matrix.  On the matrices of the 8B model int8 is realised from 1000 to 1700 rows on, nf4 from 320 to
  // 640 (with narrow bands back and forth where a round of blocks ends); for w1|w3 the staged kernel comes first in between.
  const float moved = (float)((double)wrows * a.K * (kind == JSGRAD_W_I8 ? 3.0 : 2.5)), big = moved - 120e6f;
  const float realise_us = pin.family == 't' ? 0.0f : moved / 8.5e6f + (big > 0.0f ? big / 18e6f : 0.0f) + 3.7f + 4.5f * (EPI == GEPI_STORE ? 0 : EPI == GEPI_SWIGLU ? 1 : 2);
  const TileShape *qs = kind == JSGRAD_W_I8 ? QTILE_SHAPES_I8 : QTILE_SHAPES_NF4;
  // qtile_kernel brings scales by direct loads of four bytes; a pointer between two of those (a slice) is read half by half elsewhere
  const bool dwords = (((uintptr_t)a.s0 | (uintptr_t)a.s1 | (uintptr_t)a.s2) & 3) == 0;
  const Choice q = dwords ? choose_tile(qs, N_QSHAPES, EPI, a.M, wrows, a.K, ws_limit, pinned('q')) : Choice{0.0f, -1, 1};
  const TileShape *ss = kind == JSGRAD_W_I8 ? STAGED_SHAPES_I8 : STAGED_SHAPES_NF4;
  const Choice st = choose_tile(ss, N_STAGED, EPI, a.M, wrows, a.K, 0, pinned('s'));   // takes every call
  const bool staged = q.shape < 0 || st.us < q.us;
  // int8 rows of 512 codes: a block of the group kernel, which has its unit to itself, is over in a turn or two, and there are rounds of them.  us, 16 rows,
  // that | the staged kernel, several of whose blocks share a unit: 65536 x 512 12.7 | 11.4, 128256 x 512 23.4 | 17.5 (x 1024 32.5 | 35 and more).
  if constexpr (EPI != GEPI_SWIGLU)
    if (!pin.family && kind == JSGRAD_W_I8 && a.M <= 32 && a.K <= 512 && wrows > 192 * state().cu_count) return gemm_staged(EPI, kind, 32, 128, a, prof_kind);
  if (group_first(std::min(staged ? st.us : q.us, f.shape >= 0 ? f.us + realise_us : st.us))) return run_group(EPI, kind, a, g, prof_kind);
  const size_t bytes = (size_t)wrows * a.K * 2;
  if (f.shape >= 0 && f.us + realise_us < (staged ? st.us : q.us) && bytes <= REALISED_LIMIT) {
    // into the workspace, with the K parts' sums behind it
    const size_t sums = sums_bytes(TILE_SHAPES, f, a.M, wrows);
    if (!ws.get(bytes + sums) && sums && ws.get(bytes)) f = choose_tile(TILE_SHAPES, N_SHAPES, EPI, a.M, wrows, a.K, 0, pinned('t'));
    if (ws.p) {
      _Float16 *const out = (_Float16 *)ws.p;
      const int n_mats = EPI == GEPI_ROPE_KV ? 3 : NMAT;
      for (int m = 0, base = 0; m < n_mats; m++) {
        const int rows = EPI == GEPI_ROPE_KV ? n[m] : a.N;
        if (int rc = realise(kind, w[m], sc[m], rows, a.K, out + (size_t)base * a.K, prof_kind)) return rc;
        base += rows;
      }
      t.b[0] = out;
      t.b[1] = t.b[2] = out + (size_t)a.N * a.K;
      t.b_end[0] = t.b_end[1] = a.N;
      return run(f, (float *)((unsigned char *)ws.p + bytes), launch_shape<EPI>);
    }
  }
  if (staged) return gemm_staged(EPI, kind, ss[st.shape].bm, ss[st.shape].bn, a, prof_kind);
  return kind == JSGRAD_W_I8 ? run_whole(qs, N_QSHAPES, q, pinned('q'), launch_qshape<JSGRAD_W_I8, EPI>) : run_whole(qs, N_QSHAPES, q, pinned('q'), launch_qshape<JSGRAD_W_NF4, EPI>);
}

int gemm_tiled(int epi, int kind, const GemmArgs &a, int prof_kind) {
  if (epi == GEPI_STORE) return gemm_tiled_epi<GEPI_STORE>(kind, a, prof_kind);
  if (epi == GEPI_ROPE_KV) return gemm_tiled_epi<GEPI_ROPE_KV>(kind, a, prof_kind);
  return gemm_tiled_epi<GEPI_SWIGLU>(kind, a, prof_kind);
}

}  // namespace jsg
