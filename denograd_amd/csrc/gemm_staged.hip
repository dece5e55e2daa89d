// Several-row linear layers with int8 or NF4 weights that are dequantised on their way into LDS: y[M][N] = x[M][K] . W[N][K]^T; what the
// reference computes is in gemm_tile.hip, whose kernels are faster for most sizes.  This one needs no memory of its own, takes scales at any
// even address and rows of any length, and is the faster one where realising the matrix in fp16 is out of the question (a graph
// capture, a full device) or costs too much for the rows there are: gemm_tile.hip chooses (us, the tiled kernels | this one:
// w1|w3 of the 8B shape, int8 512 rows 139 | 122, 1000 rows 247 | 236, nf4 200 rows 106 | 93, 371 rows 152 | 130, 512 rows 157 | 135;
// captured, 8192 rows, int8 1970 | 1740, nf4 3050 | 1940).
//
// A thread takes 16 bytes of codes of a row to registers a K tile ahead, and RN16(code * scale) of them to LDS: the weight tile there is
// exactly the realised matrix, made once per block; v_pk_mul_f16 of the exact fp16 code by the fp16 scale is the single rounding.
// 256 threads = 4 wavefronts laid out WGM x WGN; a wavefront owns TM x TN tiles of 32x32 outputs and walks K in steps of 16 with
// v_mfma_f32_32x32x16_f16.  Both operands are K-contiguous in memory, so a lane's 8-element operand fragment is one 128-bit LDS read.
// LDS rows are padded by 8 halves, which spreads the 32 rows of a fragment read over all banks.
//
// Two loop shapes.  128x128, 256x128, or 32x128 for few rows, out of one LDS buffer (two barriers per K tile, the next tile prefetched
// into registers) with two or three blocks per CU, whose wavefronts cover each other's barriers and conversions.  256x256 out of two, one block per CU (one
// wavefront per SIMD): one barrier per K tile, and the instruction order of a K tile is spelled out so that fragment reads,
// conversion, LDS writes and the requests of the tile after next sit between the matrix instructions.
#include <type_traits>

#include "gemm.h"

namespace jsg {

typedef float f16_t __attribute__((ext_vector_type(16)));

constexpr int STAGED_BK = 64;         // K elements per LDS tile
constexpr int STAGED_STRIDE = 72;     // halves per LDS row (64 + 8 padding)
constexpr int STAGED_THREADS = 256;

template <int KIND, int EPI, int WGM, int WGN, int TM, int TN, bool DB = false>
__global__ __launch_bounds__(STAGED_THREADS, (TM * TN > 8 ? 1 : (TM * TN > 4 ? 2 : 3))) void staged_kernel(GemmArgs a) {
  static_assert(WGM * WGN == 4, "four wavefronts");
  static_assert(EPI != GEPI_SWIGLU || TN % 2 == 0, "a wavefront holds the w1 and the w3 tile of the same columns");
  constexpr int BM = WGM * TM * 32, BN = WGN * TN * 32, LS = STAGED_STRIDE;
  constexpr int A_LOADS = BM / 32;                                                    // 16-byte loads per thread per K tile
  constexpr int B_ROWS_PER_PASS = KIND == JSGRAD_W_I8 ? 64 : 128;
  constexpr int B_CHUNKS = STAGED_THREADS / B_ROWS_PER_PASS;                             // 16-byte chunks per row of the K tile
  constexpr int B_LOADS = BN / B_ROWS_PER_PASS;
  static_assert(B_LOADS >= 1, "tile too narrow for this weight format");
  constexpr int BUF = (BM + BN) * LS;                     // halves per LDS buffer
  extern __shared__ __align__(16) _Float16 staged_lds[];   // one or two buffers of [BM + BN rows][LS], then 32 spare bytes and the 256-entry NF4 table
  _Float16 *As = staged_lds, *Bs = staged_lds + BM * LS, *lut = staged_lds + (DB ? 2 : 1) * BUF;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WGN, wn = wave % WGN;
  const int l32 = lane & 31, lg = lane >> 5;

  // NF4: one table entry per BYTE, the two code values of its nibbles as a packed pair (element 2j is the high nibble,
  // llama3.ts:92-94), so a byte costs one LDS read and one packed multiplication by the block scale
  uint32_t *pairs = (uint32_t *)(lut + 16);
  if constexpr (KIND == JSGRAD_W_NF4) {
    pairs[tid] = nf4_code_bits(tid >> 4) | (nf4_code_bits(tid & 15) << 16);   // from literals: no memory round trip at the head of the launch
  }

  // ---- tile id: XCD-contiguous, then grouped so that neighbouring ids share an x tile column-block
  const int tiles_m = (a.M + BM - 1) / BM, tiles_n = a.N / (EPI == GEPI_SWIGLU ? BN / 2 : BN);
  const int nblocks = tiles_m * tiles_n;
  int bid = blockIdx.x;
  {
    const int per = nblocks / 8;
    if (bid < per * 8) bid = (bid & 7) * per + (bid >> 3);
  }
  constexpr int GROUP = 4;                                // weight tiles are half or a quarter of the bytes of an x tile: more of them per XCD
  const int in_group = GROUP * tiles_n;
  const int first_m = (bid / in_group) * GROUP;
  const int gsz = min(tiles_m - first_m, GROUP);
  const int tm_ = first_m + (bid % in_group) % gsz, tn_ = (bid % in_group) / gsz;
  const int m0 = tm_ * BM;
  const int n0_out = tn_ * (EPI == GEPI_SWIGLU ? BN / 2 : BN);   // first output column of this tile

  // ---- B source of every row this thread loads: (matrix, row) is fixed over the K loop
  const unsigned char *bsrc[B_LOADS];
  h2_t bscale[B_LOADS];
  const _Float16 *bscale_ptr[B_LOADS];
  const int brow_t = tid / B_CHUNKS, bchunk = tid % B_CHUNKS;
#pragma unroll
  for (int i = 0; i < B_LOADS; i++) {
    const int r = brow_t + i * B_ROWS_PER_PASS;      // row inside the B tile
    const void *w; const _Float16 *s; int row;
    if constexpr (EPI == GEPI_SWIGLU) {
      const bool up = r >= BN / 2;
      w = up ? a.w1 : a.w0; s = up ? a.s1 : a.s0; row = n0_out + (up ? r - BN / 2 : r);
    } else if constexpr (EPI == GEPI_ROPE_KV) {
      const int n = n0_out + r;
      if (n < a.n0) { w = a.w0; s = a.s0; row = n; }
      else if (n < a.n0 + a.n1) { w = a.w1; s = a.s1; row = n - a.n0; }
      else { w = a.w2; s = a.s2; row = n - a.n0 - a.n1; }
    } else { w = a.w0; s = a.s0; row = n0_out + r; }
    const size_t e = (size_t)row * a.K;              // element offset of the row
    if constexpr (KIND == JSGRAD_W_I8) { bsrc[i] = (const unsigned char *)w + e + bchunk * 16; const _Float16 sv = s[row]; bscale[i] = h2_t{sv, sv}; }
    else { bsrc[i] = (const unsigned char *)w + e / 2 + bchunk * 16; bscale_ptr[i] = s + e / 64; }
  }
  const unsigned char *asrc[A_LOADS];
  const int arow_t = tid / 8, achunk = tid % 8;
#pragma unroll
  for (int i = 0; i < A_LOADS; i++) {
    int m = m0 + arow_t + i * 32;
    if (m >= a.M) m = a.M - 1;                        // rows past the end are computed and never stored
    asrc[i] = (const unsigned char *)(a.x + (size_t)m * a.K) + achunk * 16;
  }

  f16_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;

  u4_t ga[A_LOADS], gb[B_LOADS];
  _Float16 gs[B_LOADS];
  auto issue_a = [&](int kt) {
    const size_t ko = (size_t)kt * STAGED_BK;
#pragma unroll
    for (int i = 0; i < A_LOADS; i++) ga[i] = *(const u4_t *)(asrc[i] + ko * 2);
  };
  auto issue_b = [&](int kt, int lo = 0, int hi = 1 << 30) {
    const size_t ko = (size_t)kt * STAGED_BK;
#pragma unroll
    for (int i = 0; i < B_LOADS; i++) {
      if (i < lo || i >= hi) continue;
      if constexpr (KIND == JSGRAD_W_I8) gb[i] = *(const u4_t *)(bsrc[i] + ko);
      else { gb[i] = *(const u4_t *)(bsrc[i] + ko / 2); gs[i] = bscale_ptr[i][kt]; }
    }
  };
  auto issue = [&](int kt) { issue_a(kt); issue_b(kt); };
  auto commit_a = [&](int buf) {
#pragma unroll
    for (int i = 0; i < A_LOADS; i++) *(u4_t *)&As[buf * BUF + (arow_t + i * 32) * LS + achunk * 8] = ga[i];
  };
  auto commit_b = [&](int buf, int lo = 0, int hi = 1 << 30) {
#pragma unroll
    for (int i = 0; i < B_LOADS; i++) {
      if (i < lo || i >= hi) continue;
      _Float16 *dst = &Bs[buf * BUF + (brow_t + i * B_ROWS_PER_PASS) * LS];
      if constexpr (KIND == JSGRAD_W_I8) {
        u4_t o0, o1;
        uint32_t lo, hi;
        i8x4_to_h2x2(gb[i].x, lo, hi); o0.x = pk_mul_h2(lo, bscale[i]); o0.y = pk_mul_h2(hi, bscale[i]);
        i8x4_to_h2x2(gb[i].y, lo, hi); o0.z = pk_mul_h2(lo, bscale[i]); o0.w = pk_mul_h2(hi, bscale[i]);
        i8x4_to_h2x2(gb[i].z, lo, hi); o1.x = pk_mul_h2(lo, bscale[i]); o1.y = pk_mul_h2(hi, bscale[i]);
        i8x4_to_h2x2(gb[i].w, lo, hi); o1.z = pk_mul_h2(lo, bscale[i]); o1.w = pk_mul_h2(hi, bscale[i]);
        *(u4_t *)(dst + bchunk * 16) = o0;
        *(u4_t *)(dst + bchunk * 16 + 8) = o1;
      } else {
        // 16 bytes = 32 elements; the high nibble of a byte is the even element (llama3.ts:92-94)
        const h2_t sv = {gs[i], gs[i]};
        uint32_t wds[4] = {gb[i].x, gb[i].y, gb[i].z, gb[i].w};
#pragma unroll
        for (int d = 0; d < 4; d++) {
          u4_t o;
          uint32_t outw[4];
#pragma unroll
          for (int b = 0; b < 4; b++) {
            const uint32_t byte = (wds[d] >> (8 * b)) & 0xffu;
            outw[b] = pk_mul_h2(pairs[byte], sv);
          }
          o.x = outw[0]; o.y = outw[1]; o.z = outw[2]; o.w = outw[3];
          *(u4_t *)(dst + bchunk * 32 + d * 8) = o;
        }
      }
    }
  };
  auto commit = [&](int buf = 0) { commit_a(buf); commit_b(buf); };

  auto frags = [&](int buf, int kk, h8_t *af, h8_t *bf) {
#pragma unroll
    for (int i = 0; i < TM; i++) af[i] = *(const h8_t *)&As[buf * BUF + ((wm * TM + i) * 32 + l32) * LS + kk * 16 + lg * 8];
#pragma unroll
    for (int j = 0; j < TN; j++) {
      int rbase;
      if constexpr (EPI == GEPI_SWIGLU) rbase = j < TN / 2 ? (wn * (TN / 2) + j) * 32 : BN / 2 + (wn * (TN / 2) + j - TN / 2) * 32;
      else rbase = (wn * TN + j) * 32;
      bf[j] = *(const h8_t *)&Bs[buf * BUF + (rbase + l32) * LS + kk * 16 + lg * 8];
    }
  };
  auto mfmas = [&](const h8_t *af, const h8_t *bf) {
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(bf[j], af[i], acc[i][j], 0, 0, 0);   // D = W tile . x tile^T
  };

  const int nk = a.K / STAGED_BK;
  issue(0);
  if constexpr (KIND == JSGRAD_W_NF4) __syncthreads();   // the code table is in LDS
  if constexpr (DB) {
    // Two LDS buffers, one barrier per K tile: while the matrix cores work on tile kt out of one buffer, the same
    // wavefront turns the registers of tile kt+1 into the other buffer and requests tile kt+2 into the registers just
    // freed: the x half in K step 0, the weight half in K steps 1 and 2 (half of its loads each, which also spreads the
    // conversion of quantised weights), so every request has a whole tile's time to arrive and the requests of a CU
    // (64 KiB per tile through a 64 B/clock L1) are spread over the tile.
    // The barrier sits between K steps 2 and 3.  By then every wavefront has written its share of tile kt+1 and has
    // read all fragments of tile kt (those of step 3 are read during step 2), so during step 3 the fragments of the
    // first step of tile kt+1 are read and the matrix instructions run on across the end of the tile.  The buffer
    // written during tile kt is the one read during tile kt-1, whose last reads precede the barrier of kt-1.  The
    // barrier waits for LDS traffic only, so the requests stay in flight across it.
    commit(0);
    if (nk > 1) issue(1);
    lds_barrier();
    h8_t af[2][TM], bf[2][TN];
    frags(0, 0, af[0], bf[0]);
    for (int kt = 0; kt < nk; kt++) {
      const int cur = kt & 1;
      const int after_next = min(kt + 2, nk - 1);   // past the last tile the same steps run on the last tile again, into
                                                    // the buffer nobody computes from any more: a straight-line loop body
      __builtin_amdgcn_sched_barrier(0);
      auto k_step = [&](auto KK) {
        constexpr int kk = decltype(KK)::value;
        constexpr int LAST = STAGED_BK / 16 - 1;
        if (kk == LAST) lds_barrier();
        if (kk < LAST) frags(cur, kk + 1, af[(kk + 1) & 1], bf[(kk + 1) & 1]);
        else frags(cur ^ 1, 0, af[0], bf[0]);
        if (kk == 0) { commit_a(cur ^ 1); issue_a(after_next); }
        constexpr int HB = B_LOADS > 1 ? B_LOADS / 2 : 1;   // weight loads of K step 1; the rest in step 2
        if (kk == 1) { commit_b(cur ^ 1, 0, HB); issue_b(after_next, 0, HB); }
        if (kk == 2) { commit_b(cur ^ 1, HB, B_LOADS); issue_b(after_next, HB, B_LOADS); }
        mfmas(af[kk & 1], bf[kk & 1]);
        // The order inside this K step, spelled out for the instruction scheduler: every matrix instruction is followed by
        // a share of the other work of the step (fragment reads of the next step, conversion and LDS writes of the next
        // tile, then the requests of the tile after it), so that work runs while the matrix core is busy.  Left alone the
        // scheduler puts each fragment read directly before its first use and waits out the LDS latency every time.
        constexpr int NMF = TM * TN;
        constexpr int BL = kk == 1 ? HB : B_LOADS - HB;
        constexpr int LOADS = kk == 0 ? A_LOADS : BL;
        constexpr int WRITES = kk == 0 ? A_LOADS : (KIND == JSGRAD_W_I8 ? 2 * BL : 4 * BL);
        constexpr int WSTEPS = NMF - (LOADS < NMF / 2 ? LOADS : NMF / 2);     // matrix instructions that carry the writes
#pragma unroll
        for (int i = 0; i < NMF; i++) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                          // one MFMA
          if (i < TM + TN) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);          // one LDS read
          if (kk < LAST && LOADS > 0) {
            if (i < WSTEPS) {
              if (kk > 0) __builtin_amdgcn_sched_group_barrier(0x002, KIND == JSGRAD_W_I8 ? 6 : 10, 0);
              if constexpr (kk > 0 && KIND == JSGRAD_W_NF4) __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);   // table look-ups
              __builtin_amdgcn_sched_group_barrier(0x200, (WRITES + WSTEPS - 1) / WSTEPS, 0);
            } else {
              __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
              __builtin_amdgcn_sched_group_barrier(0x020, (LOADS + NMF - WSTEPS - 1) / (NMF - WSTEPS), 0);
            }
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      };
      static_assert(STAGED_BK / 16 == 4, "four K steps per tile");
      k_step(std::integral_constant<int, 0>{});
      k_step(std::integral_constant<int, 1>{});
      k_step(std::integral_constant<int, 2>{});
      k_step(std::integral_constant<int, 3>{});
    }
  } else {
    for (int kt = 0; kt < nk; kt++) {
      commit();
      __syncthreads();
      if (kt + 1 < nk) issue(kt + 1);
#pragma unroll
      for (int kk = 0; kk < STAGED_BK / 16; kk++) {
        h8_t af[TM], bf[TN];
        frags(0, kk, af, bf);
        mfmas(af, bf);
      }
      __syncthreads();
    }
  }

  // ---- epilogue.  The weight fragment is the first MFMA operand, so the 32x32 result tile is held transposed: a lane has
  // output row m = lane % 32 and, in accumulators 4g .. 4g+3, the four neighbouring output columns 8g + 4 * (lane / 32) + 0..3.
  // Stored from there, one instruction would touch 32 output rows with 8 bytes each.  Instead every wavefront turns 32 rows
  // x its CW columns at a time through its own piece of LDS (free after the K loop; rows padded by 8 bytes, which spreads
  // the 8-byte writes of 16 rows over all banks) and reads them back as 16-byte pieces along the rows: a store instruction
  // then covers whole cache lines, and so do the loads of the residual and of the rope table.
  constexpr int TNE = EPI == GEPI_SWIGLU ? TN / 2 : TN;   // 32-column tiles of output per wavefront and row tile
  constexpr int CW = TNE * 32, RS = CW + 4;               // columns per wavefront; halves per LDS row
  constexpr int CPR = CW / 8;                             // 16-byte pieces per row
  static_assert((size_t)4 * 32 * RS <= (size_t)(BM + BN) * LS, "the transposing pieces fit the K-loop buffer");
  _Float16 *ep = staged_lds + wave * 32 * RS;
  const int ncol0 = n0_out + wn * CW;                     // first output column of this wavefront
  // the residual of the whole wavefront tile is requested at once (the registers of the K loop are free): one trip to
  // memory instead of one per 32 rows
  h8_t res[EPI == GEPI_STORE ? TM : 1][EPI == GEPI_STORE ? 2 * TNE : 1];
  if constexpr (EPI == GEPI_STORE) {
    if (a.residual) {
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int p = 0; p < 2 * TNE; p++) {
          const int q = p * 64 + lane, row = q / CPR, piece = q % CPR;
          int m = m0 + (wm * TM + i) * 32 + row;
          if (m >= a.M) m = a.M - 1;
          res[i][p] = *(const h8_t *)&a.residual[(size_t)m * a.N + ncol0 + piece * 8];
        }
    }
  }
  __syncthreads();                                        // every wavefront is done with the K-loop buffers
#pragma unroll
  for (int i = 0; i < TM; i++) {
#pragma unroll
    for (int j = 0; j < TNE; j++) {
#pragma unroll
      for (int g = 0; g < 4; g++) {
        h4_t o;
#pragma unroll
        for (int c = 0; c < 4; c++) {
          if constexpr (EPI == GEPI_SWIGLU) {
            // silu(w1 x) * (w3 x), each GEMM output and the product stored as fp16 (llama.ts:108-110)
            const float gt = rn16(acc[i][j][4 * g + c]), up = rn16(acc[i][j + TN / 2][4 * g + c]);
            o[c] = (_Float16)(silu_act<_Float16>(gt) * up);
          } else {
            o[c] = (_Float16)acc[i][j][4 * g + c];
          }
        }
        *(h4_t *)&ep[l32 * RS + j * 32 + 8 * g + 4 * lg] = o;
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the wavefront's own writes, before its own reads
    const int mrow0 = m0 + (wm * TM + i) * 32;
#pragma unroll
    for (int p = 0; p < 2 * TNE; p++) {
      const int q = p * 64 + lane, row = q / CPR, piece = q % CPR;
      const int m = mrow0 + row, n = ncol0 + piece * 8;
      const h8_t v = *(const h8_t *)&ep[row * RS + piece * 8];
      if (m >= a.M) continue;
      if constexpr (EPI == GEPI_SWIGLU) {
        *(h8_t *)&a.y[(size_t)m * a.N + n] = v;
      } else if constexpr (EPI == GEPI_STORE) {
        h8_t o = v;
        if (a.residual) {
#pragma unroll
          for (int c = 0; c < 8; c++) o[c] = (_Float16)((float)res[i][p][c] + (float)v[c]);
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
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the reads, before the next row tile overwrites the piece
  }
}

template <int KIND, int EPI, int WGM, int WGN, int TM, int TN, bool DB = false> static int launch_staged(const GemmArgs &a, int prof_kind) {
  constexpr int BM = WGM * TM * 32, BN = WGN * TN * 32;
  const int tiles = ((a.M + BM - 1) / BM) * (a.N / (EPI == GEPI_SWIGLU ? BN / 2 : BN));
  constexpr size_t lds = (size_t)(DB ? 2 : 1) * (BM + BN) * STAGED_STRIDE * sizeof(_Float16) + 32 + (KIND == JSGRAD_W_NF4 ? 1024 : 0);
  static_assert(lds <= 160 * 1024, "LDS of one compute unit");
  if constexpr (lds > 64 * 1024) {
    static bool raised = false;   // one process, one device, one thread: set once per instantiation
    if (!raised) {
      JSG_HIP(hipFuncSetAttribute((const void *)staged_kernel<KIND, EPI, WGM, WGN, TM, TN, DB>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
      raised = true;
    }
  }
  JSG_LAUNCH(prof_kind, (staged_kernel<KIND, EPI, WGM, WGN, TM, TN, DB>), dim3(tiles), dim3(STAGED_THREADS), lds, a);
  return 0;
}
template <int KIND, int EPI> static int gemm_staged_as(int bm, int bn, const GemmArgs &a, int prof_kind) {
  if (bn == 256) return launch_staged<KIND, EPI, 2, 2, 4, 4, true>(a, prof_kind);
  if (bm == 256) return launch_staged<KIND, EPI, 2, 2, 4, 2>(a, prof_kind);
  if constexpr (EPI != GEPI_SWIGLU)
    if (bm == 32) return launch_staged<KIND, EPI, 1, 4, 1, 1>(a, prof_kind);
  return launch_staged<KIND, EPI, 2, 2, 2, 2>(a, prof_kind);
}
template <int KIND> static int gemm_staged_kind(int epi, int bm, int bn, const GemmArgs &a, int prof_kind) {
  if (epi == GEPI_STORE) return gemm_staged_as<KIND, GEPI_STORE>(bm, bn, a, prof_kind);
  if (epi == GEPI_ROPE_KV) return gemm_staged_as<KIND, GEPI_ROPE_KV>(bm, bn, a, prof_kind);
  return gemm_staged_as<KIND, GEPI_SWIGLU>(bm, bn, a, prof_kind);
}
int gemm_staged(int epi, int kind, int bm, int bn, const GemmArgs &a, int prof_kind) {
  return kind == JSGRAD_W_I8 ? gemm_staged_kind<JSGRAD_W_I8>(epi, bm, bn, a, prof_kind) : gemm_staged_kind<JSGRAD_W_NF4>(epi, bm, bn, a, prof_kind);
}

}  // namespace jsg
