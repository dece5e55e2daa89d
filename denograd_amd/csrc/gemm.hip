// Several-row linear layers, few rows: y[M][N] = x[M][K] . W[N][K]^T for 1 to 32 rows of fp16 activations (batched decode), fp32
// accumulate, fp16 out, and the entry points for any number of rows (more rows: gemm_tile.hip and gemm_staged.hip; wide or long matrices with up to
// 32 rows: gemm_group.hip; fp16 and short int8 matrices with
// at most 16 rows: gemm_few.hip).
//
// What the reference computes (/root/reference/jsgrad/tensor.ts:2593-2605 `dot`, :3800 `linear`; Int8Linear.call
// /root/reference/jsgrad/models/llama3.ts:35; NF4Linear.call :91-97): with more than one input row the weight operand is
// expanded over the rows, so a quantised weight is first realised in fp16, W = RN16(code * scale), and the products of
// two fp16 values are then summed in float.  v_pk_mul_f16 of the exact fp16 code by the fp16 scale is that single rounding.
#include <type_traits>

#include "gemm.h"

namespace jsg {

// ---- at most 32 rows (batched decode): the weights are streamed once, straight from memory into the B operand ------------
//
// With a handful of rows the launch is bound by reading W once, so it is laid out like the one-row GEMV, not like a tiled
// GEMM.  v_mfma_f32_16x16x32_f16 takes, per lane, 8 consecutive K elements of one weight row as B and of one x row as
// A; a lane's 16-byte load is 8 fp16, 16 int8 codes or 32 nf4 codes of weight row n0 + lane % 16, i.e. one, two or four
// MFMAs, and goes from memory to registers with nothing in between (int8 and nf4 codes become RN16(code * scale) in
// registers: the realised fp16 matrix the reference multiplies by; nf4 through a 256-entry table of code pairs in LDS, one
// look-up per byte, with the scale of the lane's 64-element block loaded beside the codes).  The loads run through a register ring of 12 to 16 loads per wavefront.
// Only x goes through LDS, in K chunks of 512, four buffers.  The fifth wavefront of a block does nothing but move
// x chunks from memory to LDS (direct loads, no registers), up to three chunks ahead: a wavefront's loads return in order, so x loads issued by
// the arithmetic wavefronts would have to be waited for together with every weight load issued before them, which
// empties the ring once per chunk.
//
// A block owns 16 weight rows and its four arithmetic wavefronts split K: each takes a quarter of the k-blocks of every
// chunk, and the partial accumulators are added in wavefront order through LDS.  N/16 blocks fill the chip even for
// N = 4096.  (A block shape with 128 weight rows, which reads x once for all of them instead of once per 16, was tried for
// the wide layers: faster for the lm_head only, and its register ring did not survive the register allocator.)
template <int KIND> struct SkFmt {
  static constexpr int VEC = KIND == JSGRAD_W_F16 ? 8 : (KIND == JSGRAD_W_I8 ? 16 : 32);   // K elements per 16-byte load of a lane
  static constexpr int KB = 4 * VEC;                          // K elements per wavefront load (a k-block)
  static constexpr int KC = 512;                              // K elements per x chunk: 1 KiB per x row, one direct load
  static constexpr int KBC = KC / KB;                         // k-blocks per chunk
};
constexpr int SK_THREADS = 320;
constexpr int SK_KS = 4;                                      // wavefronts that split K
constexpr int SK_XBUF = 4;                                    // x chunks in LDS: one being read, up to three on their way
template <int KIND, int EPI, int RTW> struct SkShape {
  static constexpr int NMAT = EPI == GEPI_SWIGLU ? 2 : 1;
  static constexpr int SPC = SkFmt<KIND>::KBC / SK_KS;        // k-blocks of a chunk one wavefront walks
  static constexpr int RS = 8;                                // k-blocks in the ring
  static constexpr int BR = 16 * RTW;                         // weight rows per block: RTW tiles of 16
  static_assert(RS % SPC == 0, "chunk ends fall on fixed ring slots");
};

// Block barriers of the weight-streaming kernel.  __syncthreads() also waits for every global load of the wavefront (the
// counter that tracks loads tracks stores too, and a barrier publishes stores), which would empty the ring of weight loads
// at every x chunk; what has to be finished at these barriers is only LDS traffic, or, for the wavefront that moves x,
// its direct loads into LDS.
__device__ __forceinline__ void sk_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <int KIND, int EPI, int MB, int RTW>
__global__ __launch_bounds__(SK_THREADS, 2) void skinny_gemm_kernel(GemmArgs a) {
  static_assert(KIND == JSGRAD_W_F16 || KIND == JSGRAD_W_I8 || KIND == JSGRAD_W_NF4, "fp16, int8 and nf4 weights");
  typedef SkFmt<KIND> F;
  typedef SkShape<KIND, EPI, RTW> S;
  constexpr int NMAT = S::NMAT, SPC = S::SPC, RS = S::RS;
  constexpr int NMF = F::VEC / 8;                        // MFMAs per load
  constexpr int LS = F::KC + 8;                          // halves per LDS row of x (padded: rows start in different banks)
  constexpr int XROWS = MB * 16;
  constexpr int PPR = F::KC / 8;                         // 16-byte pieces per x row of a chunk
  static_assert(PPR % 64 == 0, "a direct load of the wavefront fills 1 KiB of one LDS row");
  constexpr int XLOADS = XROWS * PPR / 64;               // direct loads per chunk
  extern __shared__ __align__(16) _Float16 sk_lds[];     // SK_XBUF x [XROWS][LS]; afterwards the partial accumulators

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, lq = lane >> 4;
  const int nchunks = a.K / F::KC;
  // NF4: one table entry per BYTE, the code values of its two nibbles as a packed pair (element 2j, the high nibble, in the
  // low half: llama3.ts:92-94); written here, read after the first barrier of either path below
  __shared__ uint32_t pairs[KIND == JSGRAD_W_NF4 ? 256 : 1];
  if constexpr (KIND == JSGRAD_W_NF4) {
    if (tid < 256) pairs[tid] = nf4_code_bits(tid >> 4) | (nf4_code_bits(tid & 15) << 16);
  }

  if (wave == 4) {
    // ---- the x mover: up to three chunks ahead of the one being read (a chunk takes a trip to L2 to arrive, longer than
    // the others need for a chunk), into the buffer whose readers passed the barrier of the chunk before
    auto move = [&](int c) {
      _Float16 *dst = sk_lds + (c % SK_XBUF) * XROWS * LS;
#pragma unroll
      for (int i = 0; i < XLOADS; i++) {
        const int r = (i * 64) / PPR, c8 = (i * 64) % PPR + lane;
        const int m = r < a.M ? r : a.M - 1;             // rows past the end are computed and never stored
        const _Float16 *src = a.x + (size_t)m * a.K + (size_t)c * F::KC + c8 * 8;
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src,
                                         (__attribute__((address_space(3))) void *)(dst + r * LS + ((i * 64) % PPR) * 8), 16, 0, 0);
      }
    };
    // wait until chunk `target` has landed: the direct loads complete in order, so whatever was issued after it may stay
    // in flight (the counter holds 63 loads at most)
    constexpr int MAX_BEHIND = 63 / XLOADS < 2 ? 63 / XLOADS : 2;
    int issued = 0;
    auto landed = [&](int target) {
      const int behind = issued - target - 1;
      if (MAX_BEHIND >= 2 && behind >= 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * XLOADS <= 63 ? 2 * XLOADS : 0) : "memory");
      else if (MAX_BEHIND >= 1 && behind >= 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(XLOADS <= 63 ? XLOADS : 0) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    };
    while (issued < SK_XBUF - 1 && issued < nchunks) move(issued++);
    landed(0);
    sk_barrier();
    for (int c = 0; c < nchunks; c++) {
      if (issued < nchunks) move(issued++);              // into the buffer of chunk c - 1
      if (c + 1 < nchunks) landed(c + 1);
      sk_barrier();
    }
    sk_barrier();
    return;
  }

  const int ks = wave;
  const int n_first = blockIdx.x * S::BR;               // first weight row of the block
  // ---- the weight rows of this lane: row n_first + rt * 16 + lane % 16 of matrix q
  const unsigned char *wrow[RTW][NMAT];
  h2_t wscale[RTW][NMAT];
  const _Float16 *srow[RTW][NMAT];
#pragma unroll
  for (int rt = 0; rt < RTW; rt++)
#pragma unroll
    for (int q = 0; q < NMAT; q++) {
      const int n = n_first + rt * 16 + l16;
      const void *w; const _Float16 *sc; int row;
      if constexpr (EPI == GEPI_SWIGLU) { w = q ? a.w1 : a.w0; sc = q ? a.s1 : a.s0; row = n; }
      else if constexpr (EPI == GEPI_ROPE_KV) {
        if (n < a.n0) { w = a.w0; sc = a.s0; row = n; }
        else if (n < a.n0 + a.n1) { w = a.w1; sc = a.s1; row = n - a.n0; }
        else { w = a.w2; sc = a.s2; row = n - a.n0 - a.n1; }
      } else { w = a.w0; sc = a.s0; row = n; }
      const size_t e = (size_t)row * a.K;
      wrow[rt][q] = (const unsigned char *)w + (KIND == JSGRAD_W_F16 ? e * 2 : (KIND == JSGRAD_W_I8 ? e : e / 2)) + lq * 16;
      if constexpr (KIND == JSGRAD_W_I8) { const _Float16 sv = sc[row]; wscale[rt][q] = h2_t{sv, sv}; }
      // nf4: a scale per 64 elements of the flattened matrix; a lane's 32 elements of a k-block share one (two per k-block)
      if constexpr (KIND == JSGRAD_W_NF4) srow[rt][q] = sc + (e >> 6) + (lq >> 1);
    }
  // Step s of this wavefront is k-block ks * SPC + s % SPC of chunk s / SPC: its SPC k-blocks of a chunk are neighbours, so
  // that the halves of a 128-byte line of a weight row are asked for by one wavefront, back to back.  Byte offset of the
  // step inside a weight row.  Past the end the last k-block is asked for again: the refills of the last RS steps keep the
  // number of loads in flight the same on every path, and a line that was fetched a moment ago costs no HBM traffic (the
  // first k-block of the row, read at the start, has long left the caches by then: that was 1.2-1.5x the bytes).
  const int nsteps = nchunks * SPC;
  auto woff = [&](int s) -> uint32_t {
    const int sc = s < nsteps ? s : nsteps - 1;
    const int kb = (sc / SPC) * F::KBC + ks * SPC + sc % SPC;
    return (uint32_t)(kb * 4) * 16u;
  };

  u4_t ring[RS][RTW][NMAT];
  _Float16 rsc[KIND == JSGRAD_W_NF4 ? RS : 1][RTW][NMAT];   // nf4: the block scale travels with its load
  f4_t acc[NMAT][RTW][MB];
#pragma unroll
  for (int q = 0; q < NMAT; q++)
#pragma unroll
    for (int rt = 0; rt < RTW; rt++)
#pragma unroll
      for (int mb = 0; mb < MB; mb++) acc[q][rt][mb] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int i = 0; i < RS; i++)
#pragma unroll
    for (int rt = 0; rt < RTW; rt++)
#pragma unroll
      for (int q = 0; q < NMAT; q++) {
        ring[i][rt][q] = ldg_stream16(wrow[rt][q] + woff(i));
        if constexpr (KIND == JSGRAD_W_NF4) rsc[i][rt][q] = ldg(srow[rt][q] + (woff(i) >> 5));   // 64 bytes of codes per k-block = two scales
        __builtin_amdgcn_sched_barrier(0);               // issued in the order the loop consumes them: the waits count on it
      }
  sk_barrier();                                          // x chunk 0 is in LDS

  // The ring slots are refilled on every path, also by the steps past the end (the number of loads in flight then is the
  // same wherever the wait counters are set, so they can let RS - 1 steps stay in flight instead of none).
  for (int s0 = 0; s0 < nsteps; s0 += RS) {
#pragma unroll
    for (int i = 0; i < RS; i++) {
      const int s = s0 + i;
      const bool on = s < nsteps;                        // same for every thread of the block
      const int c = s / SPC, kb = ks * SPC + s % SPC;
      const _Float16 *xs = sk_lds + (c % SK_XBUF) * XROWS * LS;
      if (on) {
        h8_t af[NMF][MB];
#pragma unroll
        for (int f = 0; f < NMF; f++)
#pragma unroll
          for (int mb = 0; mb < MB; mb++) af[f][mb] = *(const h8_t *)&xs[(mb * 16 + l16) * LS + kb * F::KB + lq * F::VEC + f * 8];
#pragma unroll
        for (int rt = 0; rt < RTW; rt++)
#pragma unroll
          for (int q = 0; q < NMAT; q++) {
            const u4_t raw = ring[i][rt][q];
            h8_t bf[NMF];
            if constexpr (KIND == JSGRAD_W_F16) bf[0] = __builtin_bit_cast(h8_t, raw);
            else if constexpr (KIND == JSGRAD_W_NF4) {
              const _Float16 s1 = rsc[i][rt][q];
              const h2_t sv = {s1, s1};
              const uint32_t wds[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
              for (int d = 0; d < 4; d++) {                // a dword = 8 elements = one matrix instruction
                u4_t o;
                o.x = pk_mul_h2(pairs[wds[d] & 0xffu], sv);
                o.y = pk_mul_h2(pairs[(wds[d] >> 8) & 0xffu], sv);
                o.z = pk_mul_h2(pairs[(wds[d] >> 16) & 0xffu], sv);
                o.w = pk_mul_h2(pairs[wds[d] >> 24], sv);
                bf[d] = __builtin_bit_cast(h8_t, o);
              }
            } else {
              const h2_t sc = wscale[rt][q];
              u4_t o0, o1;
              uint32_t lo, hi;
              i8x4_to_h2x2(raw.x, lo, hi); o0.x = pk_mul_h2(lo, sc); o0.y = pk_mul_h2(hi, sc);
              i8x4_to_h2x2(raw.y, lo, hi); o0.z = pk_mul_h2(lo, sc); o0.w = pk_mul_h2(hi, sc);
              i8x4_to_h2x2(raw.z, lo, hi); o1.x = pk_mul_h2(lo, sc); o1.y = pk_mul_h2(hi, sc);
              i8x4_to_h2x2(raw.w, lo, hi); o1.z = pk_mul_h2(lo, sc); o1.w = pk_mul_h2(hi, sc);
              bf[0] = __builtin_bit_cast(h8_t, o0);
              bf[NMF - 1] = __builtin_bit_cast(h8_t, o1);
            }
#pragma unroll
            for (int f = 0; f < NMF; f++)
#pragma unroll
              for (int mb = 0; mb < MB; mb++) acc[q][rt][mb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[f][mb], bf[f], acc[q][rt][mb], 0, 0, 0);
          }
      }
      // The slots are refilled only now that their old contents are used up (and the scheduler may not move the loads up):
      // issued earlier, a load gets registers of its own and a copy into the slot afterwards, and the copy waits for the
      // load on the spot.
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int rt = 0; rt < RTW; rt++)
#pragma unroll
        for (int q = 0; q < NMAT; q++) {
          ring[i][rt][q] = ldg_stream16(wrow[rt][q] + woff(s + RS));
          if constexpr (KIND == JSGRAD_W_NF4) rsc[i][rt][q] = ldg(srow[rt][q] + (woff(s + RS) >> 5));
        }
      if (on && (s + 1) % SPC == 0) sk_barrier();        // chunk c is consumed, chunk c + 1 is in the other buffer
    }
  }

  // ---- epilogue of one 16x16 tile.  Accumulator r of a lane is output row 4 * (lane / 16) + r, column lane % 16.
  auto epilogue = [&](const f4_t (&tot)[NMAT], int n_tile, int mb) {
    const int n = n_tile + l16;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int m = mb * 16 + lq * 4 + r;
      if constexpr (EPI == GEPI_SWIGLU) {
        const float g = rn16(tot[0][r]), u = rn16(tot[NMAT - 1][r]);
        if (m < a.M) a.y[(size_t)m * a.N + n] = (_Float16)(silu_act<_Float16>(g) * u);
      } else if constexpr (EPI == GEPI_STORE) {
        if (m < a.M) {
          float v = rn16(tot[0][r]);
          if (a.residual) v = (float)a.residual[(size_t)m * a.N + n] + v;
          a.y[(size_t)m * a.N + n] = (_Float16)v;
        }
      } else {
        const int which = n < a.n0 ? 0 : (n < a.n0 + a.n1 ? 1 : 2);
        const int nl = which == 0 ? n : (which == 1 ? n - a.n0 : n - a.n0 - a.n1);
        const int pair = (nl % a.head_dim) >> 1;
        const bool odd = nl & 1;
        const float own = rn16(tot[0][r]);
        const float other = dpp_f<0xB1>(own);            // the neighbouring column: the other half of the pair
        if (m < a.M) {
          const int b = m / a.seq_len, pos = a.start_pos + m % a.seq_len;
          float v = own;
          if (which < 2) {
            const h2_t cs = *(const h2_t *)(a.rope_table + ((size_t)pos * (a.head_dim / 2) + pair) * 2);
            const float cc = (float)cs.x, dd = (float)cs.y;
            v = odd ? other * dd + own * cc : own * cc - other * dd;
          }
          if (which == 0) a.y[(size_t)m * a.n0 + nl] = (_Float16)v;
          else {
            _Float16 *cache = which == 1 ? a.cache_k : a.cache_v;
            cache[((size_t)b * a.max_context + pos) * a.n1 + nl] = (_Float16)v;
          }
        }
      }
    }
  };

  // the four K parts, added in wavefront order; the (tile, row block) pairs are dealt to the wavefronts
  constexpr int NACC = NMAT * RTW * MB;
  float *red = (float *)sk_lds;                          // [4][NACC][64 lanes] x 4 floats
#pragma unroll
  for (int q = 0; q < NMAT; q++)
#pragma unroll
    for (int rt = 0; rt < RTW; rt++)
#pragma unroll
      for (int mb = 0; mb < MB; mb++) *(f4_t *)&red[((wave * NACC + (q * RTW + rt) * MB + mb) * 64 + lane) * 4] = acc[q][rt][mb];
  sk_barrier();
  for (int item = wave; item < RTW * MB; item += 4) {
    const int rt = item / MB, mb = item % MB;
    f4_t tot[NMAT];
#pragma unroll
    for (int q = 0; q < NMAT; q++) {
      tot[q] = *(const f4_t *)&red[((0 * NACC + (q * RTW + rt) * MB + mb) * 64 + lane) * 4];
#pragma unroll
      for (int w = 1; w < 4; w++) tot[q] += *(const f4_t *)&red[((w * NACC + (q * RTW + rt) * MB + mb) * 64 + lane) * 4];
    }
    epilogue(tot, n_first + rt * 16, mb);
  }
}

// ---- host side ---------------------------------------------------------------------------------------------------

template <int KIND, int EPI, int MB, int RTW> static int launch_skinny(const GemmArgs &a, int prof_kind) {
  typedef SkFmt<KIND> F;
  typedef SkShape<KIND, EPI, RTW> S;
  constexpr size_t x_bytes = (size_t)SK_XBUF * MB * 16 * (F::KC + 8) * sizeof(_Float16);
  constexpr size_t red_bytes = (size_t)4 * S::NMAT * RTW * MB * 64 * 4 * sizeof(float);
  constexpr size_t lds = x_bytes > red_bytes ? x_bytes : red_bytes;
  if constexpr (lds > 64 * 1024) {
    static bool raised = false;   // one process, one device, one thread: set once per instantiation
    if (!raised) {
      JSG_HIP(hipFuncSetAttribute((const void *)skinny_gemm_kernel<KIND, EPI, MB, RTW>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
      raised = true;
    }
  }
  JSG_LAUNCH(prof_kind, (skinny_gemm_kernel<KIND, EPI, MB, RTW>), dim3(a.N / S::BR), dim3(SK_THREADS), lds, a);
  return 0;
}
// Few rows: the weight-streaming kernel when K is whole chunks.  Every block reads all of x; with two tiles of 16 weight
// rows per block that is half as often.  Measured on the lm_head (8016 tiles) the two-tile shape is no faster and moves
// more HBM bytes (1.5x the weights against 1.24x), so it is only taken when pinned.
template <int KIND, int EPI> static int dispatch_skinny(const GemmArgs &a, int prof_kind, bool *taken) {
  *taken = a.M <= 32 && a.K % SkFmt<KIND>::KC == 0 && a.K / SkFmt<KIND>::KC >= 2 && a.N % 16 == 0 && !pin_env(a, "JSG_GEMM_NO_SKINNY");
  if (!*taken) return 0;
  const char *pin = pin_env(a, "JSG_GEMM_SKINNY_TILES");     // "1" or "2": tests run small matrices through both
  const bool two = a.N % 32 == 0 && pin && pin[0] == '2';
  if (a.M <= 16) return two ? launch_skinny<KIND, EPI, 1, 2>(a, prof_kind) : launch_skinny<KIND, EPI, 1, 1>(a, prof_kind);
  return two ? launch_skinny<KIND, EPI, 2, 2>(a, prof_kind) : launch_skinny<KIND, EPI, 2, 1>(a, prof_kind);
}

// x normed into xn, which is what the product reads then
static int norm_first(GemmArgs &a, _Float16 *xn) {
  if (const int rc = jsgrad_hip_rmsnorm_rows(a.x, a.norm_w, xn, a.M, a.K, a.eps)) return rc;
  a.x = xn;
  a.norm_w = nullptr;
  return 0;
}
template <int EPI> static int dispatch_gemm(int kind, GemmArgs a, int prof_kind, _Float16 *xn = nullptr) {
  bool taken = false;
  const char *const pin = pin_env(a, "JSG_GEMM_TILE");
  const bool group = pin && *pin == 'g';                      // tests
  int rc = group ? 0 : gemm_few(EPI, kind, a, prof_kind, &taken);
  if (taken || rc) return rc;
  if (a.norm_w) {
    if ((rc = norm_first(a, xn))) return rc;
    // what cannot norm such an input on its way may still be the kernel for it normed (us, norm and product, this | the kernels below: fp16
    // 8 x 4096 x 8192 17.6 | 19.8, 1 x 2048 x 6144 9.9 | 12.7; int8 3 x 4096 x 6144 11.1 | 13.2)
    rc = group ? 0 : gemm_few(EPI, kind, a, prof_kind, &taken);
    if (taken || rc) return rc;
  }
  rc = gemm_group(EPI, kind, a, prof_kind, &taken);
  if (taken || rc) return rc;
  if (kind == JSGRAD_W_F16) { rc = dispatch_skinny<JSGRAD_W_F16, EPI>(a, prof_kind, &taken); if (taken) return rc; }
  if (kind == JSGRAD_W_I8) { rc = dispatch_skinny<JSGRAD_W_I8, EPI>(a, prof_kind, &taken); if (taken) return rc; }
  if (kind == JSGRAD_W_NF4) { rc = dispatch_skinny<JSGRAD_W_NF4, EPI>(a, prof_kind, &taken); if (taken) return rc; }
  return gemm_tiled(EPI, kind, a, prof_kind);
}

// largest column tile any configuration uses: output widths must be multiples of it
constexpr int GEMM_N_ALIGN = 128;
constexpr int GEMM_K_ALIGN = 64;   // a K tile

static bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

static int check_gemm(const char *who, int kind, int rows, int in_f) {
  JSG_REQUIRE(kind == JSGRAD_W_F16 || kind == JSGRAD_W_I8 || kind == JSGRAD_W_NF4, "%s: weight kind %d is not built for several rows (fp16, int8 and nf4 are)", who, kind);
  JSG_REQUIRE(rows > 0, "%s: %d rows", who, rows);
  JSG_REQUIRE(in_f > 0 && in_f % GEMM_K_ALIGN == 0, "%s: in_features %d must be a positive multiple of %d", who, in_f, GEMM_K_ALIGN);
  return 0;
}

// An input that is normed first: its norm's weights, and rows of memory for the result where no kernel norms x on its way
struct NormFirst { const void *weight; float eps; void *xn; };
static int set_norm(const char *who, const NormFirst *norm, GemmArgs &a) {
  if (!norm) return 0;
  JSG_REQUIRE(norm->weight && norm->xn, "%s: null pointer argument", who);
  JSG_REQUIRE(aligned16(norm->xn), "%s: xn must be 16-byte aligned", who);   // the weight may lie anywhere, as in jsgrad_hip_rmsnorm_rows
  a.norm_w = (const _Float16 *)norm->weight;
  a.eps = norm->eps;
  a.inv_k = (float)(1.0 / (double)a.K);
  return 0;
}

static int plain_gemm(const char *who, const NormFirst *norm, int kind, const void *w, const void *scale, int out_f, int in_f, const void *x, int rows,
                      void *y, const void *residual) {
  if (int rc = check_gemm(who, kind, rows, in_f)) return rc;
  JSG_REQUIRE(w && x && y, "%s: null pointer argument", who);
  JSG_REQUIRE(kind == JSGRAD_W_F16 || scale, "%s: quantised weights need their scales", who);
  JSG_REQUIRE(out_f > 0 && out_f % GEMM_N_ALIGN == 0, "%s: out_features %d must be a positive multiple of %d", who, out_f, GEMM_N_ALIGN);
  JSG_REQUIRE(aligned16(w) && aligned16(x) && aligned16(y) && aligned16(residual), "%s: w, x, y and residual must be 16-byte aligned", who);
  GemmArgs a = {};
  a.pins = any_pins();
  a.w0 = w; a.s0 = (const _Float16 *)scale; a.n0 = out_f;
  a.M = rows; a.N = out_f; a.K = in_f;
  a.x = (const _Float16 *)x; a.y = (_Float16 *)y; a.residual = (const _Float16 *)residual;
  if (int rc = set_norm(who, norm, a)) return rc;
  return dispatch_gemm<GEPI_STORE>(kind, a, PROF_GEMM, norm ? (_Float16 *)norm->xn : nullptr);
}

static int qkv_rope_gemm(const char *who, const NormFirst *norm, int kind, const void *wq, const void *sq, const void *wk, const void *sk, const void *wv, const void *sv,
                         const void *x, int rows, int seq_len, int start_pos, const void *rope_table, void *q_out, void *cache_k, void *cache_v, int dim,
                         int n_heads, int n_kv_heads, int head_dim, int max_context) {
  if (int rc = check_gemm(who, kind, rows, dim)) return rc;
  JSG_REQUIRE(wq && wk && wv && x && rope_table && q_out && cache_k && cache_v, "%s: null pointer argument", who);
  JSG_REQUIRE(kind == JSGRAD_W_F16 || (sq && sk && sv), "%s: quantised weights need their scales", who);
  JSG_REQUIRE(head_dim > 0 && head_dim % 8 == 0 && n_heads > 0 && n_kv_heads > 0, "%s: bad head geometry (head_dim a multiple of 8)", who);
  JSG_REQUIRE(aligned16(wq) && aligned16(wk) && aligned16(wv) && aligned16(x) && aligned16(rope_table) && aligned16(q_out) && aligned16(cache_k) && aligned16(cache_v),
              "%s: weights, x, rope_table, q_out and the caches must be 16-byte aligned", who);
  const int nq = n_heads * head_dim, nkv = n_kv_heads * head_dim;
  JSG_REQUIRE(nq % GEMM_N_ALIGN == 0 && nkv % GEMM_N_ALIGN == 0, "%s: n_heads*head_dim %d and n_kv_heads*head_dim %d must be multiples of %d", who, nq, nkv,
              GEMM_N_ALIGN);
  JSG_REQUIRE(seq_len > 0 && rows % seq_len == 0, "%s: %d rows are not whole sequences of %d", who, rows, seq_len);
  JSG_REQUIRE(start_pos >= 0 && start_pos + seq_len <= max_context, "%s: positions [%d, %d) outside the cache of %d", who, start_pos,
              start_pos + seq_len, max_context);
  GemmArgs a = {};
  a.pins = any_pins();
  a.w0 = wq; a.w1 = wk; a.w2 = wv;
  a.s0 = (const _Float16 *)sq; a.s1 = (const _Float16 *)sk; a.s2 = (const _Float16 *)sv;
  a.n0 = nq; a.n1 = nkv; a.n2 = nkv;
  a.M = rows; a.N = nq + 2 * nkv; a.K = dim;
  a.x = (const _Float16 *)x; a.y = (_Float16 *)q_out;
  a.rope_table = (const _Float16 *)rope_table; a.cache_k = (_Float16 *)cache_k; a.cache_v = (_Float16 *)cache_v;
  a.seq_len = seq_len; a.start_pos = start_pos; a.head_dim = head_dim; a.max_context = max_context;
  if (int rc = set_norm(who, norm, a)) return rc;
  return dispatch_gemm<GEPI_ROPE_KV>(kind, a, PROF_GEMM, norm ? (_Float16 *)norm->xn : nullptr);
}

static int ffn_gate_gemm(const char *who, const NormFirst *norm, int kind, const void *w1, const void *s1, const void *w3, const void *s3,
                         const void *x, int rows, void *y, int dim, int hidden) {
  if (int rc = check_gemm(who, kind, rows, dim)) return rc;
  JSG_REQUIRE(w1 && w3 && x && y, "%s: null pointer argument", who);
  JSG_REQUIRE(kind == JSGRAD_W_F16 || (s1 && s3), "%s: quantised weights need their scales", who);
  JSG_REQUIRE(hidden > 0 && hidden % GEMM_N_ALIGN == 0, "%s: hidden_dim %d must be a positive multiple of %d", who, hidden, GEMM_N_ALIGN);
  JSG_REQUIRE(aligned16(w1) && aligned16(w3) && aligned16(x) && aligned16(y), "%s: w1, w3, x and g must be 16-byte aligned", who);
  GemmArgs a = {};
  a.pins = any_pins();
  a.w0 = w1; a.w1 = w3; a.s0 = (const _Float16 *)s1; a.s1 = (const _Float16 *)s3;
  a.n0 = hidden; a.n1 = hidden;
  a.M = rows; a.N = hidden; a.K = dim;
  a.x = (const _Float16 *)x; a.y = (_Float16 *)y;
  if (int rc = set_norm(who, norm, a)) return rc;
  return dispatch_gemm<GEPI_SWIGLU>(kind, a, PROF_GEMM, norm ? (_Float16 *)norm->xn : nullptr);
}

}  // namespace jsg

using namespace jsg;

extern "C" {

int jsgrad_hip_gemm(int kind, const void *w, const void *scale, int out_f, int in_f, const void *x, int rows, void *y, const void *residual) {
  JSG_READY();
  return plain_gemm("jsgrad_hip_gemm", nullptr, kind, w, scale, out_f, in_f, x, rows, y, residual);
}
int jsgrad_hip_gemm_norm(int kind, const void *w, const void *scale, int out_f, int in_f, const void *x, const void *norm_weight, float eps, void *xn,
                         int rows, void *y) {
  JSG_READY();
  const NormFirst norm = {norm_weight, eps, xn};
  return plain_gemm("jsgrad_hip_gemm_norm", &norm, kind, w, scale, out_f, in_f, x, rows, y, nullptr);
}

int jsgrad_hip_gemm_qkv_rope(int kind, const void *wq, const void *sq, const void *wk, const void *sk, const void *wv, const void *sv, const void *x,
                             int rows, int seq_len, int start_pos, const void *rope_table, void *q_out, void *cache_k, void *cache_v, int dim,
                             int n_heads, int n_kv_heads, int head_dim, int max_context) {
  JSG_READY();
  return qkv_rope_gemm("jsgrad_hip_gemm_qkv_rope", nullptr, kind, wq, sq, wk, sk, wv, sv, x, rows,
                       seq_len, start_pos, rope_table, q_out, cache_k, cache_v, dim, n_heads, n_kv_heads, head_dim, max_context);
}
int jsgrad_hip_gemm_qkv_rope_norm(int kind, const void *wq, const void *sq, const void *wk, const void *sk, const void *wv, const void *sv,
                                  const void *x, const void *norm_weight, float eps, void *xn, int rows, int seq_len, int start_pos,
                                  const void *rope_table, void *q_out, void *cache_k, void *cache_v, int dim, int n_heads, int n_kv_heads,
                                  int head_dim, int max_context) {
  JSG_READY();
  const NormFirst norm = {norm_weight, eps, xn};
  return qkv_rope_gemm("jsgrad_hip_gemm_qkv_rope_norm", &norm, kind, wq, sq, wk, sk, wv, sv, x, rows,
                       seq_len, start_pos, rope_table, q_out, cache_k, cache_v, dim, n_heads, n_kv_heads, head_dim, max_context);
}

int jsgrad_hip_gemm_ffn_gate(int kind, const void *w1, const void *s1, const void *w3, const void *s3, const void *x, int rows, void *y, int dim,
                             int hidden) {
  JSG_READY();
  return ffn_gate_gemm("jsgrad_hip_gemm_ffn_gate", nullptr, kind, w1, s1, w3, s3, x, rows, y, dim, hidden);
}
int jsgrad_hip_gemm_ffn_gate_norm(int kind, const void *w1, const void *s1, const void *w3, const void *s3, const void *x, const void *norm_weight,
                                  float eps, void *xn, int rows, void *y, int dim, int hidden) {
  JSG_READY();
  const NormFirst norm = {norm_weight, eps, xn};
  return ffn_gate_gemm("jsgrad_hip_gemm_ffn_gate_norm", &norm, kind, w1, s1, w3, s3, x, rows, y, dim, hidden);
}

}  // extern "C"
