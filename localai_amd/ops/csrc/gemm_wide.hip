// Quantised GEMM of 65 to some hundred rows (decode batches, short prompts):
//   out[s][m][n] = sum_{k in split s} X[m,k] * W[n,k]   (fp32 slabs, or bf16 [M][N] at one split)
//   h[m][j]      = act(x Wg[j]^T) * (x Wu[j]^T)          (bf16)
//
// Shape of the work (MI355X):
//  * Workgroup = 8 waves, two per SIMD, over BM = 64 RB rows x 128 columns.  Waves 0-3 and 4-7 are two K groups: of
//    every step of 64 k the first takes 32 and the second the other 32; a group's waves are 2 (rows) x 2 (columns), so
//    a wave holds 32 RB rows x 64 columns (v_mfma_f32_32x32x16_bf16).  That is the tile whose LDS reads stay below
//    its MFMAs (an A fragment feeds two column blocks: 0.5 KiB per MFMA; with all rows x 32 columns per wave it is
//    1 KiB, the whole of the LDS rate), and the second group gives each SIMD a wave to dequantise while the other
//    multiplies.  The groups' sums meet in LDS once, at the end.
//  * X and the raw weight bytes arrive by LDS-DMA: X in three slots of 64 k, weights in three of 128 k (64 bytes of a
//    Q4_K row), scales four super-blocks at a time (qstage.h).  A weight is dequantised by the two row waves of its
//    group only, straight into the B fragment.  Counted vmcnt, one barrier per step; a step's raw bytes and scales
//    are read from LDS a step early.
//  * lane half h of MFMA step s multiplies k = 16 h + 8 s .. + 8 of the group's 32: a lane's raw bytes are one
//    16-byte read.
//  * The second half of a step is multiplied beside the first dequantisation of the next (sched_group_barrier: six
//    vector instructions after an MFMA), so neither waits for the other inside a wave.
// What bounds it: vector issue and MFMAs need about 1000 of the SIMD's cycles a step of 64 k each (6.5 vector
// instructions an MFMA) and would overlap; a step takes 1900 (45 % MFMA, 55 % vector pipe busy), the rest is lost where
// the two waves of a SIMD wait for each other at the barrier.  Kept out of the way of the MFMAs: waits for LDS (operands
// are pinned behind the previous half-step; without that the compiler waits for every outstanding read: 78 -> 75 us),
// the DMA's issue (one instruction after an MFMA, not all behind the barrier: -> 71 us), address arithmetic (scalar).
// gate|up 28672 x 4096 of Q4_K with its activation: 256 rows 78 (gemm_bs.hip) -> 71 us, 128 rows 68 (gemm_q32.hip) ->
// 55, 701 rows 229 (copy, library, activation) -> 208 with the first of these three steps and 6 % less with all; 4096 x
// 14336 at 400 rows 115 (copy, library) -> 80, 4096 x 4096 42 -> 36.  Plain products of up to 256 rows with few columns
// stay with the other kernels: the autotuner times them all.  Inside a step of 256 rows the gated product is level with
// gemm_q32.hip's (2357 and 2346 us): there the weights' bytes in flight are the bound.
#include <type_traits>

#include "qstage.h"

namespace la {

typedef float f32x16w __attribute__((ext_vector_type(16)));

// LDS addresses of a lane's weight row (column c of a block of 32: row c & 15 of one of the block's two 16-row tiles)
// that no step changes; a step adds scalars and flips bits, one instruction each.
struct WdLane {
  uint32_t raw, raw2, q, d;
};
// keeps the loads of v before this place: without it the compiler waits for every outstanding LDS read at v's first use
template <typename T>
LA_DEV void wd_pin(T& v) {
  asm volatile("" : "+v"(v));
}

// Raw bytes and scales for a step.  P: which half of the tile's 128 k, gs: which 32 of the step's 64 k.  load(): wo, qo
// the offsets of the macro's slot and of the quad's buffer, j the step, o / oq of the column block's tile.
template <int FMT> struct WdW;

template <> struct WdW<FMT_Q4_K> {
  static constexpr int BYTES = 1024, PIECES = 1, QBYTES = SkW<FMT_Q4_K>::QBYTES;
  struct Ptr {
    const uint8_t* raw;
    typename SkW<FMT_Q4_K>::Ptr q;
  };
  template <typename Row>
  LA_DEV static Ptr ptr(const QW& w, int lane, Row row) {
    const int rr = lane >> 2;
    return Ptr{w.p0 + (size_t)row(rr) * (w.K >> 1) + 16 * ((lane & 3) ^ (rr >> 2)), SkW<FMT_Q4_K>::ptr(w, lane, row)};
  }
  LA_DEV static void issue(const Ptr& p, int m, uint8_t* dst) { sk_dma16(p.raw + 64 * m, dst); }
  u32x4 q;
  uint32_t scm, dd;
  float D, Mn;
  LA_DEV static WdLane lane(uint32_t raw, uint32_t qd, int r, int h, int gs, int) {
    return WdLane{raw + 64 * r + 16 * (h ^ (r >> 2)), 0, qd + sk_quad(r, 0), qd + 1024 + 16 * r};
  }
  template <int P>
  LA_DEV void load(const uint8_t* lds, const WdLane& a, uint32_t wo, uint32_t qo, int t, int o, int oq) {
    const int i = (t >> 2) & 3;
    q = *(const u32x4*)(lds + ((a.raw ^ (32 * P)) + wo) + o);
    scm = *(const uint32_t*)(lds + ((a.q ^ (16 * i)) + (qo + 4 * (t & 3))) + oq);
    dd = *(const uint32_t*)(lds + (a.d + (qo + 4 * i)) + oq);
  }
  LA_DEV void pin() { wd_pin(q), wd_pin(scm), wd_pin(dd); }
  LA_DEV void prep(int gs) {
    const uint32_t s = scm >> (16 * gs);
    D = h2f(dd & 0xFFFFu) * 512.f * ubyte_f(s, 0);
    Mn = -h2f(dd >> 16) * ubyte_f(s, 1);
  }
  template <int S>
  LA_DEV bf16x8 deq(int, int gs) const {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    const uint32_t a = ((S ? q.z : q.x) >> (4 * gs)) & 0x0F0F0F0Fu, b = ((S ? q.w : q.y) >> (4 * gs)) & 0x0F0F0F0Fu;
    const f32x2 a0 = __builtin_amdgcn_cvt_pk_f32_fp8(a, false), a1 = __builtin_amdgcn_cvt_pk_f32_fp8(a, true);
    const f32x2 b0 = __builtin_amdgcn_cvt_pk_f32_fp8(b, false), b1 = __builtin_amdgcn_cvt_pk_f32_fp8(b, true);
    const u32x4 v = {pk_bf16(fmaf(D, a0.x, Mn), fmaf(D, a0.y, Mn)), pk_bf16(fmaf(D, a1.x, Mn), fmaf(D, a1.y, Mn)),
                     pk_bf16(fmaf(D, b0.x, Mn), fmaf(D, b0.y, Mn)), pk_bf16(fmaf(D, b1.x, Mn), fmaf(D, b1.y, Mn))};
    return __builtin_bit_cast(bf16x8, v);
  }
};

// A step is two quarters of the half-block, a group one of them: quarter 2 (t & 1) + gs.
template <> struct WdW<FMT_Q6_K> {
  static constexpr int BYTES = 1024 + 512, PIECES = 2, QBYTES = SkW<FMT_Q6_K>::QBYTES;
  struct Ptr {
    const uint8_t *ql, *qh;
    typename SkW<FMT_Q6_K>::Ptr q;
  };
  template <typename Row>
  LA_DEV static Ptr ptr(const QW& w, int lane, Row row) {
    const int rr = lane >> 2, rh = (lane & 31) >> 1;
    return Ptr{w.p0 + (size_t)row(rr) * (w.K >> 1) + 16 * ((lane & 3) ^ (rr >> 2)),
               w.p1 + (size_t)row(rh) * (w.K >> 2) + 16 * ((lane & 1) ^ (rh >> 3)), SkW<FMT_Q6_K>::ptr(w, lane, row)};
  }
  LA_DEV static void issue(const Ptr& p, int m, uint8_t* dst) {
    sk_dma16(p.ql + 64 * m, dst);
    if ((threadIdx.x & 63) < 32) sk_dma16(p.qh + 32 * m, dst + 1024);
  }
  u32x4 l4, h4;
  int sc;
  uint32_t dbits;
  float D;
  // the quad's first d is at the lane's parity in its aligned dwords (4 super-blocks: an even number)
  LA_DEV static WdLane lane(uint32_t raw, uint32_t qd, int r, int h, int gs, int idx) {
    return WdLane{raw + 64 * r + 16 * ((2 * gs + h) ^ (r >> 2)), raw + 1024 + 32 * r + 16 * (h ^ (r >> 3)),
                  qd + sk_quad(r, 0) + 2 * gs + h, qd + 1024 + 16 * r + 2 * (idx & 1)};
  }
  template <int P>
  LA_DEV void load(const uint8_t* lds, const WdLane& a, uint32_t wo, uint32_t qo, int t, int o, int oq) {
    const int i = (t >> 2) & 3;
    l4 = *(const u32x4*)(lds + (a.raw + wo) + o);
    h4 = *(const u32x4*)(lds + (a.raw2 + wo) + o);
    sc = *(const int8_t*)(lds + ((a.q ^ (16 * i)) + (qo + 4 * (t & 3))) + oq);
    dbits = *(const uint16_t*)(lds + (a.d + (qo + 2 * i)) + oq);
  }
  LA_DEV void pin() { wd_pin(l4), wd_pin(h4), wd_pin(sc), wd_pin(dbits); }
  LA_DEV void prep(int) { D = h2f(dbits) * (float)sc; }
  template <int S>
  LA_DEV bf16x8 deq(int t, int gs) const {
    const int ls = 4 * (t & 1), hs = 4 * (t & 1) + 2 * gs;
    const uint32_t u0 = opaque((((S ? l4.z : l4.x) >> ls) & 0x0F0F0F0Fu) | ((((S ? h4.z : h4.x) >> hs) & 0x03030303u) << 4));
    const uint32_t u1 = opaque((((S ? l4.w : l4.y) >> ls) & 0x0F0F0F0Fu) | ((((S ? h4.w : h4.y) >> hs) & 0x03030303u) << 4));
    return bytes_bf16(u0, u1, D, -32.f * D);
  }
};

template <> struct WdW<FMT_Q8_0> {
  static constexpr int BYTES = 2048, PIECES = 2, QBYTES = SkW<FMT_Q8_0>::QBYTES;
  struct Ptr {
    const uint8_t *a, *b;
    typename SkW<FMT_Q8_0>::Ptr q;
  };
  template <typename Row>
  LA_DEV static Ptr ptr(const QW& w, int lane, Row row) {
    const int rr = lane >> 3;
    return Ptr{w.p0 + (size_t)row(rr) * w.K + 16 * ((lane & 7) ^ (rr >> 1)),
               w.p0 + (size_t)row(8 + rr) * w.K + 16 * ((lane & 7) ^ (4 + (rr >> 1))), SkW<FMT_Q8_0>::ptr(w, lane, row)};
  }
  LA_DEV static void issue(const Ptr& p, int m, uint8_t* dst) {
    sk_dma16(p.a + 128 * m, dst);
    sk_dma16(p.b + 128 * m, dst + 1024);
  }
  u32x4 q;
  uint32_t dbits;
  float D;
  LA_DEV static WdLane lane(uint32_t raw, uint32_t qd, int r, int h, int gs, int) {
    return WdLane{raw + 128 * r + 16 * ((2 * gs + h) ^ (r >> 1)), 0, qd + sk_quad(r, 0) + 2 * gs, 0};
  }
  template <int P>
  LA_DEV void load(const uint8_t* lds, const WdLane& a, uint32_t wo, uint32_t qo, int t, int o, int oq) {
    q = *(const u32x4*)(lds + ((a.raw ^ (64 * P)) + wo) + o);
    dbits = *(const uint16_t*)(lds + ((a.q ^ (16 * ((t >> 2) & 3))) + (qo + 4 * (t & 3))) + oq);
  }
  LA_DEV void pin() { wd_pin(q), wd_pin(dbits); }
  LA_DEV void prep(int) { D = h2f(dbits); }
  template <int S>
  LA_DEV bf16x8 deq(int, int) const {
    return bytes_bf16(opaque((S ? q.z : q.x) ^ 0x80808080u), opaque((S ? q.w : q.y) ^ 0x80808080u), D, -128.f * D);
  }
};

// The gated form's second weight: gate rows oa .. oa + F of the first, up rows ob .. ob + F of this one.
struct WdGlu {
  QW b;
  int oa, ob, F, act;
};

LA_DEV float wd_gelu_tanh(float x) { return 0.5f * x * (1.f + tanhf(0.7978845608f * (x + 0.044715f * x * x * x))); }

template <int FMT, int RB>
struct WdCfg {
  using W = WdW<FMT>;
  static constexpr int XB = 64 * RB * 128, XS = 3 * XB, WS = 8 * W::BYTES, WB = 3 * WS, QB = 2 * 8 * W::QBYTES;
  static constexpr int LDS = XS + WB + QB;
  static_assert(LDS <= 160 * 1024 && RB * 32 * 1024 <= LDS, "ring; the groups' exchange");
};

template <int FMT, int RB, bool GLU>
LA_DEV void wd_tile(uint8_t* lds, const QW& w, int tile, int m0, const bf16* __restrict__ X, int ldx, int M, int macros,
                    float* __restrict__ out, bf16* __restrict__ outb, int ldo, long slab, const WdGlu& glu) {
  using W = WdW<FMT>;
  using C = WdCfg<FMT, RB>;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 31, h = lane >> 5;
  const int gs = wave >> 2, mw = (wave >> 1) & 1, nw = wave & 1;
  const int N = GLU ? glu.F : w.N;
  const int M0 = blockIdx.z * macros, mend = min(w.K >> 7, M0 + macros);   // this split's 128-k macros
  const int t0 = 2 * M0, t1 = 2 * mend;

  // sources: the wave fetches RB pieces (8 rows) of X and one of the 8 weight tiles (GLU: 0-3 gate, 4-7 up)
  uint32_t xo[RB];   // bytes; a scalar base and a 32-bit offset need no address arithmetic in the vector pipe
#pragma unroll
  for (int i = 0; i < RB; ++i) {
    const int row = 8 * (wave * RB + i) + (lane >> 3);
    xo[i] = ((uint32_t)min(m0 + row, M - 1) * ldx + ((lane & 7) ^ ((row >> 1) & 7)) * 8) * 2;
  }
  const bool up = GLU && wave >= 4;
  auto trow = [&](int tl, int i) {   // weight row of row i of tile tl (rows past N repeat the last)
    if (GLU) return (tl >= 4 ? glu.ob : glu.oa) + min(64 * tile + 16 * (tl & 3) + i, N - 1);
    return min(128 * tile + 16 * tl + i, N - 1);
  };
  const typename W::Ptr wp = W::ptr(up ? glu.b : w, lane, [&](int i) { return trow(wave, i); });
  uint8_t* wring = lds + C::XS;
  uint8_t* quads = wring + C::WB;
  auto issue_x = [&](int t, int slot) {
#pragma unroll
    for (int i = 0; i < RB; ++i) sk_dma16((const uint8_t*)(X + min(t, t1 - 1) * 64) + xo[i], lds + slot * C::XB + (wave * RB + i) * 1024);
  };
  auto issue_w = [&](int m, int slot) { W::issue(wp, min(m, mend - 1), wring + slot * C::WS + wave * W::BYTES); };
  auto issue_quad = [&](int qd) { SkW<FMT>::issue_quad(wp.q, 4 * qd, quads + ((qd & 1) * 8 + wave) * W::QBYTES, lane); };
  // the wave's column block b: tiles tl(b) and tl(b) + 1; the lane's column is row r & 15 of tile tl(b) + (r >> 4)
  constexpr int TB = GLU ? 4 : 2;    // tiles from block 0 to block 1
  const int tl0 = (GLU ? 2 : 4) * nw + (r >> 4);
  const WdLane la0 = W::lane(C::XS + tl0 * W::BYTES, C::XS + C::WB + tl0 * W::QBYTES, r & 15, h, gs, trow(tl0, r & 15) * (w.K >> 8));
  const WdLane la1 = W::lane(C::XS + tl0 * W::BYTES, C::XS + C::WB + tl0 * W::QBYTES, r & 15, h, gs, trow(tl0 + TB, r & 15) * (w.K >> 8));
  auto fetch = [&](W (&f)[2], int t, auto odd, int wslot) {
    const uint32_t wo = wslot * C::WS, qo = ((t >> 4) & 1) * 8 * W::QBYTES;
    f[0].template load<decltype(odd)::value>(lds, la0, wo, qo, t, 0, 0);
    f[1].template load<decltype(odd)::value>(lds, la1, wo, qo, t, TB * W::BYTES, TB * W::QBYTES);
  };

  f32x16w acc[RB][2];
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[i][b][j] = 0.f;
  // A fragments: row 32 (RB mw + i) + r, chunk 4 gs + 2 h + s of the step
  int aoff[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) aoff[s] = (32 * RB * mw + r) * 128 + 16 * ((4 * gs + 2 * h + s) ^ ((r >> 1) & 7));

  // In flight, oldest first, when step t waits for its X: [X(t)] W X(t + 1), with W(m) issued two macros ahead
  issue_quad(t0 >> 4);
  issue_quad((t0 >> 4) + 1);
  issue_w(M0, 0);
  issue_x(t0, 0);
  issue_w(M0 + 1, 1);
  issue_x(t0 + 1, 1);
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * RB + W::PIECES) : "memory");
  W f[2][2];
  fetch(f[0], t0, std::false_type{}, 0);
  int xs = 0, ws = 0;                // slots of step t's X and of its macro
  // Half a step (one MFMA per block pair and 16 k) is multiplied while the next half is dequantised: the second half
  // of step t - 1 beside the first dequantisation of step t, so a wave has vector work between all its MFMAs.
  u32x4 a0[RB], a1[RB];
  bf16x8 b0[2], b1[2];
#pragma unroll
  for (int i = 0; i < RB; ++i) a1[i] = u32x4{};
#pragma unroll
  for (int b = 0; b < 2; ++b) b1[b] = bf16x8{};
  auto mul = [&](const u32x4 (&a)[RB], const bf16x8 (&bb)[2]) {
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int b = 0; b < 2; ++b) acc[i][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a[i]), bb[b], acc[i][b], 0, 0, 0);
  };
  auto mix = [&](bool dma) {         // an MFMA, then its share of the vector instructions and of the DMA
#pragma unroll
    for (int i = 0; i < 2 * RB; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
      if (dma) __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);
    }
  };
  auto step = [&](W (&cur)[2], W (&nxt)[2], int t, auto odd) {
#pragma unroll
    for (int i = 0; i < RB; ++i) wd_pin(a1[i]);
    cur[0].pin(), cur[1].pin();
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(RB + W::PIECES) : "memory");
    if ((t & 15) == 0 && t != t0) issue_quad((t >> 4) + 1);
    const uint8_t* x = lds + xs * C::XB;
#pragma unroll
    for (int i = 0; i < RB; ++i) a0[i] = *(const u32x4*)(x + aoff[0] + i * (32 * 128));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      cur[b].prep(gs);
      b0[b] = cur[b].template deq<0>(t, gs);
    }
    issue_x(t + 2, xs == 0 ? 2 : xs - 1);
    if (!decltype(odd)::value) issue_w((t >> 1) + 2, ws == 0 ? 2 : ws - 1);
    mul(a1, b1);
    mix(true);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < RB; ++i) wd_pin(a0[i]);
#pragma unroll
    for (int i = 0; i < RB; ++i) a1[i] = *(const u32x4*)(x + aoff[1] + i * (32 * 128));
    if (decltype(odd)::value) ws = ws == 2 ? 0 : ws + 1;
    fetch(nxt, t + 1, std::bool_constant<!decltype(odd)::value>{}, ws);
    xs = xs == 2 ? 0 : xs + 1;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int b = 0; b < 2; ++b) b1[b] = cur[b].template deq<1>(t, gs);
    mul(a0, b0);
    mix(false);
    __builtin_amdgcn_sched_barrier(0);
  };
  for (int t = t0; t < t1; t += 2) {
    step(f[0], f[1], t, std::false_type{});
    step(f[1], f[0], t + 1, std::true_type{});
  }
  mul(a1, b1);
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");   // every DMA has landed, every read is done

  // sums of the two K groups: each keeps half of the row blocks and hands the other half over
  constexpr int HB = RB / 2;
  f32x4* ex = (f32x4*)lds;
  auto place = [&](int wv, int i, int b, int q) { return ((((wv * HB + i) * 2 + b) * 4 + q) << 6) + lane; };
#pragma unroll
  for (int i = 0; i < HB; ++i)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        f32x4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = gs ? acc[i][b][4 * q + j] : acc[HB + i][b][4 * q + j];
        ex[place(wave, i, b, q)] = v;
      }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < HB; ++i) {
    f32x16w o[2];
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4 v = ex[place(wave ^ 4, i, b, q)];
#pragma unroll
        for (int j = 0; j < 4; ++j) o[b][4 * q + j] = v[j] + (gs ? acc[HB + i][b][4 * q + j] : acc[i][b][4 * q + j]);
      }
    const int mb = m0 + 32 * (RB * mw + (gs ? HB : 0) + i) + 4 * h;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int m = mb + 8 * (j >> 2) + (j & 3);
      if (m >= M) continue;
      if constexpr (GLU) {
        const int n = 64 * tile + 32 * nw + r;
        const float g = o[0][j];
        const float a = glu.act == 0 ? silu(g) : wd_gelu_tanh(g);
        if (n < N) outb[(size_t)m * ldo + n] = (bf16)(a * o[1][j]);
      } else {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const int n = 128 * tile + 64 * nw + 32 * b + r;
          if (n >= N) continue;
          if (outb) outb[(size_t)m * ldo + n] = (bf16)o[b][j];
          else out[(size_t)blockIdx.z * slab + (size_t)m * ldo + n] = o[b][j];
        }
      }
    }
  }
}

template <int FMT, int RB, bool GLU>
__global__ __launch_bounds__(512, 2) void wgemm_kernel(QW w, const bf16* __restrict__ X, int ldx, int M, int macros,
                                                       float* __restrict__ out, bf16* __restrict__ outb, int ldo,
                                                       long slab, WdGlu glu) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[WdCfg<FMT, RB>::LDS];
  wd_tile<FMT, RB, GLU>(lds, w, blockIdx.x, blockIdx.y * 64 * RB, X, ldx, M, macros, out, outb, ldo, slab, glu);
}

// A Q4_K weight and a Q6_K weight side by side (q|k beside v): the first tiles_a workgroups of a row are the former's.
template <int FA, int FB, int RB>
__global__ __launch_bounds__(512, 2) void wgemm2_kernel(QW wa, QW wb, int tiles_a, const bf16* __restrict__ X, int ldx,
                                                        int M, int macros, float* __restrict__ out,
                                                        bf16* __restrict__ outb, int ldo, long slab) {
  constexpr int LA = WdCfg<FA, RB>::LDS, LB = WdCfg<FB, RB>::LDS;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[LA > LB ? LA : LB];
  const int t = blockIdx.x, m0 = blockIdx.y * 64 * RB;
  if (t < tiles_a) wd_tile<FA, RB, false>(lds, wa, t, m0, X, ldx, M, macros, out, outb, ldo, slab, WdGlu{});
  else
    wd_tile<FB, RB, false>(lds, wb, t - tiles_a, m0, X, ldx, M, macros, out ? out + wa.N : nullptr,
                           outb ? outb + wa.N : nullptr, ldo, slab, WdGlu{});
}

static QW wd_qw(const void* const* p, int n, int K) {
  return QW{(const uint8_t*)p[0], (const uint8_t*)p[1], (const uint8_t*)p[2], (const uint8_t*)p[3], n, K};
}
static bool wd_odd(int fmt, int n, int K) { return fmt == FMT_Q6_K && (n & 1) && ((K >> 8) & 1); }   // whole dwords of d

}  // namespace la

// C ABI ---------------------------------------------------------------------------
// rb: rows of a workgroup in units of 64 (2, 4).  splits cut K in multiples of 128, all but the last equal.
extern "C" int la_wgemm(int fmt, const void* const* a, int N, int K, const void* X, int ldx, int M, int splits, void* out,
                        int ldo, long slab, int out_bf16, int rb, void* stream) {
  using namespace la;
  const int total = K >> 7, per = splits > 0 ? (total + splits - 1) / splits : 0;
  if (M < 1 || N < 1 || (K & 255) || splits < 1 || (long)per * (splits - 1) >= total || ldo < N || ldx < K || (ldx & 7) || (long)M * ldx >= (1L << 31) ||
      (out_bf16 ? splits != 1 : slab < (long)M * ldo) || wd_odd(fmt, N, K))
    return -1;
  const QW w = wd_qw(a, N, K);
  const dim3 grid((N + 127) / 128, (M + 64 * rb - 1) / (64 * rb), splits);
  hipStream_t st = (hipStream_t)stream;
  float* o = out_bf16 ? nullptr : (float*)out;
  bf16* ob = out_bf16 ? (bf16*)out : nullptr;
#define WD(F, R) hipLaunchKernelGGL((wgemm_kernel<F, R, false>), grid, dim3(512), 0, st, w, (const bf16*)X, ldx, M, per, o, ob, ldo, slab, WdGlu{})
#define WD_R(F)           \
  if (rb == 4) WD(F, 4);  \
  else if (rb == 2) WD(F, 2); \
  else return -2;         \
  break
  switch (fmt) {
    case FMT_Q4_K: WD_R(FMT_Q4_K);
    case FMT_Q6_K: WD_R(FMT_Q6_K);
    case FMT_Q8_0: WD_R(FMT_Q8_0);
    default: return -2;
  }
#undef WD_R
#undef WD
  return (int)hipGetLastError();
}

extern "C" int la_wgemm2(const void* const* a, int Na, const void* const* b, int Nb, int K, const void* X, int ldx, int M,
                         int splits, void* out, int ldo, long slab, int out_bf16, int rb, void* stream) {
  using namespace la;
  const int total = K >> 7, per = splits > 0 ? (total + splits - 1) / splits : 0;
  if (M < 1 || Na < 1 || Nb < 1 || (K & 255) || splits < 1 || (long)per * (splits - 1) >= total || ldo < Na + Nb || ldx < K ||
      (ldx & 7) || (long)M * ldx >= (1L << 31) || (out_bf16 ? splits != 1 : slab < (long)M * ldo) || wd_odd(FMT_Q6_K, Nb, K))
    return -1;
  const QW wa = wd_qw(a, Na, K), wb = wd_qw(b, Nb, K);
  const int ta = (Na + 127) / 128;
  const dim3 grid(ta + (Nb + 127) / 128, (M + 64 * rb - 1) / (64 * rb), splits);
  hipStream_t st = (hipStream_t)stream;
  float* o = out_bf16 ? nullptr : (float*)out;
  bf16* ob = out_bf16 ? (bf16*)out : nullptr;
  if (rb == 4)
    hipLaunchKernelGGL((wgemm2_kernel<FMT_Q4_K, FMT_Q6_K, 4>), grid, dim3(512), 0, st, wa, wb, ta, (const bf16*)X, ldx, M, per, o, ob, ldo, slab);
  else if (rb == 2)
    hipLaunchKernelGGL((wgemm2_kernel<FMT_Q4_K, FMT_Q6_K, 2>), grid, dim3(512), 0, st, wa, wb, ta, (const bf16*)X, ldx, M, per, o, ob, ldo, slab);
  else return -2;
  return (int)hipGetLastError();
}

// h = act(x Wg^T) * (x Wu^T) -> bf16 [M][ldo], F columns; gate and up rows as in la_qgemm_skinny_glu.
extern "C" int la_wgemm_glu(int fmt, const void* const* a, int oa, const void* const* b, int ob, int F, int K, const void* X,
                            int ldx, int M, void* out, int ldo, int act, int rb, void* stream) {
  using namespace la;
  if (M < 1 || F < 1 || (K & 255) || ldo < F || ldx < K || (ldx & 7) || (long)M * ldx >= (1L << 31) || (act != 0 && act != 3) || wd_odd(fmt, oa + F, K) ||
      wd_odd(fmt, ob + F, K))
    return -1;
  const QW w = wd_qw(a, oa + F, K);
  const WdGlu glu{wd_qw(b, ob + F, K), oa, ob, F, act};
  const dim3 grid((F + 63) / 64, (M + 64 * rb - 1) / (64 * rb), 1);
  hipStream_t st = (hipStream_t)stream;
#define WD(Q, R) hipLaunchKernelGGL((wgemm_kernel<Q, R, true>), grid, dim3(512), 0, st, w, (const bf16*)X, ldx, M, K >> 7, nullptr, (bf16*)out, ldo, 0L, glu)
#define WD_R(Q)           \
  if (rb == 4) WD(Q, 4);  \
  else if (rb == 2) WD(Q, 2); \
  else return -2;         \
  break
  switch (fmt) {
    case FMT_Q4_K: WD_R(FMT_Q4_K);
    case FMT_Q6_K: WD_R(FMT_Q6_K);
    case FMT_Q8_0: WD_R(FMT_Q8_0);
    default: return -2;
  }
#undef WD_R
#undef WD
  return (int)hipGetLastError();
}
