// Quantised "skinny" GEMM for decode / small batches:  out[s][m][n] = sum_{k in split s} X[m,k] * W[n,k]
// and its gated form                                   out[m][j]    = act(x Wg[j]^T) * (x Wu[j]^T)   (bf16)
//
// Shape of the work:
//  * A workgroup of 4 waves owns 64 NW output columns (wave: NW tiles of 16) and all M <= 64 rows; a stage is 128 k.
//  * Weights and activations arrive by LDS-DMA in NS-slot rings.  A weight row's bytes of a stage are contiguous (64
//    of Q4_K), so an instruction reads whole 64-byte pieces of 16 rows: with each lane loading its own fragment
//    straight to registers neighbouring lanes are in different rows, every lane is a line look-up of its own, and
//    that, not HBM, was the bound (390 cycles of the CU's address path per 16 x 256 weights; about 110 here).
//  * A wave dequantises its own columns to bf16 for v_mfma_f32_16x16x32_bf16; the raw bytes are private to the wave,
//    the activations shared by the 4 waves; counted vmcnt, one barrier per stage.
//  * 16-byte chunks are exchanged inside their row by an XOR on the SOURCE address, chosen so that the lanes which
//    ds_read_b128 serves together (0-3, 12-15, 20-27; 4-11, 16-19, 28-31; the same + 32) hit different banks.
//  * A stage's weights are read from LDS an iteration before they are used, and all its activations before the first
//    product, so the vector pipe does not wait for LDS between its dequantisations.
//  * K is split over grid.y where the columns leave CUs idle: fp32 slabs summed by the consuming kernel (rmsnorm /
//    rope prologue), never by atomics.
// What bounds it: 28672 x 4096 of Q4_K (74 MB) gated, 4 to 16 rows: 23.4 us, of which 16.5 remain without the
// arithmetic (2.6 vector instructions a weight: about 10 us of every SIMD).  Before: 28.5 us ungated and 4.6 for the
// activation kernel; 50 rows 43 + 4.8 -> 33; 128256 x 4096 of Q6_K, 16 rows: 131 -> 113; 4096 x 14336 of Q6_K:
// 22.4 -> 17.5; the gated 8-bit form 38 + 4.6 -> 27.5.
#include "qstage.h"

namespace la {

// The gated form's second weight: gate rows oa .. oa + F of the first, up rows ob .. ob + F of this one.
struct SkGlu {
  QW b;
  int oa, ob, F, act;
  bf16* out;
};

LA_DEV float sk_gelu_tanh(float x) { return 0.5f * x * (1.f + tanhf(0.7978845608f * (x + 0.044715f * x * x * x))); }

template <int FMT, int MT, int WV, bool GLU>
struct SkCfg {
  using W = SkW<FMT>;
  static constexpr int XB = 16 * MT * SK_K * 2, SLOT = XB + WV * W::BYTES, QUADS = 2 * WV * W::QBYTES;
  // slots of the ring: for two to three workgroups of 4 waves a CU, or one of 8
  static constexpr int WANT = ((WV == 8 ? 150 : 52) * 1024 - QUADS) / SLOT;
  static constexpr int FIT = (160 * 1024 - QUADS) / SLOT;
  static constexpr int NS = WANT >= 4 ? (WANT > 8 ? 8 : WANT) : FIT < 4 ? FIT : 4;
  static_assert(NS >= 3, "ring");
  static constexpr int LDS = NS * SLOT + QUADS;
};

template <int FMT, int MT, int WV, bool GLU>
LA_DEV void sk_tile(uint8_t* lds, const QW& w, int tile, const bf16* __restrict__ X, int ldx, int M, int k_per_split,
                    float* __restrict__ out, int ldo, long slab, const SkGlu& glu) {
  static_assert(!GLU || WV == 8, "4 waves of gate and 4 of up tiles");
  using W = SkW<FMT>;
  using C = SkCfg<FMT, MT, WV, GLU>;
  constexpr int NS = C::NS;
  constexpr int PX = 4 * MT < WV ? 1 : 4 * MT / WV;    // pieces (4 rows) of X a wave fetches; MT 1, 8 waves: each by two
  constexpr int L = PX + W::PIECES;                    // DMAs of a wave per stage
  static_assert((NS - 3) * L < 64 && NS <= 8, "vmcnt; a quad's scales have landed 8 stages later");

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, r = lane & 15;
  const int N = GLU ? glu.F : w.N;
  const int nst = k_per_split / SK_K, ks0 = blockIdx.y * nst;
  const bool up = GLU && wave >= 4;
  const int c0 = GLU ? (tile * 4 + (wave & 3)) * 16 : (tile * WV + wave) * 16;   // the wave's first column

  // sources: pieces of X, the tile's planes (rows past N repeat the last)
  const bf16* xp[PX];
#pragma unroll
  for (int i = 0; i < PX; ++i) {
    const int row = 4 * ((wave * PX + i) % (4 * MT)) + (lane >> 4);
    xp[i] = X + (size_t)min(row, M - 1) * ldx + ((lane & 15) ^ sk_rot<W::XD>(row & 15)) * 8;
  }
  const QW wt = up ? glu.b : w;
  auto row = [&](int i) { return (GLU ? (up ? glu.ob : glu.oa) : 0) + min(c0 + i, N - 1); };
  const typename W::Ptr wp = W::ptr(wt, lane, row);
  const int idx = row(r) * (w.K >> 8);
  auto issue = [&](int t, int slot) {        // (clamped, never behind a branch: the count of DMAs in flight is fixed)
    uint8_t* s = lds + slot * C::SLOT;
    const int ks = ks0 + min(t, nst - 1);
#pragma unroll
    for (int i = 0; i < PX; ++i) sk_dma16(xp[i] + ks * SK_K, s + ((wave * PX + i) % (4 * MT)) * 1024);
    W::issue(wp, ks, s + C::XB + wave * W::BYTES);
  };
  uint8_t* quads = lds + NS * C::SLOT + wave * (2 * W::QBYTES);
  auto issue_quad = [&](int t, int buf) {    // scales of the stages t .. t + 7
    W::issue_quad(wp, (ks0 + t) >> 1, quads + buf * W::QBYTES, lane);
  };
  auto fetch = [&](W& f, int t, int slot) {
    f.load(lds + slot * C::SLOT + C::XB + wave * W::BYTES, quads + ((t >> 3) & 1) * W::QBYTES, t, r, g, idx, (ks0 + t) >> 1);
  };

  f32x4 acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  int xoff[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) xoff[s] = r * (SK_K * 2) + 16 * (W::chunk(s, g) ^ sk_rot<W::XD>(r));

  issue_quad(0, 0);
#pragma unroll
  for (int t = 0; t < NS - 1; ++t) issue(t, t);
  W f[2];
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 2) * L) : "memory");
  fetch(f[0], 0, 0);
  int slot = 0;
  // Iteration t multiplies stage t: its weights are in registers, read from LDS during iteration t - 1
  auto step = [&](W& cur, W& nxt, int t) {
    // this wave's part of stage t + 1 has landed; with the barrier everyone's part of stage t has (waited for an
    // iteration ago), and the slot of stage t - 1 is free
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NS - 3) * L) : "memory");
    if ((t & 7) == 0) issue_quad(t + 8, ((t >> 3) + 1) & 1);
    issue(t + NS - 1, slot == 0 ? NS - 1 : slot - 1);
    const uint8_t* s = lds + slot * C::SLOT;
    bf16x8 a[4][MT];
    slot = slot == NS - 1 ? 0 : slot + 1;
#pragma unroll
    for (int q = 0; q < (MT > 2 ? 1 : 4); ++q)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) a[q][mt] = *(const bf16x8*)(s + xoff[q] + mt * (16 * SK_K * 2));
    fetch(nxt, t + 1, slot);
    __builtin_amdgcn_sched_barrier(0);
    cur.prep(g);
#define SK_STEP(S)                                                                                    \
  {                                                                                                   \
    if constexpr (MT > 2 && S < 3) {                                                                  \
      _Pragma("unroll") for (int mt = 0; mt < MT; ++mt)                                               \
        a[S + 1][mt] = *(const bf16x8*)(s + xoff[S + 1] + mt * (16 * SK_K * 2));                      \
    }                                                                                                 \
    const bf16x8 b = cur.template deq<S>();                                                           \
    _Pragma("unroll") for (int mt = 0; mt < MT; ++mt)                                                 \
      acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[S][mt], b, acc[mt], 0, 0, 0);               \
  }
    SK_STEP(0) SK_STEP(1) SK_STEP(2) SK_STEP(3)
#undef SK_STEP
  };
  for (int t = 0; t < nst; t += 2) {         // (a split is whole super-blocks: an even number of stages)
    step(f[0], f[1], t);
    step(f[1], f[0], t + 1);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the clamped last stages: nothing may land after the wave's end

  const int n = c0 + r;
  if constexpr (GLU) {
    __syncthreads();
    f32x4* ex = (f32x4*)lds;
    if (up) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) ex[((wave - 4) * MT + mt) * 64 + lane] = acc[mt];
    }
    __syncthreads();
    if (up || n >= N) return;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const f32x4 u = ex[(wave * MT + mt) * 64 + lane];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = mt * 16 + 4 * g + i;
        const float a = glu.act == 0 ? silu(acc[mt][i]) : sk_gelu_tanh(acc[mt][i]);
        if (m < M) glu.out[(size_t)m * ldo + n] = (bf16)(a * u[i]);
      }
    }
  } else {
    if (n >= N) return;
    float* o = out + (size_t)blockIdx.y * slab;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = mt * 16 + 4 * g + i;
        if (m < M) o[(size_t)m * ldo + n] = acc[mt][i];
      }
  }
}

template <int FMT, int MT, int WV, bool GLU>
__global__ __launch_bounds__(64 * WV, 2) void qgemm_skinny_kernel(
    QW w, const bf16* __restrict__ X, int ldx, int M, int k_per_split, float* __restrict__ out, int ldo,
    long slab, SkGlu glu) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[SkCfg<FMT, MT, WV, GLU>::LDS];
  sk_tile<FMT, MT, WV, GLU>(lds, w, blockIdx.x, X, ldx, M, k_per_split, out, ldo, slab, glu);
}

// Two weights of the same K and different formats side by side (q|k in Q4_K beside v in Q6_K): columns 0 .. wa.N of
// the output from the first tiles_a workgroups of every split, the others from the rest.  v alone is 16 workgroups.
template <int FA, int FB, int MT, int WV>
__global__ __launch_bounds__(64 * WV, 2) void qgemm_skinny2_kernel(
    QW wa, QW wb, int tiles_a, const bf16* __restrict__ X, int ldx, int M, int k_per_split, float* __restrict__ out,
    int ldo, long slab) {
  constexpr int LA = SkCfg<FA, MT, WV, false>::LDS, LB = SkCfg<FB, MT, WV, false>::LDS;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[LA > LB ? LA : LB];
  const int t = blockIdx.x;
  if (t < tiles_a) sk_tile<FA, MT, WV, false>(lds, wa, t, X, ldx, M, k_per_split, out, ldo, slab, SkGlu{});
  else sk_tile<FB, MT, WV, false>(lds, wb, t - tiles_a, X, ldx, M, k_per_split, out + wa.N, ldo, slab, SkGlu{});
}

// Waves of a workgroup: 4 up to 32 rows; 8 above, where half the staged activations per column count for more than a
// second workgroup on the CU (28672 x 4096 Q4_K, 50 rows: 35 us against 47), and for the gated form, which has about
// one workgroup a CU.
template <int FMT, int MT, bool GLU>
static void launch_skinny_t(const QW& w, const bf16* X, int ldx, int M, int splits, float* out, int ldo, long slab,
                            const SkGlu& glu, hipStream_t st) {
  constexpr int WV = GLU ? 8 : MT == 4 ? 8 : 4;
  const int cols = GLU ? 64 : 16 * WV;
  dim3 grid(((GLU ? glu.F : w.N) + cols - 1) / cols, splits);
  hipLaunchKernelGGL((qgemm_skinny_kernel<FMT, MT, WV, GLU>), grid, dim3(64 * WV), 0, st, w, X, ldx, M,
                     w.K / splits, out, ldo, slab, glu);
}

template <int FMT, bool GLU>
static void launch_skinny_f(const QW& w, const bf16* X, int ldx, int M, int splits, float* out, int ldo, long slab,
                            const SkGlu& glu, hipStream_t st) {
  if (M <= 16) launch_skinny_t<FMT, 1, GLU>(w, X, ldx, M, splits, out, ldo, slab, glu, st);
  else if (M <= 32) launch_skinny_t<FMT, 2, GLU>(w, X, ldx, M, splits, out, ldo, slab, glu, st);
  else launch_skinny_t<FMT, 4, GLU>(w, X, ldx, M, splits, out, ldo, slab, glu, st);
}

template <int FA, int FB, int MT, int WV>
static void launch_skinny2(const QW& wa, const QW& wb, const bf16* X, int ldx, int M, int splits, float* out, int ldo,
                           long slab, hipStream_t st) {
  const int cols = 16 * WV, ta = (wa.N + cols - 1) / cols, tb = (wb.N + cols - 1) / cols;
  hipLaunchKernelGGL((qgemm_skinny2_kernel<FA, FB, MT, WV>), dim3(ta + tb, splits), dim3(64 * WV), 0, st, wa, wb, ta, X,
                     ldx, M, wa.K / splits, out, ldo, slab);
}

}  // namespace la

// C ABI ---------------------------------------------------------------------------
extern "C" int la_qgemm_skinny(int fmt, const void* p0, const void* p1, const void* p2, const void* p3,
                               int N, int K, const void* X, int ldx, int M, int splits, void* out,
                               int ldo, long slab, void* stream) {
  using namespace la;
  if (M < 1 || M > 64 || (K & 255) || splits < 1 || ((K >> 8) % splits) || ldo < N || slab < (long)M * ldo) return -1;
  if (fmt == FMT_Q6_K && (N & 1) && ((K >> 8) & 1)) return -1;   // SkW<FMT_Q6_K>: whole dwords of the plane of d
  QW w{(const uint8_t*)p0, (const uint8_t*)p1, (const uint8_t*)p2, (const uint8_t*)p3, N, K};
  hipStream_t st = (hipStream_t)stream;
  const bf16* x = (const bf16*)X;
  float* o = (float*)out;
  switch (fmt) {
    case FMT_Q4_K: launch_skinny_f<FMT_Q4_K, false>(w, x, ldx, M, splits, o, ldo, slab, SkGlu{}, st); break;
    case FMT_Q6_K: launch_skinny_f<FMT_Q6_K, false>(w, x, ldx, M, splits, o, ldo, slab, SkGlu{}, st); break;
    case FMT_Q8_0: launch_skinny_f<FMT_Q8_0, false>(w, x, ldx, M, splits, o, ldo, slab, SkGlu{}, st); break;
    case FMT_BF16: launch_skinny_f<FMT_BF16, false>(w, x, ldx, M, splits, o, ldo, slab, SkGlu{}, st); break;
    default: return -2;
  }
  return (int)hipGetLastError();
}

// h = act(x Wg^T) * (x Wu^T) -> bf16 [M][ldo], F columns.  Gate rows oa .. oa + F of planes a, up rows ob .. ob + F of
// planes b (the same planes with ob = F for one fused [2 F, K] weight).  act: 0 SwiGLU, 3 GeGLU (ops.ACT_*).
extern "C" int la_qgemm_skinny_glu(int fmt, const void* const* a, int oa, const void* const* b, int ob, int F, int K,
                                   const void* X, int ldx, int M, void* out, int ldo, int act, void* stream) {
  using namespace la;
  if (M < 1 || M > 64 || F < 1 || (K & 255) || ldo < F || ldx < K || (ldx & 7) || (act != 0 && act != 3)) return -1;
  if (fmt == FMT_Q6_K && ((K >> 8) & 1) && (((oa + F) & 1) || ((ob + F) & 1))) return -1;   // whole dwords of the plane of d
  auto qw = [K](const void* const* p, int n) {
    return QW{(const uint8_t*)p[0], (const uint8_t*)p[1], (const uint8_t*)p[2], (const uint8_t*)p[3], n, K};
  };
  QW w = qw(a, oa + F);
  const SkGlu glu{qw(b, ob + F), oa, ob, F, act, (bf16*)out};
  hipStream_t st = (hipStream_t)stream;
  const bf16* x = (const bf16*)X;
  switch (fmt) {
    case FMT_Q4_K: launch_skinny_f<FMT_Q4_K, true>(w, x, ldx, M, 1, nullptr, ldo, 0, glu, st); break;
    case FMT_Q6_K: launch_skinny_f<FMT_Q6_K, true>(w, x, ldx, M, 1, nullptr, ldo, 0, glu, st); break;
    case FMT_Q8_0: launch_skinny_f<FMT_Q8_0, true>(w, x, ldx, M, 1, nullptr, ldo, 0, glu, st); break;
    case FMT_BF16: launch_skinny_f<FMT_BF16, true>(w, x, ldx, M, 1, nullptr, ldo, 0, glu, st); break;
    default: return -2;
  }
  return (int)hipGetLastError();
}

// [x Wa^T | x Wb^T] of a Q4_K and a Q6_K weight of the same K in one launch: fp32 slabs [splits][M][ldo].
extern "C" int la_qgemm_skinny2(const void* const* a, int Na, const void* const* b, int Nb, int K, const void* X, int ldx,
                                int M, int splits, void* out, int ldo, long slab, void* stream) {
  using namespace la;
  if (M < 1 || M > 64 || Na < 1 || Nb < 1 || (K & 255) || splits < 1 || ((K >> 8) % splits) || ldo < Na + Nb ||
      slab < (long)M * ldo || ldx < K || (ldx & 7))
    return -1;
  if ((Nb & 1) && ((K >> 8) & 1)) return -1;   // SkW<FMT_Q6_K>: whole dwords of the plane of d
  const QW wa{(const uint8_t*)a[0], (const uint8_t*)a[1], (const uint8_t*)a[2], (const uint8_t*)a[3], Na, K};
  const QW wb{(const uint8_t*)b[0], (const uint8_t*)b[1], (const uint8_t*)b[2], (const uint8_t*)b[3], Nb, K};
  hipStream_t st = (hipStream_t)stream;
  const bf16* x = (const bf16*)X;
  float* o = (float*)out;
  if (M <= 16) launch_skinny2<FMT_Q4_K, FMT_Q6_K, 1, 4>(wa, wb, x, ldx, M, splits, o, ldo, slab, st);
  else if (M <= 32) launch_skinny2<FMT_Q4_K, FMT_Q6_K, 2, 4>(wa, wb, x, ldx, M, splits, o, ldo, slab, st);
  else launch_skinny2<FMT_Q4_K, FMT_Q6_K, 4, 8>(wa, wb, x, ldx, M, splits, o, ldo, slab, st);
  return (int)hipGetLastError();
}
