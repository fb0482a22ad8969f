// Quantised weight rows by LDS-DMA for the GEMMs that dequantise them in registers: a stage is 16 rows x 128 k.
#pragma once
#include "qweight.h"

namespace la {

constexpr int SK_K = 128;              // k of one stage

LA_DEV void sk_dma16(const void* g, void* l) {
  __builtin_amdgcn_global_load_lds(g, (__attribute__((address_space(3))) void*)l, 16, 0, 0);
}
LA_DEV void sk_dma4(const void* g, void* l) {
  __builtin_amdgcn_global_load_lds(g, (__attribute__((address_space(3))) void*)l, 4, 0, 0);
}

// Rows 0-3, 12-15 and 4-11 each numbered 0 .. 7: the two sets of rows that one phase reads at chunks c and c ^ d.
// sk_rot spreads them over the 8 chunks of which bit d is clear.
LA_DEV int sk_idx(int r) { return (r & 3) | ((r & 8) >> 1); }
template <int D>
LA_DEV int sk_rot(int r) {
  const int i = sk_idx(r);
  return D == 1 ? i << 1 : D == 2 ? (i & 1) | ((i & 6) << 1) : (i & 3) | ((i & 4) << 1);
}

// Per format: the 16 weight rows of a tile over one stage.  ptr(): this lane's source addresses (row(i): row i of the
// tile); issue(): DMA of stage ks to dst; issue_quad(): of the scales of four super-blocks; load() / prep() / deq<S>():
// lane (g, r)'s 32 weights of row r, 8 for each of the 4 MFMA steps; chunk(s, g): which 8 k of the stage those are.
template <int FMT> struct SkW;

// Scales are fetched for four super-blocks (a quad: 8 stages) at a time, 64 bytes of a row's scale plane: by the stage
// every row would cost two more requests of 4 or 8 bytes, three times as many in all.  Row r's 16 bytes of super-block i
// of the quad lie at 64 r + 16 (i ^ (r >> 2)).
LA_DEV int sk_quad(int r, int i) { return 64 * r + 16 * (i ^ (r >> 2)); }

// Q4_K: 64 bytes a row (two groups of 32: low nibbles the first 32 k, high nibbles the next), 4 (sc, m) pairs, d, dmin.
// Lane g: bytes 16 g .. 16 g + 15, i.e. 16 k of the blocks 2 (g >> 1) and 2 (g >> 1) + 1.  Codes 0 .. 15 read as fp8
// e4m3 are exactly code / 512, so one v_cvt_pk_f32_fp8 makes two of them.
template <> struct SkW<FMT_Q4_K> {
  static constexpr int BYTES = 1024, PIECES = 1, XD = 2, QBYTES = 1024 + 256;
  LA_DEV static int chunk(int s, int g) { return 8 * (g >> 1) + 4 * (s >> 1) + 2 * (g & 1) + (s & 1); }
  struct Ptr {
    const uint8_t *raw, *scm, *dd;
    int nsb, qi;
  };
  template <typename Row>
  LA_DEV static Ptr ptr(const QW& w, int lane, Row row) {
    Ptr p;
    const int rr = lane >> 2;
    p.nsb = w.K >> 8;
    p.qi = (lane & 3) ^ (rr >> 2);
    p.raw = w.p0 + (size_t)row(rr) * (w.K >> 1) + 16 * ((lane & 3) ^ (2 * (rr >> 3)));
    p.scm = w.p2 + (size_t)row(rr) * p.nsb * 16;
    p.dd = w.p3 + (size_t)row(rr) * p.nsb * 4;
    return p;
  }
  LA_DEV static void issue(const Ptr& p, int ks, uint8_t* dst) { sk_dma16(p.raw + 64 * ks, dst); }
  LA_DEV static void issue_quad(const Ptr& p, int sb, uint8_t* dst, int lane) {
    sk_dma16(p.scm + 16 * min(sb + p.qi, p.nsb - 1), dst);
    sk_dma4(p.dd + 4 * min(sb + (lane & 3), p.nsb - 1), dst + 1024);
  }
  u32x4 q;
  uint32_t scm, dd;
  float D[2], Mn[2];
  LA_DEV void load(const uint8_t* l, const uint8_t* qd, int t, int r, int g, int, int) {
    const int i = (t >> 1) & 3;
    q = *(const u32x4*)(l + 64 * r + 16 * (g ^ (2 * (r >> 3))));
    scm = *(const uint32_t*)(qd + sk_quad(r, i) + 8 * (t & 1) + 4 * (g >> 1));
    dd = *(const uint32_t*)(qd + 1024 + 16 * r + 4 * i);
  }
  LA_DEV void prep(int) {
    const float d = h2f(dd & 0xFFFFu) * 512.f, dmin = -h2f(dd >> 16);
    D[0] = d * ubyte_f(scm, 0);
    Mn[0] = dmin * ubyte_f(scm, 1);
    D[1] = d * ubyte_f(scm, 2);
    Mn[1] = dmin * ubyte_f(scm, 3);
  }
  template <int S>
  LA_DEV bf16x8 deq() const {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    constexpr int h = S >> 1;
    const uint32_t a = ((S & 1 ? q.z : q.x) >> (4 * h)) & 0x0F0F0F0Fu, b = ((S & 1 ? q.w : q.y) >> (4 * h)) & 0x0F0F0F0Fu;
    const f32x2 a0 = __builtin_amdgcn_cvt_pk_f32_fp8(a, false), a1 = __builtin_amdgcn_cvt_pk_f32_fp8(a, true);
    const f32x2 b0 = __builtin_amdgcn_cvt_pk_f32_fp8(b, false), b1 = __builtin_amdgcn_cvt_pk_f32_fp8(b, true);
    const u32x4 v = {pk_bf16(fmaf(D[h], a0.x, Mn[h]), fmaf(D[h], a0.y, Mn[h])),
                     pk_bf16(fmaf(D[h], a1.x, Mn[h]), fmaf(D[h], a1.y, Mn[h])),
                     pk_bf16(fmaf(D[h], b0.x, Mn[h]), fmaf(D[h], b0.y, Mn[h])),
                     pk_bf16(fmaf(D[h], b1.x, Mn[h]), fmaf(D[h], b1.y, Mn[h]))};
    return __builtin_bit_cast(bf16x8, v);
  }
};

// Q6_K: a stage is one 128-half of the block: ql 64 bytes (l and 32 + l; low nibbles k 0-63, high 64-127), qh 32 bytes
// (2 bits for each quarter of 32 k), 8 scales of 16 k, d.  Lane g: l = 8 g .. 8 g + 7, step s the quarter s.
template <> struct SkW<FMT_Q6_K> {
  static constexpr int BYTES = 1024 + 512, PIECES = 2, XD = 1, QBYTES = 1024 + 256;
  LA_DEV static int chunk(int s, int g) { return 4 * s + g; }
  struct Ptr {
    const uint8_t *ql, *qh, *sc, *d;
    int nsb, qi, idx, last;   // idx: the row's first index in the plane of 2-byte scales, last: the plane's last dword
  };
  template <typename Row>
  LA_DEV static Ptr ptr(const QW& w, int lane, Row row) {
    Ptr p;
    const int rr = lane >> 2, rh = (lane & 31) >> 1;
    p.nsb = w.K >> 8;
    p.qi = (lane & 3) ^ (rr >> 2);
    p.ql = w.p0 + (size_t)row(rr) * (w.K >> 1) + 16 * ((lane & 3) ^ (rr >> 2));
    p.qh = w.p1 + (size_t)row(rh) * (w.K >> 2) + 16 * ((lane & 1) ^ (rh >> 3));
    p.sc = w.p2 + (size_t)row(rr) * p.nsb * 16;
    p.d = w.p3;
    p.idx = row(rr) * p.nsb;
    p.last = (w.N * p.nsb >> 1) - 1;
    return p;
  }
  LA_DEV static void issue(const Ptr& p, int ks, uint8_t* dst) {
    sk_dma16(p.ql + 64 * ks, dst);
    if ((threadIdx.x & 63) < 32) sk_dma16(p.qh + 32 * ks, dst + 1024);
  }
  // d is 2 bytes at any even address: the aligned dwords that hold a row's four of them (three at most)
  LA_DEV static void issue_quad(const Ptr& p, int sb, uint8_t* dst, int lane) {
    sk_dma16(p.sc + 16 * min(sb + p.qi, p.nsb - 1), dst);
    sk_dma4(p.d + 4 * (size_t)min(((p.idx + sb) >> 1) + (lane & 3), p.last), dst + 1024);
  }
  u32x2 la, lb, qh, sc;
  uint16_t dbits;
  float S[4];
  LA_DEV void load(const uint8_t* l, const uint8_t* qd, int t, int r, int g, int idx, int sb) {
    const int i = (t >> 1) & 3;
    const uint8_t* b = l + 64 * r + 8 * (g & 1);
    la = *(const u32x2*)(b + 16 * ((g >> 1) ^ (r >> 2)));
    lb = *(const u32x2*)(b + 16 * ((2 + (g >> 1)) ^ (r >> 2)));
    qh = *(const u32x2*)(l + 1024 + 32 * r + 16 * ((g >> 1) ^ (r >> 3)) + 8 * (g & 1));
    sc = *(const u32x2*)(qd + sk_quad(r, i) + 8 * (t & 1));
    const int q0 = idx + sb - i, e = idx + sb;     // the quad's first and this super-block's place in the plane
    dbits = *(const uint16_t*)(qd + 1024 + 16 * r + 4 * ((e >> 1) - (q0 >> 1)) + 2 * (e & 1));
  }
  LA_DEV void prep(int g) {
    const float d = h2f(dbits);
    const int sh = 8 * (g >> 1);
    S[0] = d * (float)((int)(sc.x << (24 - sh)) >> 24);
    S[1] = d * (float)((int)(sc.x << (8 - sh)) >> 24);
    S[2] = d * (float)((int)(sc.y << (24 - sh)) >> 24);
    S[3] = d * (float)((int)(sc.y << (8 - sh)) >> 24);
  }
  template <int St>
  LA_DEV bf16x8 deq() const {
    const u32x2 L = (St & 1) ? lb : la;
    constexpr int ls = 4 * (St >> 1), hs = 2 * St;
    const uint32_t u0 = opaque(((L.x >> ls) & 0x0F0F0F0Fu) | (((qh.x >> hs) & 0x03030303u) << 4));
    const uint32_t u1 = opaque(((L.y >> ls) & 0x0F0F0F0Fu) | (((qh.y >> hs) & 0x03030303u) << 4));
    return bytes_bf16(u0, u1, S[St], -32.f * S[St]);
  }
};

// Q8_0: 128 bytes and 4 scales a row.  Lane g: block g.
template <> struct SkW<FMT_Q8_0> {
  static constexpr int BYTES = 2048, PIECES = 2, XD = 4, QBYTES = 1024;
  LA_DEV static int chunk(int s, int g) { return 4 * g + s; }
  // 8 chunks a row, 2 g and 2 g + 1 read: as sk_rot with 3 bits, bit 1 clear, for the 8 rows of one parity
  LA_DEV static int rot(int r) { return ((r >> 1) & 1) | (((r >> 3) & 1) << 2); }
  struct Ptr {
    const uint8_t *a, *b, *d;
    int nsb, qi;
  };
  template <typename Row>
  LA_DEV static Ptr ptr(const QW& w, int lane, Row row) {
    Ptr p;
    const int rr = lane >> 3;
    p.nsb = w.K >> 8;
    p.qi = (lane & 3) ^ (lane >> 4);
    p.a = w.p0 + (size_t)row(rr) * w.K + 16 * ((lane & 7) ^ rot(rr));
    p.b = w.p0 + (size_t)row(8 + rr) * w.K + 16 * ((lane & 7) ^ rot(8 + rr));
    p.d = w.p1 + (size_t)row(lane >> 2) * p.nsb * 16;
    return p;
  }
  LA_DEV static void issue(const Ptr& p, int ks, uint8_t* dst) {
    sk_dma16(p.a + 128 * ks, dst);
    sk_dma16(p.b + 128 * ks, dst + 1024);
  }
  LA_DEV static void issue_quad(const Ptr& p, int sb, uint8_t* dst, int) {
    sk_dma16(p.d + 16 * min(sb + p.qi, p.nsb - 1), dst);
  }
  u32x4 a, b;
  uint16_t dbits;
  float d;
  LA_DEV void load(const uint8_t* l, const uint8_t* qd, int t, int r, int g, int, int) {
    a = *(const u32x4*)(l + 128 * r + 16 * ((2 * g) ^ rot(r)));
    b = *(const u32x4*)(l + 128 * r + 16 * ((2 * g + 1) ^ rot(r)));
    dbits = *(const uint16_t*)(qd + sk_quad(r, (t >> 1) & 3) + 8 * (t & 1) + 2 * g);
  }
  LA_DEV void prep(int) {
    d = h2f(dbits);
  }
  template <int S>
  LA_DEV bf16x8 deq() const {
    const u32x4 v = S < 2 ? a : b;
    const uint32_t lo = (S & 1) ? v.z : v.x, hi = (S & 1) ? v.w : v.y;
    // signed bytes with the sign bit flipped: 0 .. 255, 128 too much
    return bytes_bf16(opaque(lo ^ 0x80808080u), opaque(hi ^ 0x80808080u), d, -128.f * d);
  }
};

template <> struct SkW<FMT_BF16> {
  static constexpr int BYTES = 4096, PIECES = 4, XD = 4, QBYTES = 0;
  LA_DEV static int chunk(int s, int g) { return 4 * g + s; }
  struct Ptr {
    const uint8_t* p[4];
  };
  template <typename Row>
  LA_DEV static Ptr ptr(const QW& w, int lane, Row row) {
    Ptr p;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int rr = 4 * i + (lane >> 4);
      p.p[i] = w.p0 + (size_t)row(rr) * w.K * 2 + 16 * ((lane & 15) ^ sk_rot<XD>(rr));
    }
    return p;
  }
  LA_DEV static void issue(const Ptr& p, int ks, uint8_t* dst) {
#pragma unroll
    for (int i = 0; i < 4; ++i) sk_dma16(p.p[i] + 256 * ks, dst + 1024 * i);
  }
  LA_DEV static void issue_quad(const Ptr&, int, uint8_t*, int) {}
  bf16x8 v[4];
  LA_DEV void prep(int) {}
  LA_DEV void load(const uint8_t* l, const uint8_t*, int, int r, int g, int, int) {
#pragma unroll
    for (int s = 0; s < 4; ++s) v[s] = *(const bf16x8*)(l + 256 * r + 16 * (chunk(s, g) ^ sk_rot<XD>(r)));
  }
  template <int S>
  LA_DEV bf16x8 deq() const { return v[S]; }
};

}  // namespace la
