// Causal prompt attention over the paged cache for plain softmax layers (no score extras), head widths 64 and 128.
//
// Workgroup = 64 query rows x HPW query heads of one kv head; every wave holds 32 rows of one head, so K and V are
// staged in LDS once for all the heads that share them.  Tiles of 64 keys:
//   S^T[32 keys x 32 rows] = K . Q^T      (v_mfma_f32_32x32x16_bf16, keys on MFMA rows)
//   O^T[32 d x 32 rows]   += V^T . P^T
// A lane owns one query row in both products: maxima and sums are in-lane but for one exchange with lane ^ 32, the
// rescale factor is one register, and P never leaves the registers.  For that, MFMA row m of a block of 32 keys
// takes key flash_key(m) (bits 2 and 3 swapped): a lane's scores 8j .. 8j+7 are then the 8 CONSECUTIVE keys
// 16j + 8 (lane >> 5) .. +7, which is the B fragment that the second product wants beside V's 16-byte units
// ([key group of 8][d][8] in the cache and in LDS alike).
// K rows lie in LDS with their 16-byte chunks rotated by an XOR with m & 15, so the 32 rows of a fragment read
// start in different banks; V units are read and written in order.  Global loads of tile t + 1 are in flight while
// tile t is multiplied; one barrier per tile.
//
// What bounds it: per tile and wave 32 MFMAs (1024 cycles), 32 KiB of LDS reads (the four SIMDs' share of a cycle's
// 128 bytes: 1024 cycles too) and about as many cycles of softmax arithmetic, which two waves per SIMD overlap in part.
// 2048 rows behind 10007 keys, 32 heads over 8, width 128: 3233 us with the 64 x 32 tile of one head that
// attn_prefill_kernel takes (114 TFLOP/s), 451 us here (821); one prompt of 701 tokens 96 -> 26 us; 64 of 128 164 -> 51.
// A third schedule, with the next tile's score product between the exponentials, was 5 % slower (V arrives one half
// iteration later, the waves of a SIMD overlap the two anyway).  39 % MFMA and 42 % vector pipe busy, a third of the
// waves' time is waits; four waves a SIMD (two key groups in one workgroup) spill: a wave holds 172 registers.
// Few rows behind a long context leave most of the chip idle: there a tile's keys are shared by several workgroups
// (FlashSplit; 100 rows behind 8000 keys 215 -> 41 us, 16 behind 2000 56 -> 16).
#pragma once
#include "common.h"

namespace la {

constexpr int FL_KT = 64;  // keys per tile
constexpr int FL_QT = 64;  // query rows per workgroup (the rows of a prefill work tile)

// Keys split over grid.z: unnormalised sums [P][T][Hq][DH] and (maximum, sum) [P][T][Hq], merged by flash_merge_kernel.
struct FlashSplit {
  float* o;
  float2* ml;
  int T;
};

LA_DEV int flash_key(int m) { return (m & ~12) | ((m & 4) << 1) | ((m & 8) >> 1); }

template <int DH, int HPW, bool SPLIT>
__global__ __launch_bounds__(HPW * 128) __attribute__((amdgpu_waves_per_eu(2))) void prefill_flash_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ kc, const bf16* __restrict__ vc,
    const int* __restrict__ tiles, const int* __restrict__ cu_q, const int* __restrict__ ctx_lens,
    const int* __restrict__ block_tables, int max_blocks, int Hq, int Hkv, int bs_shift, float sl2,
    bf16* __restrict__ out, FlashSplit sp) {
  constexpr int NT = HPW * 128;
  constexpr int CH = DH / 8;                 // 16-byte chunks of a K row
  constexpr int KS = DH / 16;                // MFMA k steps of the score product
  constexpr int ND = DH / 32;                // 32-wide d tiles of the output
  constexpr int NU = FL_KT * CH / NT;        // 16-byte units of K (and of V) a thread stages per tile
  __shared__ __attribute__((aligned(16))) bf16 sk[2][FL_KT * DH];
  __shared__ __attribute__((aligned(16))) bf16 sv[2][FL_KT * DH];

  // kv heads fastest: with 8 of them a head's K and V stay in one XCD's L2.  Later rows have more keys: first.
  const int G = Hq / Hkv;
  const int kvh = blockIdx.x % Hkv, tile = gridDim.y - 1 - blockIdx.y;
  const int s = tiles[2 * tile], r0 = tiles[2 * tile + 1];
  const int qbeg = cu_q[s], qlen = cu_q[s + 1] - qbeg;
  const int L = ctx_lens[s], pos0 = L - qlen;
  const int* bt = block_tables + (long)s * max_blocks;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lq = lane & 31, lh = lane >> 5;
  const int h = kvh * G + (blockIdx.x / Hkv) * HPW + (wave >> 1);
  const int w0 = r0 + 32 * (wave & 1);       // the wave's first row
  const int kend = min(L, pos0 + min(qlen, r0 + FL_QT));
  // a row past the prompt's end repeats the last one (not stored)
  const int row = min(w0 + lq, qlen - 1);
  const int qpos = pos0 + row;
  const int qfirst = pos0 + min(w0, qlen - 1), qlast = pos0 + min(w0 + 31, qlen - 1);

  bf16x8 qf[KS];
#pragma unroll
  for (int c = 0; c < KS; ++c)
    qf[c] = *(const bf16x8*)(q + ((long)(qbeg + row) * Hq + h) * DH + 16 * c + 8 * lh);

  f32x16 o[ND];
#pragma unroll
  for (int i = 0; i < ND; ++i)
#pragma unroll
    for (int j = 0; j < 16; ++j) o[i][j] = 0.f;
  float m = -INFINITY, l = 0.f;

  const long page = (long)Hkv << bs_shift;   // K rows (and V rows) of a page over all kv heads
  // K unit u: key u / CH, chunk u % CH; V unit u: key group u / DH, d = u % DH.  64 units lie in one 16-key run,
  // which is contiguous in K's and in V's page alike.
  int blk[NU];
  auto pages = [&](int k0) {
#pragma unroll
    for (int j = 0; j < NU; ++j) {
      const int run = __builtin_amdgcn_readfirstlane((tid + j * NT) / (16 * CH));
      blk[j] = bt[min(k0 + 16 * run, kend - 1) >> bs_shift];
    }
  };
  bf16x8 rk[NU], rv[NU];
  auto load_tile = [&](int k0) {
#pragma unroll
    for (int j = 0; j < NU; ++j) {
      const int u = tid + j * NT;
      const int run = __builtin_amdgcn_readfirstlane(u / (16 * CH));
      const int off = min(k0 + 16 * run, (kend - 1) & ~15) & ((1 << bs_shift) - 1);
      const long at = ((long)blk[j] * page + ((long)kvh << bs_shift) + off) * DH + (u - run * 16 * CH) * 8;
      rk[j] = *(const bf16x8*)(kc + at);
      rv[j] = *(const bf16x8*)(vc + at);
    }
  };
  auto store_tile = [&](int k0, int buf) {
#pragma unroll
    for (int j = 0; j < NU; ++j) {
      const int u = tid + j * NT;
      const int key = u / CH, c = u % CH;
      *(bf16x8*)(sk[buf] + key * DH + (c ^ (flash_key(key & 31) & (CH - 1) & 15)) * 8) = rk[j];
      bf16x8 v = rv[j];
      if (k0 + FL_KT > kend) {               // a masked key's weight is 0: its V must not be an infinity or a NaN
        const int k = k0 + 8 * (u / DH);
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (k + i >= kend) v[i] = (bf16)0.f;
      }
      *(bf16x8*)(sv[buf] + (long)u * 8) = v;
    }
  };

  // this workgroup's keys: all, or an equal share of the tiles
  const int share = SPLIT ? ((kend + FL_KT - 1) / FL_KT + (int)gridDim.z - 1) / (int)gridDim.z * FL_KT : 0;
  const int kbeg = SPLIT ? (int)blockIdx.z * share : 0, klim = SPLIT ? min(kend, kbeg + share) : kend;
  pages(kbeg);
  load_tile(kbeg);
  pages(kbeg + FL_KT);
  store_tile(kbeg, 0);
  __syncthreads();
  for (int k0 = kbeg, buf = 0; k0 < klim; k0 += FL_KT, buf ^= 1) {
    if (k0 + FL_KT < klim) load_tile(k0 + FL_KT);
    pages(k0 + 2 * FL_KT);
    if (k0 <= qlast) {
      f32x16 sc[2];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        f32x16 a;
#pragma unroll
        for (int i = 0; i < 16; ++i) a[i] = 0.f;
        const bf16* krow = sk[buf] + (32 * b + flash_key(lq)) * DH;
#pragma unroll
        for (int c = 0; c < KS; ++c) {
          const bf16x8 kf = *(const bf16x8*)(krow + (((2 * c + lh) ^ (lq & (CH - 1) & 15)) * 8));
          a = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[c], a, 0, 0, 0);
        }
        sc[b] = a;
      }
      if (k0 + FL_KT - 1 > qfirst) {         // the tile reaches past some row's own position
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int key = k0 + 32 * b + 16 * (i >> 3) + 8 * lh + (i & 7);
            if (key > qpos) sc[b][i] = -INFINITY;
          }
      }
      float mx = -INFINITY;
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, sc[b][i]);
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64)) * sl2;
      const float mnew = fmaxf(m, mx);
      const float ms = mnew == -INFINITY ? 0.f : mnew;
      if (__any(mnew > m)) {                 // once a row's maximum stands, nothing is rescaled
        const float alpha = exp2f(m - ms);
        l *= alpha;
#pragma unroll
        for (int i = 0; i < ND; ++i)
#pragma unroll
          for (int j = 0; j < 16; ++j) o[i][j] *= alpha;
        m = mnew;
      }
      bf16x8 pf[4];
      float sum[2] = {0.f, 0.f};
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float e = __builtin_amdgcn_exp2f(fmaf(sc[b][i], sl2, -ms));
          sum[b] += e;
          pf[2 * b + (i >> 3)][i & 7] = (bf16)e;
        }
      l += sum[0] + sum[1];
#pragma unroll
      for (int kk = 0; kk < FL_KT / 16; ++kk)
#pragma unroll
        for (int nd = 0; nd < ND; ++nd) {
          const bf16x8 vf = *(const bf16x8*)(sv[buf] + ((2 * kk + lh) * DH + 32 * nd + lq) * 8);
          o[nd] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf[kk], o[nd], 0, 0, 0);
        }
    }
    if (k0 + FL_KT < klim) store_tile(k0 + FL_KT, buf ^ 1);
    __syncthreads();
  }

  l += __shfl_xor(l, 32, 64);
  if (w0 + lq >= qlen) return;
  if constexpr (SPLIT) {
    const long at = ((long)blockIdx.z * sp.T + qbeg + row) * Hq + h;
    if (lh == 0) sp.ml[at] = float2{m, l};
    if (m == -INFINITY) return;               // none of its keys: nobody reads the sums
#pragma unroll
    for (int nd = 0; nd < ND; ++nd)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *(float4*)(sp.o + at * DH + 32 * nd + 8 * j + 4 * lh) =
            float4{o[nd][4 * j], o[nd][4 * j + 1], o[nd][4 * j + 2], o[nd][4 * j + 3]};
    return;
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  bf16* orow = out + ((long)(qbeg + row) * Hq + h) * DH;
#pragma unroll
  for (int nd = 0; nd < ND; ++nd)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      bf16x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = (bf16)(o[nd][4 * j + i] * inv);
      *(bf16x4*)(orow + 32 * nd + 8 * j + 4 * lh) = v;
    }
}

// out row = sum_p o_p exp2(m_p - m) / sum_p l_p exp2(m_p - m).  A workgroup per head and 256 / (DH / 4) rows of a work tile;
// the loads of eight partials in flight (one after the other it took longer than the shares).
template <int DH>
__global__ __launch_bounds__(256) void flash_merge_kernel(FlashSplit sp, int P, const int* __restrict__ tiles,
                                                          const int* __restrict__ cu_q, int Hq, bf16* __restrict__ out) {
  constexpr int L4 = DH / 4, RP = 256 / L4;    // threads of a row, rows of a workgroup
  const int s = tiles[2 * blockIdx.y], h = blockIdx.x;
  const int r = tiles[2 * blockIdx.y + 1] + blockIdx.z * RP + threadIdx.x / L4;
  const int qbeg = cu_q[s], qlen = cu_q[s + 1] - qbeg;
  const int d = threadIdx.x % L4 * 4;
  if (r >= qlen) return;
  const long at = (long)(qbeg + r) * Hq + h, step = (long)sp.T * Hq;
  float m = -INFINITY, l = 0.f;
  float4 a = {0.f, 0.f, 0.f, 0.f};
  for (int p0 = 0; p0 < P; p0 += 8) {
    float2 v[8];
    float4 x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const long k = at + min(p0 + i, P - 1) * step;
      v[i] = sp.ml[k];
      x[i] = *(const float4*)(sp.o + k * DH + d);
    }
    float mn = m;
#pragma unroll
    for (int i = 0; i < 8; ++i) mn = p0 + i < P ? fmaxf(mn, v[i].x) : mn;
    const float w0 = m == -INFINITY ? 0.f : exp2f(m - mn);
    l *= w0, a.x *= w0, a.y *= w0, a.z *= w0, a.w *= w0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (p0 + i >= P || v[i].x == -INFINITY) continue;   // a share without keys wrote no sums
      const float w = exp2f(v[i].x - mn);
      l += v[i].y * w;
      a.x += x[i].x * w, a.y += x[i].y * w, a.z += x[i].z * w, a.w += x[i].w * w;
    }
    m = mn;
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  *(bf16x4*)(out + at * DH + d) = bf16x4{(bf16)(a.x * inv), (bf16)(a.y * inv), (bf16)(a.z * inv), (bf16)(a.w * inv)};
}

}  // namespace la
