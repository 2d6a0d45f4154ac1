// Multi-row products and causal attention of the decoder (prefill, replay,
// all-row forward) on operands kept in MFMA fragment order (frag.h).
//
// y[M][N] = x[M][K] Wdeq^T + bias contracts fp16 hi/lo activation fragments (~22 bits) with
// the codes, exact in fp16 as q - 128 (8-bit) or q - 8 (4-bit), two products on
// v_mfma_f32_32x32x16_f16 per K step, and folds each 64-group's scale into an fp32
// accumulator: acc += s[g, n] P.  The groups' bias term, sum_g b'[n, g] sum_{k in g} x[m, k]
// with b' = b + 128 s (or 8 s), is itself a product over G more K values, of bf16 triples: the
// activation planes carry the groups' sums as further K steps, the weights' b' planes hold the
// other operand.  Triples keep both as the fp32 values they are, over fp32's range: as fp16
// pairs, sums past 8188 an element lost bits and sums past 16376 overflowed.
//
// Activation planes ("rows"): per 32-row block, K / 16 steps of fp16 pairs, then ceil(G / 16)
// steps of group sums.  Inside a 64-group the K order is permuted so that a lane's codes of two
// steps are one contiguous read: chunk c8 (8 values) is half (c8 >> 1) & 1 of step 2 (c8 >> 2) +
// (c8 & 1).
// The codes are held a second time in that order (per 32 columns and group, two 32-value
// halves of 64 lanes x 16 codes): a fragment load is then one coalesced run, where the
// row-major codes touch 32 rows (886 x 5120 x 1280: 32.7 against 46.7 us).
#include "frag.h"
#include "kernels.h"

namespace itts {

namespace {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

// pieces of a row block: nk steps of K, nx of group sums
__host__ __device__ inline size_t rows_block(int nk, int nx) { return (size_t)nk * 128 + (size_t)nx * 192; }
__device__ __forceinline__ size_t rows_block_of(int d) { return rows_block(d / 16, (d / 64 + 15) / 16); }
// piece of (row, chunk c of K): hi plane; lo 64 pieces on.  rb: rows_block of the planes.
__device__ __forceinline__ size_t rows_piece(int row, int c, size_t rb) {
  const int step = (c >> 3) * 4 + ((c >> 2) & 1) * 2 + (c & 1);
  return (row >> 5) * rb + (size_t)(step * 128 + ((c >> 1) & 1) * 32 + (row & 31));
}
// piece of (row, chunk g8 of groups) of rb pieces a block whose group steps start at piece at; plane 0 of three
__device__ __forceinline__ size_t group_piece(int row, int g8, size_t rb, int at) {
  return (row >> 5) * rb + (size_t)(at + (g8 >> 1) * 192 + (g8 & 1) * 32 + (row & 31));
}
// group g's sum v: element of the group steps
__device__ __forceinline__ void put_group_sum(u32x4 *o, int row, int g, int nk, size_t rb, float v) {
  __bf16 *p = reinterpret_cast<__bf16 *>(o + group_piece(row, g >> 3, rb, nk * 128)) + (g & 7);
#pragma unroll
  for (int i = 0; i < 3; i++) {
    const __bf16 h = (__bf16)v;
    p[i * 64 * 8] = h;
    v -= (float)h;
  }
}

__device__ __forceinline__ float sum8(float v) {  // over eight consecutive lanes
  v += dpp_pair<0xB1>(v);
  v += dpp_pair<0x4E>(v);
  return v + dpp_pair<0x141>(v);
}

// LayerNorm of M rows (a second one with w2; none without w) as planes and group sums.  Half a
// wave a row (lane c of it: chunks c, c + 32, ..); the row in NC chunks of registers, loaded with
// its parameters in one memory round trip, or any d with NC = 0 (read again for each pass).
// Bound by latency: 886 x 1280 6.1 us (7.3 with a quarter of a wave a row, 12 with a row a
// wave, read again for each pass).
template <int NC>
__global__ __launch_bounds__(64) void ln_planes_kernel(const float *x, const float *w, const float *b, const float *w2,
                                                       const float *b2, int M, int d, u32x4 *out) {
  constexpr int ND = NC ? NC : 1;
  const int lane = threadIdx.x, c = lane & 31, row = blockIdx.x * 2 + (lane >> 5);
  const int nc = d / 8, nk = d / 16, nj = (nc + 31) / 32;
  const size_t rb = rows_block_of(d);
  const float *xr = x + (size_t)min(row, M - 1) * d;
  float v[ND][8], g[ND][8], h[ND][8];  // the row and its LayerNorm's parameters
  auto load8 = [&](const float *p, float (&o)[8]) __attribute__((always_inline)) {
    const float4 a = reinterpret_cast<const float4 *>(p)[0], e = reinterpret_cast<const float4 *>(p)[1];
    o[0] = a.x, o[1] = a.y, o[2] = a.z, o[3] = a.w, o[4] = e.x, o[5] = e.y, o[6] = e.z, o[7] = e.w;
  };
  auto params = [&](const float *gw, const float *gb, int k, int i) __attribute__((always_inline)) {
    load8(gw + k * 8, g[i]);
    load8(gb + k * 8, h[i]);
  };
  float m1 = 0.0f, r1 = 1.0f, m2 = 0.0f, r2 = 1.0f;
  int done = 0;  // LayerNorms applied to v
  auto norm = [&](float (&y)[8], int i, float m, float r) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 8; e++) y[e] = (y[e] - m) * r * g[i][e] + h[i][e];
  };
  // f(chunk, register index, live) over the lane's chunks; chunks past the row repeat its last one
  auto each = [&](auto f) __attribute__((always_inline)) {
    if constexpr (NC > 0) {
#pragma unroll
      for (int j = 0; j < NC; j++) f(min(c + 32 * j, nc - 1), j, c + 32 * j < nc);
    } else {
      for (int j = 0; j < nj; j++) {
        const int k = min(c + 32 * j, nc - 1);
        load8(xr + k * 8, v[0]);
        if (done > 0) {
          params(w, b, k, 0);
          norm(v[0], 0, m1, r1);
        }
        if (done > 1) {
          params(w2, b2, k, 0);
          norm(v[0], 0, m2, r2);
        }
        f(k, 0, c + 32 * j < nc);
      }
    }
  };
  auto stats = [&](float &mean, float &rstd) __attribute__((always_inline)) {
    float s = 0.0f, q = 0.0f;
    each([&](int, int i, bool live) __attribute__((always_inline)) {
      const float t = ((v[i][0] + v[i][1]) + (v[i][2] + v[i][3])) + ((v[i][4] + v[i][5]) + (v[i][6] + v[i][7]));
      s += live ? t : 0.0f;
    });
    mean = half32_sum(s) / (float)d;
    each([&](int, int i, bool live) __attribute__((always_inline)) {
      float t = 0.0f;
#pragma unroll
      for (int e = 0; e < 8; e++) t += (v[i][e] - mean) * (v[i][e] - mean);
      q += live ? t : 0.0f;
    });
    rstd = 1.0f / sqrtf(half32_sum(q) / (float)d + 1e-5f);
  };
  if constexpr (NC > 0) {
    each([&](int k, int i, bool) __attribute__((always_inline)) {
      load8(xr + k * 8, v[i]);
      if (w) params(w, b, k, i);
    });
  }
  if (w) {
    stats(m1, r1);
    if constexpr (NC > 0) {
      each([&](int k, int i, bool) __attribute__((always_inline)) {
        norm(v[i], i, m1, r1);
        if (w2) params(w2, b2, k, i);
      });
    }
    done = 1;
  }
  if (w2) {
    stats(m2, r2);
    if constexpr (NC > 0) {
      each([&](int, int i, bool) __attribute__((always_inline)) { norm(v[i], i, m2, r2); });
    }
    done = 2;
  }
  each([&](int k, int i, bool live) __attribute__((always_inline)) {
    const float t = ((v[i][0] + v[i][1]) + (v[i][2] + v[i][3])) + ((v[i][4] + v[i][5]) + (v[i][6] + v[i][7]));
    const float gs = sum8(t);
    if (!live || row >= M) return;
    u32x4 hi, lo;
    split8(v[i], hi, lo);
    const size_t p = rows_piece(row, k, rb);
    out[p] = hi;
    out[p + 64] = lo;
    if ((k & 7) == 0) put_group_sum(out, row, k >> 3, nk, rb, gs);
  });
}

// ---- weights ----------------------------------------------------------------------------
// scale [G][ldn] fp32 and the (scale, bias) words transposed alike (columns past N zero), and b' =
// b + off s as the group steps' planes
template <int PT>
__global__ __launch_bounds__(256) void rows_params_kernel(const void *params, int N, int G, int ldn, float off,
                                                          float *scale, u32x4 *bw, void *words) {
  const int nx = (G + 15) / 16;
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long)ldn * nx * 2) return;
  const int n = (int)(i % ldn), g8 = (int)(i / ldn);
  float v[8];
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const int g = g8 * 8 + j;
    float2 sb = make_float2(0.0f, 0.0f);
    if (n < N && g < G) sb = load_param<PT>(params, (size_t)n * G + g);
    if (g < G) {
      const size_t i = (size_t)g * ldn + n;
      scale[i] = sb.x;
      if constexpr (PT == kParamF32) static_cast<float2 *>(words)[i] = sb;
      else static_cast<uint32_t *>(words)[i] = n < N ? static_cast<const uint32_t *>(params)[(size_t)n * G + g] : 0u;
    }
    v[j] = fmaf(off, sb.x, sb.y);
  }
  u32x4 pl[3];
  split8_bf16(v, pl);
  const size_t p = group_piece(n, g8, rows_block(0, nx), 0);
#pragma unroll
  for (int k = 0; k < 3; k++) bw[p + k * 64] = pl[k];
}

// codes in fragment order: lane's 16 codes (BITS * 2 bytes) of (32 columns, group, half), zero past N
template <int BITS>
__global__ __launch_bounds__(256) void rows_codes_kernel(const uint8_t *codes, int N, int K, long n, uint8_t *out) {
  constexpr int B = BITS * 2;
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int lane = (int)(i & 63), kp = (int)((i >> 6) & 1), G = K / 64;
  const long r = i >> 7;
  const int g = (int)(r % G), col = (int)(r / G) * 32 + (lane & 31);
  uint32_t w[B / 4];
#pragma unroll
  for (int j = 0; j < B / 4; j++) w[j] = 0u;
  if (col < N) {
    const uint32_t *p = reinterpret_cast<const uint32_t *>(codes + (size_t)col * (K * BITS / 8) + g * (BITS * 8) +
                                                           kp * (BITS * 4) + (lane >> 5) * B);
#pragma unroll
    for (int j = 0; j < B / 4; j++) w[j] = p[j];
  }
  uint32_t *o = reinterpret_cast<uint32_t *>(out + (size_t)i * B);
#pragma unroll
  for (int j = 0; j < B / 4; j++) o[j] = w[j];
}

// ---- the product ------------------------------------------------------------------------
// Block: one tile of BM = 32 TM rows x 64 columns by KS waves that split the K groups, their
// partial tiles added through LDS (two halves of the waves at a time).  A wave keeps a
// group of activation fragments, codes and scales in flight.
constexpr int kMaxSplit = 6;  // blocks that may share a tile's K
template <int TM_, int KS_>
struct RmCfg {
  static constexpr int TM = TM_, TN = 2, KS = KS_;
  static constexpr int BM = 32 * TM, BN = 64, LD = BN + 4, NT = 64 * KS, KL = KS > 2 ? KS / 2 : KS;
  static constexpr size_t LDS = sizeof(float) * (KL * BM * LD + 2 * BM);
  static_assert(LDS <= 65536, "dynamic LDS of a plain launch");
};

// eight 8-bit codes (two words) or 4-bit codes (one word) as fp16 q - 128 / q - 8
template <int BITS>
__device__ __forceinline__ f16x8 codes_f16(uint32_t w0, uint32_t w1) {
  u32x4 r;
  if constexpr (BITS == 8) {
    // bytes q and 0x64 make the half 1024 + q
    r[0] = __builtin_amdgcn_perm(0x64646464u, w0, 0x04010400u);
    r[1] = __builtin_amdgcn_perm(0x64646464u, w0, 0x04030402u);
    r[2] = __builtin_amdgcn_perm(0x64646464u, w1, 0x04010400u);
    r[3] = __builtin_amdgcn_perm(0x64646464u, w1, 0x04030402u);
  } else {
    const uint32_t e = w0 & 0x0f0f0f0fu, o = (w0 >> 4) & 0x0f0f0f0fu;
    r[0] = __builtin_amdgcn_perm(o, e, 0x0c040c00u) | 0x64006400u;
    r[1] = __builtin_amdgcn_perm(o, e, 0x0c050c01u) | 0x64006400u;
    r[2] = __builtin_amdgcn_perm(o, e, 0x0c060c02u) | 0x64006400u;
    r[3] = __builtin_amdgcn_perm(o, e, 0x0c070c03u) | 0x64006400u;
  }
  const _Float16 z = BITS == 8 ? (_Float16)1152.0f : (_Float16)1032.0f;
  const f16x2 zz = {z, z};
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const uint32_t w = r[i];  // (a bit cast of a vector's element reads its first)
    r[i] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, w) - zz);
  }
  return __builtin_bit_cast(f16x8, r);
}

// The attention's operands by the rows' type: q and the probabilities in T's planes, K and V in
// NP.  bf16 rows are their own single plane, so nothing of q, K, V or the probabilities is
// rounded and no magnitude is out of range; fp32 rows the same in three planes, or as pairs.
template <int KVT>
struct AttnPlanes {
  typedef Bf16Triples T;
  static constexpr int NP = KVT == kKvBf16 ? 1 : 3;
};
template <>
struct AttnPlanes<kRowsPairs> {
  typedef F16Pairs T;
  static constexpr int NP = 2;
};

template <int BITS, int EPI, int KVT, class C>
__global__ __launch_bounds__(C::NT, C::NT <= 256 ? 2 : 1) void rows_mm_kernel(RowsMm a) {
  constexpr int TM = C::TM, TN = C::TN, KS = C::KS, KL = C::KL, BM = C::BM, BN = C::BN, LD = C::LD, NT = C::NT;
  constexpr int CW = BITS == 8 ? 4 : 2;  // words of a lane's codes per 32 K values
  extern __shared__ __attribute__((aligned(16))) float red[];
  float2 *row_stat = reinterpret_cast<float2 *>(red + KL * BM * LD);
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, r31 = lane & 31;
  const int kq = __builtin_amdgcn_readfirstlane(tid >> 6);
  // block -> tile: XCD x takes every gm-th row tile and every gn-th column tile
  const int gn = 8 / a.gm, x = blockIdx.x & 7, pn = (a.nN + gn - 1) / gn, per = pn * ((a.nM + a.gm - 1) / a.gm);
  const int jb = (blockIdx.x >> 3) % per, split = (blockIdx.x >> 3) / per;  // split: part of K (a.S of them)
  const int tm = jb / pn * a.gm + x % a.gm, tn = jb % pn * gn + x / a.gm;
  if (tm >= a.nM || tn >= a.nN) return;
  const int m0 = tm * BM, n0 = tn * BN;
  const int G = a.K / 64, nk = a.K / 16, nx = (G + 15) / 16, rb = (int)rows_block(nk, nx);
  const int kk = split * KS + kq, KT = KS * a.S;
  const int g0 = G * kk / KT, g1 = G * (kk + 1) / KT;

  // wave-uniform bases with 32-bit lane offsets (registers, not 64-bit addresses, are short here)
  const u32x4 *ab = reinterpret_cast<const u32x4 *>(a.x) + (size_t)(m0 >> 5) * rb;
  const uint8_t *cb = reinterpret_cast<const uint8_t *>(a.codes) + (size_t)(n0 >> 5) * G * (BITS * 256);

  floatx16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[i][j][e] = 0.0f;

  struct Codes {
    uint32_t q[TN][2][CW];
    float s[TN];
  };
  u32x4 fa[4][TM][2];
  Codes cq;
  auto load_a = [&](int g, int s4, u32x4(&f)[TM][2]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TM; i++) {
      const u32x4 *p = ab + (size_t)i * rb + (min(g, g1 - 1) * 4 + s4) * 128;
      f[i][0] = p[lane];
      f[i][1] = p[lane + 64];
    }
  };
  auto load_c = [&](int g, Codes &c) __attribute__((always_inline)) {
    const int gc = min(g, g1 - 1);
#pragma unroll
    for (int j = 0; j < TN; j++) {
#pragma unroll
      for (int kp = 0; kp < 2; kp++) {
        const uint8_t *p = cb + (((size_t)j * G + gc) * 2 + kp) * (BITS * 128) + lane * (BITS * 2);
        if constexpr (BITS == 8) {
          const u32x4 v = *reinterpret_cast<const u32x4 *>(p);
#pragma unroll
          for (int w = 0; w < 4; w++) c.q[j][kp][w] = v[w];
        } else {
          const u32x2 v = *reinterpret_cast<const u32x2 *>(p);
#pragma unroll
          for (int w = 0; w < 2; w++) c.q[j][kp][w] = v[w];
        }
      }
      c.s[j] = (a.scale + (size_t)gc * a.ldn + n0 + j * 32)[r31];
    }
  };
  auto load_group = [&](int g) __attribute__((always_inline)) {
    load_c(g, cq);
#pragma unroll
    for (int s4 = 0; s4 < 4; s4++) load_a(g, s4, fa[s4]);
  };
  // the bias term's steps first (their loads go out ahead of the first group's)
  const int x0 = nx * kk / KT, x1 = nx * (kk + 1) / KT;
  for (int kx = x0; kx < x1; kx++) {
    u32x4 xa[TM][3], xb[TN][3];
#pragma unroll
    for (int i = 0; i < TM; i++) {
      const u32x4 *p = ab + (size_t)i * rb + nk * 128 + kx * 192;
#pragma unroll
      for (int q = 0; q < 3; q++) xa[i][q] = p[lane + 64 * q];
    }
#pragma unroll
    for (int j = 0; j < TN; j++) {
      const u32x4 *p = reinterpret_cast<const u32x4 *>(a.bw) + ((size_t)((n0 >> 5) + j) * nx + kx) * 192;
#pragma unroll
      for (int q = 0; q < 3; q++) xb[j][q] = p[lane + 64 * q];
    }
    if (kx == x0 && g0 < g1) {
      load_group(g0);
    }
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++) acc[i][j] = mma_planes<Bf16Triples, 3>(xa[i], xb[j], acc[i][j]);
  }
  if (x0 == x1 && g0 < g1) {
    load_group(g0);
  }
  // What the epilogue needs, loaded here so that its latency passes under the K loop.  A
  // thread's items are the tile's rows tid / 8 + i NT / 8 at columns 8 (tid & 7) .. +7.
  // Folded LayerNorm input: LPR lanes a row hold its groups' (mean, sum of squared
  // deviations), combined after the loop.
  constexpr bool kFold = EPI == kEpiQKV || EPI == kEpiGelu;
  constexpr int LPR = NT / BM, SG = 32 / LPR, IT = (BM * 8 + NT - 1) / NT;
  const bool fin = kFold && a.st != nullptr;
  const int ic = n0 + (tid & 7) * 8;
  float2 sv[kFold ? SG : 1];
  if constexpr (kFold) {
    const float2 *st = a.st + (size_t)min(m0 + tid / LPR, a.M - 1) * G;
#pragma unroll
    for (int i = 0; i < SG; i++) {
      const int gg = tid % LPR + i * LPR;
      sv[i] = fin && gg < G ? st[gg] : make_float2(0.0f, 0.0f);
    }
  }
  float cadd[8], cG[kFold ? 8 : 1], gam[EPI == kEpiResid ? 8 : 1];
  float4 old[EPI == kEpiResid ? IT : 1][2];
#pragma unroll
  for (int e = 0; e < 8; e++) {
    const int n = min(ic + e, a.N - 1);
    cadd[e] = (fin ? a.fc : a.bias)[n];
    if constexpr (kFold) cG[e] = fin ? a.fG[n] : 0.0f;
    if constexpr (EPI == kEpiResid) gam[e] = a.o ? a.gamma[n] : 0.0f;
  }
  if constexpr (EPI == kEpiResid) {
#pragma unroll
    for (int i = 0; i < IT; i++) {
      const float4 *o = reinterpret_cast<const float4 *>(a.y + (size_t)min(m0 + min((tid >> 3) + i * (NT / 8), BM - 1), a.M - 1) * a.N + ic);
      old[i][0] = o[0];
      old[i][1] = o[1];
    }
  }
  auto group = [&](int g) __attribute__((always_inline)) {
    floatx16 P[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int e = 0; e < 16; e++) P[i][j][e] = 0.0f;
#pragma unroll
    for (int s4 = 0; s4 < 4; s4++) {
      f16x8 b[TN];
#pragma unroll
      for (int j = 0; j < TN; j++) {
        const uint32_t *q = cq.q[j][s4 >> 1];
        b[j] = BITS == 8 ? codes_f16<BITS>(q[(s4 & 1) * 2], q[(s4 & 1) * 2 + (BITS == 8 ? 1 : 0)])
                         : codes_f16<BITS>(q[s4 & 1], 0);
      }
#pragma unroll
      for (int p = 0; p < 2; p++)
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int j = 0; j < TN; j++) P[i][j] = ITTS_MFMA16(__builtin_bit_cast(f16x8, fa[s4][i][p]), b[j], P[i][j], 0, 0, 0);
      load_a(g + 1, s4, fa[s4]);
    }
#pragma unroll
    for (int j = 0; j < TN; j++) {
      const float s = cq.s[j];
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[i][j][e] = fmaf(s, P[i][j][e], acc[i][j][e]);
    }
    load_c(g + 1, cq);
  };
  for (int g = g0; g < g1; g++) group(g);

  if constexpr (kFold) {
    if (fin) {
      auto lanes_sum = [&](float v) __attribute__((always_inline)) {
        v += dpp_pair<0xB1>(v);
        v += dpp_pair<0x4E>(v);
        if constexpr (LPR >= 8) v += dpp_pair<0x141>(v);
        if constexpr (LPR >= 16) v += dpp_pair<0x140>(v);
        return v;
      };
      float sm = 0.0f;
#pragma unroll
      for (int i = 0; i < SG; i++) sm += sv[i].x;
      const float mean = lanes_sum(sm) / (float)G;
      float m2 = 0.0f;
#pragma unroll
      for (int i = 0; i < SG; i++)
        if (tid % LPR + i * LPR < G) m2 += sv[i].y + 64.0f * ((sv[i].x - mean) * (sv[i].x - mean));
      m2 = lanes_sum(m2);
      if (tid % LPR == 0) row_stat[tid / LPR] = make_float2(mean, 1.0f / sqrtf(m2 / (float)a.K + 1e-5f));
    }
  }
  parts_to_lds<TM, TN, KS, KL, BM, LD>(red, acc, kq, h, r31);

  // eight columns of a tile row: the parts added, then the folded LayerNorm or the bias
  auto tile8 = [&](int row, int col, float v[8]) __attribute__((always_inline)) {
    parts_row8<KL, BM, LD>(red, row, col, v);
    if constexpr (kFold) {
      if (fin) {
        const float2 rs = row_stat[row];
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = rs.y * (v[e] - rs.x * cG[e]);
      }
    }
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] += cadd[e];
  };
  // K over a.S blocks (residual products): each stores its partial tile through agent-scope
  // accesses (coherent across the XCDs' L2s); the last to arrive (wrapping counter) adds the
  // others' in split order, so the result does not depend on arrival.
  __shared__ uint32_t last_flag;
  float4 sum[EPI == kEpiResid ? IT : 1][2];
  if constexpr (EPI == kEpiResid) {
    if (a.S > 1) {
      const int tile = tm * a.nN + tn;
      uint64_t *ws = reinterpret_cast<uint64_t *>(a.ws + (size_t)tile * a.S * (BM * 64));
      auto raw = [&](int q, float4(&o)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int w = 0; w < 2; w++) {
          const float *p = red + (size_t)(q >> 3) * LD + (q & 7) * 8 + 4 * w;
          float4 t = *reinterpret_cast<const float4 *>(p);
#pragma unroll
          for (int k = 1; k < KL; k++) {
            const float4 u = *reinterpret_cast<const float4 *>(p + (size_t)k * BM * LD);
            t.x += u.x, t.y += u.y, t.z += u.z, t.w += u.w;
          }
          o[w] = t;
        }
      };
      // word w of item q: [split][w][q], consecutive lanes on consecutive words
      constexpr int ITEMS_ = BM * 8;
#pragma unroll
      for (int i = 0; i < IT; i++) {
        const int q = tid + i * NT;
        if (q >= ITEMS_) break;
        raw(q, sum[i]);
        const float f[8] = {sum[i][0].x, sum[i][0].y, sum[i][0].z, sum[i][0].w,
                            sum[i][1].x, sum[i][1].y, sum[i][1].z, sum[i][1].w};
#pragma unroll
        for (int w = 0; w < 4; w++)
          __hip_atomic_store(ws + ((size_t)split * 4 + w) * ITEMS_ + q,
                             __builtin_bit_cast(uint64_t, make_float2(f[2 * w], f[2 * w + 1])), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (tid == 0) last_flag = atomicInc(a.cnt + tile, (uint32_t)(a.S - 1)) == (uint32_t)(a.S - 1) ? 1u : 0u;
      __syncthreads();
      if (!last_flag) return;
#pragma unroll
      for (int i = 0; i < IT; i++) {
        const int q = tid + i * NT;
        if (q >= ITEMS_) break;
        float2 p[kMaxSplit][4];
#pragma unroll
        for (int s2 = 0; s2 < kMaxSplit; s2++)
#pragma unroll
          for (int w = 0; w < 4; w++)
            p[s2][w] = s2 < a.S ? __builtin_bit_cast(float2, __hip_atomic_load(ws + ((size_t)s2 * 4 + w) * ITEMS_ + q,
                                                                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                                : make_float2(0.0f, 0.0f);
        float2 t[4];
#pragma unroll
        for (int w = 0; w < 4; w++) {
          t[w] = p[0][w];
#pragma unroll
          for (int s2 = 1; s2 < kMaxSplit; s2++)
            if (s2 < a.S) t[w].x += p[s2][w].x, t[w].y += p[s2][w].y;
        }
        sum[i][0] = make_float4(t[0].x, t[0].y, t[1].x, t[1].y);
        sum[i][1] = make_float4(t[2].x, t[2].y, t[3].x, t[3].y);
      }
    }
  }
  constexpr int ITEMS = BM * 8;
  if constexpr (EPI == kEpiStore) {
    for (int q = tid; q < ITEMS; q += NT) {
      const int c = q & 7, row = q >> 3, r = m0 + row, n = n0 + c * 8;
      if (r >= a.M || n >= a.N) continue;
      float v[8];
      tile8(row, c * 8, v);
      float *o = a.y + (size_t)r * a.N + n;
      if (a.N % 4 == 0 && n + 8 <= a.N) {
        reinterpret_cast<float4 *>(o)[0] = make_float4(v[0], v[1], v[2], v[3]);
        reinterpret_cast<float4 *>(o)[1] = make_float4(v[4], v[5], v[6], v[7]);
      } else {
        for (int e = 0; e < 8 && n + e < a.N; e++) o[e] = v[e];
      }
    }
  } else if constexpr (EPI == kEpiResid) {
    // x = y + v; with the fold-out, gamma x as planes, its group sum, and the group's mean and
    // sum of squared deviations (eight lanes hold a row's 64 columns)
#pragma unroll
    for (int i = 0; i < IT; i++) {
      const int q = tid + i * NT, c = q & 7, row = q >> 3, r = m0 + row, n = n0 + c * 8;
      if (q >= ITEMS) break;  // whole waves
      const bool live = r < a.M;
      float v[8];
      if (a.S > 1) {
        const float4 t0 = sum[i][0], t1 = sum[i][1];
        const float f[8] = {t0.x, t0.y, t0.z, t0.w, t1.x, t1.y, t1.z, t1.w};
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = f[e] + cadd[e];
      } else {
        tile8(row, c * 8, v);
      }
      float4 *o = reinterpret_cast<float4 *>(a.y + (size_t)min(r, a.M - 1) * a.N + n);
      const float4 p = old[i][0], t = old[i][1];
      const float yv[8] = {p.x, p.y, p.z, p.w, t.x, t.y, t.z, t.w};
#pragma unroll
      for (int e = 0; e < 8; e++) v[e] += yv[e];
      if (live) {
        o[0] = make_float4(v[0], v[1], v[2], v[3]);
        o[1] = make_float4(v[4], v[5], v[6], v[7]);
      }
      if (!a.o) continue;
      const float mean = sum8(((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]))) / 64.0f;
      float m2 = 0.0f, gs = 0.0f, y[8];
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const float d = v[e] - mean;
        m2 += d * d;
        y[e] = gam[e] * v[e];
        gs += y[e];
      }
      m2 = sum8(m2);
      gs = sum8(gs);
      if (!live) continue;
      const int onk = a.N / 16;
      const size_t orb = rows_block_of(a.N);
      u32x4 hi, lo;
      split8(y, hi, lo);
      u32x4 *out = reinterpret_cast<u32x4 *>(a.o);
      const size_t pc = rows_piece(r, n >> 3, orb);
      out[pc] = hi;
      out[pc + 64] = lo;
      if (c == 0) {
        put_group_sum(out, r, n >> 6, onk, orb, gs);
        a.so[(size_t)r * (a.N / 64) + (n >> 6)] = make_float2(mean, m2);
      }
    }
  } else if constexpr (EPI == kEpiGelu) {
    for (int q = tid; q < ITEMS; q += NT) {
      const int c = q & 7, row = q >> 3, r = m0 + row, n = n0 + c * 8;
      float v[8], gs = 0.0f;
      tile8(row, c * 8, v);
#pragma unroll
      for (int e = 0; e < 8; e++) {
        v[e] = gelu_tanh_exp(v[e]);
        gs += v[e];
      }
      gs = sum8(gs);
      if (r >= a.M) continue;
      const int onk = a.N / 16;
      const size_t orb = rows_block_of(a.N);
      u32x4 hi, lo;
      split8(v, hi, lo);
      u32x4 *out = reinterpret_cast<u32x4 *>(a.o);
      const size_t pc = rows_piece(r, n >> 3, orb);
      out[pc] = hi;
      out[pc + 64] = lo;
      if (c == 0) put_group_sum(out, r, n >> 6, onk, orb, gs);
    }
  } else {
    // the 64 columns are one head of q, k or v: the attention's fragments (q scaled by
    // log2(e) / 8; rows past M zero to the end of the 32-row tile that holds row M - 1, a tile
    // after it is not written and not read), and the cache rows
    using P = AttnPlanes<KVT>;
    constexpr int NQ = P::T::N, NP = P::NP;
    const int d = a.N / 3, which = n0 / d, head = (n0 - which * d) / 64, Tt = (a.M + 63) / 64 * 2;
    auto round_kv = [&](float v[8]) __attribute__((always_inline)) {
      if constexpr (KVT == kKvBf16) {
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = bf16_bits_to_float(float_to_bf16_bits(v[e]));
      }
    };
    u32x4 *kvf = reinterpret_cast<u32x4 *>(a.kvf) + (size_t)head * Tt * flash_tile_pieces(NP);
    for (int q = tid; q < ITEMS; q += NT) {
      const int c = q & 7, row = q >> 3, t = m0 + row;
      float v[8];
      tile8(row, c * 8, v);
      if (which == 0) {
        if (t >= Tt * 32) continue;
        if (a.q_out && t < a.M) {
          float4 *o = reinterpret_cast<float4 *>(a.q_out + (size_t)t * d + head * 64 + c * 8);
          o[0] = make_float4(v[0], v[1], v[2], v[3]);
          o[1] = make_float4(v[4], v[5], v[6], v[7]);
        }
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = t < a.M ? v[e] * (0.125f * 1.4426950408889634f) : 0.0f;
        u32x4 p[NQ];
        P::T::split(v, p);
        u32x4 *dst = reinterpret_cast<u32x4 *>(a.qf) + (((size_t)head * Tt + (t >> 5)) * 4 + (c >> 1)) * (NQ * 64) +
                     (c & 1) * 32 + (t & 31);
#pragma unroll
        for (int i = 0; i < NQ; i++) dst[i * 64] = p[i];
        continue;
      }
      round_kv(v);
      void *cache = which == 1 ? a.kc : a.vc;
      if (cache && t < a.M) {
        const size_t ci = ((size_t)head * a.max_seq + t) * 64 + c * 8;
        if constexpr (KVT == kKvBf16) {
          u32x4 w;
#pragma unroll
          for (int e = 0; e < 4; e++)
            w[e] = (__float_as_uint(v[2 * e]) >> 16) | (__float_as_uint(v[2 * e + 1]) & 0xffff0000u);
          *reinterpret_cast<u32x4 *>(static_cast<uint16_t *>(cache) + ci) = w;
        } else {
          float4 *o = reinterpret_cast<float4 *>(static_cast<float *>(cache) + ci);
          o[0] = make_float4(v[0], v[1], v[2], v[3]);
          o[1] = make_float4(v[4], v[5], v[6], v[7]);
        }
      }
      if (which == 1 && t < Tt * 32) {
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = t < a.M ? v[e] : 0.0f;
        u32x4 p[NQ];
        P::T::split(v, p);
        u32x4 *dst = kvf + (size_t)(t >> 5) * flash_tile_pieces(NP) + (c >> 1) * NP * 64 + (c & 1) * 32 + (t & 31);
#pragma unroll
        for (int i = 0; i < NP; i++) dst[i * 64] = p[i];
      }
    }
    if (which == 2) {
      // dim e, key positions 8 k8 .. +7: keys 16 s + 4 hh + {0..3, 8..11}
      // (e is the same for a thread's items)
      const float vG = fin ? a.fG[n0 + (tid & 63)] : 0.0f, vadd = (fin ? a.fc : a.bias)[n0 + (tid & 63)];
      for (int q = tid; q < ITEMS; q += NT) {
        const int e = q & 63, k8 = q >> 6, rb = (k8 >> 1) * 16 + (k8 & 1) * 4, t = m0 + rb;
        if (t >= Tt * 32) continue;
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
          const int row = rb + (j >> 2) * 8 + (j & 3);
          float s = red[(size_t)row * LD + e];
#pragma unroll
          for (int k = 1; k < KL; k++) s += red[((size_t)k * BM + row) * LD + e];
          if (fin) s = row_stat[row].y * (s - row_stat[row].x * vG);
          v[j] = s + vadd;
        }
        round_kv(v);
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = m0 + rb + (j >> 2) * 8 + (j & 3) < a.M ? v[j] : 0.0f;
        u32x4 p[NQ];
        P::T::split(v, p);
        u32x4 *dst = kvf + (size_t)(t >> 5) * flash_tile_pieces(NP) +
                     (4 + (e >> 5) * 2 + ((t >> 4) & 1)) * NP * 64 + (k8 & 1) * 32 + (e & 31);
#pragma unroll
        for (int i = 0; i < NP; i++) dst[i * 64] = p[i];
      }
    }
  }
}

// ---- causal attention -------------------------------------------------------------------
// Block: 32 query rows of one head, its four waves on a quarter of the key tiles each.  Row t
// attends to keys kstart[t] (or 0) .. t; order lists the query tiles, most keys first.
template <int KVT>
__global__ __launch_bounds__(256, 2) void rows_attn_kernel(const u32x4 *qf, const u32x4 *kvf, int M, const int *kstart,
                                                           const int *order, u32x4 *out) {
  __shared__ float buf[4 * 2112];
  const int lane = threadIdx.x & 63, g = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int head = blockIdx.x, d = gridDim.x * 64, Tt = (M + 63) / 64 * 2;
  const int qt = order ? order[blockIdx.y] : (int)(gridDim.y - 1 - blockIdx.y);
  const int t = qt * 32 + (lane & 31), tc = min(t, M - 1);
  const int ks = kstart ? kstart[tc] : 0;
  using P = AttnPlanes<KVT>;
  constexpr int NQ = P::T::N, NP = P::NP;
  u32x4 q[4][NQ];
  const u32x4 *qp = qf + (((size_t)head * Tt + qt) * 4) * (NQ * 64) + lane;
#pragma unroll
  for (int kk = 0; kk < 4; kk++)
#pragma unroll
    for (int i = 0; i < NQ; i++) q[kk][i] = qp[(kk * NQ + i) * 64];
  FlashState st;
  flash_init(st);
  const int tb = kstart ? kstart[qt * 32] / 32 : 0, nt = qt + 1 - tb;
  const int kmax = kstart ? kstart[min(qt * 32 + 31, M - 1)] : 0;
  const int per = (nt + 3) / 4, t0 = tb + g * per, t1 = min(qt + 1, t0 + per);
  auto mask = [&](int kt, floatx16 &S) __attribute__((always_inline)) {
    if (kt == qt || kt * 32 < kmax) {
#pragma unroll
      for (int i = 0; i < 16; i++) {
        const int key = kt * 32 + (i >> 2) * 8 + (lane >> 5) * 4 + (i & 3);
        if (key > tc || key < ks) S[i] = -INFINITY;
      }
    }
  };
  flash_tiles<typename P::T, NP>(kvf + (size_t)head * Tt * flash_tile_pieces(NP) + lane, t0, t1, q, mask, st);
  flash_merge<4>(st, buf, g, lane);
  if (g != 0) return;
  const float inv = 1.0f / st.l;
  const int nk = d / 16;
  const size_t rb = rows_block_of(d);
  float gs = 0.0f;
#pragma unroll
  for (int dt = 0; dt < 2; dt++)
#pragma unroll
    for (int i = 0; i < 16; i++) {
      st.O[dt][i] *= inv;
      gs += st.O[dt][i];
    }
  gs += other_half(gs, lane);
  if (t >= M) return;
#pragma unroll
  for (int dt = 0; dt < 2; dt++)
#pragma unroll
    for (int a8 = 0; a8 < 4; a8++) {
      u32x2 hi, lo;
#pragma unroll
      for (int j = 0; j < 2; j++) {
        uint32_t hw, lw;
        split_f16x2(st.O[dt][a8 * 4 + 2 * j], st.O[dt][a8 * 4 + 2 * j + 1], hw, lw);
        hi[j] = hw;
        lo[j] = lw;
      }
      u32x2 *p = reinterpret_cast<u32x2 *>(out + rows_piece(t, head * 8 + dt * 4 + a8, rb)) + (lane >> 5);
      p[0] = hi;
      p[128] = lo;
    }
  if (lane < 32) put_group_sum(out, t, head, nk, rb, gs);
}

template <int BITS, int EPI, int KVT, class C>
hipError_t run(RowsMm a, hipStream_t s) {
  a.nM = (a.M + C::BM - 1) / C::BM;
  a.nN = (a.N + C::BN - 1) / C::BN;
  a.gm = xcd_rows(a.nM, a.nN, 4.0 * C::BM * a.K, (double)C::BN * a.K * BITS / 8);
  if (a.S < 1 || EPI != kEpiResid || !a.ws || !a.cnt || a.nM * a.nN > a.cnt_words ||
      (size_t)a.nM * a.nN * a.S * C::BM * 64 > a.ws_floats)
    a.S = 1;
  const int gn = 8 / a.gm, blocks = 8 * ((a.nM + a.gm - 1) / a.gm) * ((a.nN + gn - 1) / gn) * a.S;
  hipLaunchKernelGGL((rows_mm_kernel<BITS, EPI, KVT, C>), dim3(blocks), dim3(C::NT), C::LDS, s, a);
  return hipGetLastError();
}

// 32 x 64 tiles by four waves; 64 x 64 where K is long and the tiles many.  M x N x K in us, 32 x
// 64 / 64 x 64: 35 x 1280 x 1280 7.2 / 10.1, 235 x 5120 x 1280 13.5 / 16.4, 886 x 5120 x 1280 32.7
// (355 TFLOP/s) / 34.4, 886 x 1280 x 5120 34.5 / 42.3, 2188 x 5120 x 1280 72.5 / 72.4, 2188 x 1280 x
// 5120 69.7 / 62.5 (459 TFLOP/s, 918 of fp16 products); 64 x 64 at K = 1280 too made prefills of 547
// and 886 rows 2660 -> 2730 and 3590 -> 3735 us.  (Two groups in flight instead of one
// gain nothing, eight waves on a tile lose wherever K is not split instead.)
using RmSmall = RmCfg<1, 4>;
using RmLarge = RmCfg<2, 4>;

template <int BITS, int EPI, int KVT>
hipError_t pick(RowsMm a, hipStream_t s) {
  const long tn = (a.N + 63) / 64, t32 = (a.M + 31) / 32 * tn, t64 = (a.M + 63) / 64 * tn;
  // A long K over S blocks a tile, where the tiles alone leave compute units idle: the S with the
  // least blocks-per-unit / S, plus what storing and adding a partial costs (mlp c_proj, whole
  // prefill in us, unsplit / split: 20 rows 1467 / 1198, 99 rows 1445 / 1256, 200 rows 1640 / 1538;
  // from about two blocks a compute unit on the partials cost what the balance gains).
  a.S = 1;
  if (EPI == kEpiResid && a.K >= 4096 && t32 <= 2L * a.n_cu) {
    double best = 1e30;
    for (int S = 1; S <= kMaxSplit; S++) {
      const double cost = (double)((t32 * S + a.n_cu - 1) / a.n_cu) / S + 0.07 * S;
      if (cost < best) best = cost, a.S = S;
    }
  }
  if (a.K >= 4096 && t64 >= 2L * a.n_cu) return run<BITS, EPI, KVT, RmLarge>(a, s);
  return run<BITS, EPI, KVT, RmSmall>(a, s);
}

template <int BITS>
hipError_t dispatch(const RowsMm &a, int epi, int kvt, hipStream_t s) {
  switch (epi) {
    case kEpiStore: return pick<BITS, kEpiStore, 0>(a, s);
    case kEpiResid: return a.N % 64 == 0 ? pick<BITS, kEpiResid, 0>(a, s) : hipErrorInvalidValue;
    case kEpiGelu: return a.N % 64 == 0 && a.o ? pick<BITS, kEpiGelu, 0>(a, s) : hipErrorInvalidValue;
    case kEpiQKV:
      if (a.N % 192 != 0 || !a.qf || !a.kvf) return hipErrorInvalidValue;
      if (kvt == kKvBf16) return pick<BITS, kEpiQKV, kKvBf16>(a, s);
      return kvt == kKvF32 ? pick<BITS, kEpiQKV, kKvF32>(a, s) : pick<BITS, kEpiQKV, kRowsPairs>(a, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace

size_t rows_planes_pieces(int M, int K) { return (M + 63) / 64 * 2 * rows_block(K / 16, (K / 64 + 15) / 16); }
size_t rows_q_pieces(int M, int H) { return (size_t)H * ((M + 63) / 64 * 2) * 4 * 192; }
size_t rows_kv_pieces(int M, int H) { return (size_t)H * ((M + 63) / 64 * 2) * flash_tile_pieces(3); }
int rows_ldn(int N) { return (N + 63) / 64 * 64; }
size_t rows_scale_floats(int N, int K) { return (size_t)(K / 64) * rows_ldn(N); }
size_t rows_codes_bytes(int N, int K, int bits) { return (size_t)rows_ldn(N) * K * bits / 8; }
size_t rows_bias_pieces(int N, int K) { return rows_ldn(N) / 32 * rows_block(0, (K / 64 + 15) / 16); }

hipError_t rows_params(const DevQL &ql, int bits, int ptype, uint4 *codes, float *scale, uint4 *bw, void *params,
                       hipStream_t s) {
  const long nc = (long)(rows_ldn(ql.N) / 32) * (ql.K / 64) * 128;
  const dim3 cg((unsigned)((nc + 255) / 256));
  uint8_t *co = reinterpret_cast<uint8_t *>(codes);
  if (bits == 8) hipLaunchKernelGGL(rows_codes_kernel<8>, cg, dim3(256), 0, s, ql.codes, ql.N, ql.K, nc, co);
  else hipLaunchKernelGGL(rows_codes_kernel<4>, cg, dim3(256), 0, s, ql.codes, ql.N, ql.K, nc, co);
  const int G = ql.K / 64, ldn = rows_ldn(ql.N);
  const long n = (long)ldn * ((G + 15) / 16) * 2;
  const float off = bits == 8 ? 128.0f : 8.0f;
  const dim3 grid((unsigned)((n + 255) / 256));
  if (ptype == kParamF32)
    hipLaunchKernelGGL(rows_params_kernel<kParamF32>, grid, dim3(256), 0, s, ql.params, ql.N, G, ldn, off, scale,
                       reinterpret_cast<u32x4 *>(bw), params);
  else
    hipLaunchKernelGGL(rows_params_kernel<kParamF16>, grid, dim3(256), 0, s, ql.params, ql.N, G, ldn, off, scale,
                       reinterpret_cast<u32x4 *>(bw), params);
  return hipGetLastError();
}

hipError_t rows_ln(const float *x, const float *w, const float *b, const float *w2, const float *b2, int M, int d,
                   uint4 *out, hipStream_t s) {
  auto *fn = d <= 512 ? ln_planes_kernel<2> : d <= 1280 ? ln_planes_kernel<5> : d <= 2048 ? ln_planes_kernel<8> : ln_planes_kernel<0>;
  hipLaunchKernelGGL(fn, dim3((M + 1) / 2), dim3(64), 0, s, x, w, b, w2, b2, M, d, reinterpret_cast<u32x4 *>(out));
  return hipGetLastError();
}

hipError_t rows_mm(const RowsMm &a, int bits, int epi, int kvt, hipStream_t s) {
  if (a.M < 1 || a.N < 1 || a.K < 64 || a.K % 64 != 0 || !a.x || !a.codes || !a.scale || !a.bw || !a.bias ||
      (a.st && (a.K > 2048 || !a.fG || !a.fc)))
    return hipErrorInvalidValue;
  return bits == 8 ? dispatch<8>(a, epi, kvt, s) : dispatch<4>(a, epi, kvt, s);
}

hipError_t rows_attn(const uint4 *qf, const uint4 *kvf, int M, int H, const int *kstart, const int *order, int kvt,
                     uint4 *out, hipStream_t s) {
  if (M < 1 || H < 1) return hipErrorInvalidValue;
  const dim3 grid(H, (M + 31) / 32);
  const u32x4 *q = reinterpret_cast<const u32x4 *>(qf), *kv = reinterpret_cast<const u32x4 *>(kvf);
  auto *fn = kvt == kKvBf16 ? rows_attn_kernel<kKvBf16> : kvt == kKvF32 ? rows_attn_kernel<kKvF32> : rows_attn_kernel<kRowsPairs>;
  hipLaunchKernelGGL(fn, grid, dim3(256), 0, s, q, kv, M, kstart, order, reinterpret_cast<u32x4 *>(out));
  return hipGetLastError();
}

}  // namespace itts
