// Matrix products, attention and row norms of the CFM estimator on the MFMA units
// (crates/core/src/models/cfm.rs) for forwards of 64 rows and more.
//
// Every operand lives in memory as fp16 hi/lo planes in MFMA fragment order (frag.h): the
// weights are laid out once, each activation by the kernel that produces it, so a product
// y = Ah Wh + Ah Wl + Al Wh (~22-bit operands, fp32 accumulation) loads fragments straight
// into registers.  The epilogues stage the fp32 tile in LDS and write whole pieces: bias and
// residual, the SwiGLU, WaveNet's gate and residual / skip sums, and the attention's operands
// with rope applied.
#include "frag.h"
#include "kernels.h"

namespace itts {

namespace {

constexpr int kHd = 64;

__device__ __forceinline__ float silu(float x) { return x / (1.0f + expf(-x)); }
__device__ __forceinline__ float sigm(float x) { return 1.0f / (1.0f + expf(-x)); }

// ---- operand layout ---------------------------------------------------------------------
// Weight rows W [N][ldw] (K values) -> K steps kt0 .. of the fragment planes `out` (nk K steps
// a row block), zeros past N and K.  With ilv = F (N = 2F), out row r holds row (r >> 5 & 1) F
// + 32 (r >> 6) + (r & 31): each 64-row tile is 32 rows of the first half, then the matching
// 32 of the second (zeros where 32 (r >> 6) + (r & 31) >= F).
__global__ __launch_bounds__(256) void weight_frag_kernel(const float *W, int ldw, int N, int K, int rows, int kt0,
                                                          int kts, int nk, int ilv, u32x4 *out) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long)rows * kts * 2) return;
  const int r = (int)(i % rows), k8 = (int)(i / rows);
  const int c = 32 * (r >> 6) + (r & 31);
  const int src = ilv ? (c < ilv ? ((r >> 5) & 1) * ilv + c : N) : r;
  float v[8];
#pragma unroll
  for (int j = 0; j < 8; j++) v[j] = src < N && k8 * 8 + j < K ? W[(size_t)src * ldw + k8 * 8 + j] : 0.0f;
  u32x4 hi, lo;
  split8(v, hi, lo);
  const size_t p = frag_piece(r, kt0 * 2 + k8, nk);
  out[p] = hi;
  out[p + 64] = lo;
}

// fp32 rows X [R][ld] (K values) -> fragment planes of nk K steps, zeros past K.  Lanes: 8
// rows x 8 chunks, so rows are read 256 bytes at a time and pieces written 128.
__global__ __launch_bounds__(256) void rows_frag_kernel(const float *X, int ld, int R, int K, int nk, int row0,
                                                        u32x4 *out) {
  const int r = blockIdx.x * 32 + (threadIdx.x >> 6) * 8 + ((threadIdx.x >> 3) & 7);
  const int k8 = blockIdx.y * 8 + (threadIdx.x & 7);
  if (r >= R || k8 >= 2 * nk) return;
  float v[8];
#pragma unroll
  for (int j = 0; j < 8; j++) v[j] = k8 * 8 + j < K ? X[(size_t)r * ld + k8 * 8 + j] : 0.0f;
  u32x4 hi, lo;
  split8(v, hi, lo);
  const size_t p = frag_piece(row0 + r, k8, nk);
  out[p] = hi;
  out[p + 64] = lo;
}

// AdaLN over RMSNorm (cfm.rs:173-182) or, with FINAL, the final layer's norm (cfm.rs:605-609),
// written as fragment planes.  Sixteen lanes a row (lane c of them: columns 128 j + 8 c ..),
// four rows a wave, one wave a block; NJ = d / 128 chunks in registers, everything loaded
// before the first reduction (one memory round trip), or any d with NJ = 0 (read again).
template <int NJ, bool FINAL>
__global__ __launch_bounds__(64) void norm_frag_kernel(const float *x, int R, int T, int d, const float *mod,
                                                       int ld_mod, const float *norm_w, u32x4 *out) {
  constexpr int ND = NJ ? NJ : 1;
  const int lane = threadIdx.x, c = lane & 15;
  const int rl = blockIdx.x * 4 + (lane >> 4), r = min(rl, R - 1), b = r / T;
  const int nc = d / 8;  // chunks of a row; lane c takes c, c + 16, ..
  const float4 *xr = reinterpret_cast<const float4 *>(x + (size_t)r * d);
  const float4 *m0 = reinterpret_cast<const float4 *>(mod + (size_t)b * ld_mod);
  const float4 *m1 = reinterpret_cast<const float4 *>(mod + (size_t)b * ld_mod + d);
  const float4 *nw = reinterpret_cast<const float4 *>(norm_w);
  float4 v[ND][2], w[ND][2], s[ND][2], g[ND][2];
  auto load = [&](int k, int i, bool all) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 2; q++) {
      v[i][q] = xr[2 * k + q];
      if (all) {
        w[i][q] = m0[2 * k + q];
        s[i][q] = m1[2 * k + q];
        if constexpr (!FINAL) g[i][q] = nw[2 * k + q];
      }
    }
  };
  if constexpr (NJ > 0) {
#pragma unroll
    for (int j = 0; j < NJ; j++) load(c + 16 * j, j, true);
  }
  auto row_sum = [&](float t) __attribute__((always_inline)) {  // over the row's sixteen lanes
    t += dpp_pair<0xB1>(t);
    t += dpp_pair<0x4E>(t);
    t += dpp_pair<0x141>(t);
    return t + dpp_pair<0x140>(t);
  };
  auto each = [&](bool all, auto f) __attribute__((always_inline)) {
    if constexpr (NJ > 0) {
#pragma unroll
      for (int j = 0; j < NJ; j++) f(c + 16 * j, j);
    } else {
      for (int k = c; k < nc; k += 16) {
        load(k, 0, all);
        f(k, 0);
      }
    }
  };
  float mean = 0.0f;
  if constexpr (FINAL) {
    float t = 0.0f;
    each(false, [&](int, int i) __attribute__((always_inline)) {
#pragma unroll
      for (int q = 0; q < 2; q++) t += (v[i][q].x + v[i][q].y) + (v[i][q].z + v[i][q].w);
    });
    mean = row_sum(t) / (float)d;
  }
  float t2 = 0.0f;
  each(false, [&](int, int i) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 2; q++) {
      const float4 e = make_float4(v[i][q].x - mean, v[i][q].y - mean, v[i][q].z - mean, v[i][q].w - mean);
      t2 += (e.x * e.x + e.y * e.y) + (e.z * e.z + e.w * e.w);
    }
  });
  const float rs = 1.0f / sqrtf(row_sum(t2) / (float)d + (FINAL ? 1e-6f : 1e-5f));
  each(true, [&](int k, int i) __attribute__((always_inline)) {
    float y[8];
#pragma unroll
    for (int q = 0; q < 2; q++) {
      const float xv[4] = {v[i][q].x, v[i][q].y, v[i][q].z, v[i][q].w};
      const float wv[4] = {w[i][q].x, w[i][q].y, w[i][q].z, w[i][q].w};
      const float sv[4] = {s[i][q].x, s[i][q].y, s[i][q].z, s[i][q].w};
      if constexpr (FINAL) {  // (shift, scale)
#pragma unroll
        for (int e = 0; e < 4; e++) y[4 * q + e] = ((xv[e] - mean) * rs) * (1.0f + sv[e]) + wv[e];
      } else {
        const float gv[4] = {g[i][q].x, g[i][q].y, g[i][q].z, g[i][q].w};
#pragma unroll
        for (int e = 0; e < 4; e++) y[4 * q + e] = wv[e] * (xv[e] * rs * gv[e]) + sv[e];
      }
    }
    u32x4 hi, lo;
    split8(y, hi, lo);
    if (rl < R) {
      const size_t p = frag_piece(r, k, d / 16);
      out[p] = hi;
      out[p + 64] = lo;
    }
  });
}

// ---- the product ------------------------------------------------------------------------
// A wave forms a (32 TM) x (32 TN) tile, three products each MFMA tile, from fragments loaded
// AH K steps ahead of their use.  Block: one such tile by KS waves that take a part of K (their
// partial tiles added in wave order).  The fp32 tile goes through LDS; a thread
// then takes (row, 8 columns) items.
template <int TM_, int TN_, int KS_, int AH_>
struct MmCfg {
  static constexpr int TM = TM_, TN = TN_, KS = KS_, AH = AH_;
  static constexpr int BM = 32 * TM, BN = 32 * TN, LD = BN + 4, NT = 64 * KS;
  static constexpr int KL = KS > 2 ? KS / 2 : KS;  // partial tiles held in LDS
  static constexpr size_t LDS = sizeof(float) * KL * BM * LD;
  static_assert(BN % 64 == 0, "column groups of 64");
  static_assert(128 % BN == 0 && 128 % BM == 0, "whole tiles in the planes' 128-row blocks");
};

template <class C, int EPI>
__global__ __launch_bounds__(C::NT, 2) void mm_kernel(CfmMm a) {
  constexpr int TM = C::TM, TN = C::TN, KS = C::KS, BM = C::BM, BN = C::BN, LD = C::LD, NT = C::NT, AH = C::AH;
  extern __shared__ __attribute__((aligned(16))) float red[];
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, r31 = lane & 31;
  const int kq = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Block -> tile.  Blocks go to the 8 XCDs round-robin, and each XCD reads what its tiles need
  // through its own L2: XCD x takes every gm-th row tile from x % gm and every gn-th column
  // tile from x / gm, so that the operands cross the fabric gn and gm times, not 8 times each.
  const int gn = 8 / a.gm, x = blockIdx.x & 7, j = blockIdx.x >> 3;
  const int pn = (a.nN + gn - 1) / gn;
  const int tmz = j / pn * a.gm + x % a.gm, tn = j % pn * gn + x / a.gm;
  if (tmz >= a.nM * a.nz || tn >= a.nN) return;
  const int z = tmz / a.nM, m0 = (tmz - z * a.nM) * BM, n0 = tn * BN;
  const int k0 = a.nk * kq / KS, k1 = a.nk * (kq + 1) / KS;

  const u32x4 *wp[TN], *ap[TM], *ap2[TM];
#pragma unroll
  for (int i = 0; i < TN; i++)
    wp[i] = reinterpret_cast<const u32x4 *>(a.w) + ((size_t)((n0 >> 5) + i) * a.nk) * 128 + lane;
#pragma unroll
  for (int i = 0; i < TM; i++) {
    const int row = z * a.zr + m0 + i * 32 + r31, rp = h * 32 + (row & 31);
    ap[i] = reinterpret_cast<const u32x4 *>(a.a) + z * a.sa + ((size_t)(row >> 5) * a.kt_a) * 128 + rp;
    ap2[i] = a.a2 ? reinterpret_cast<const u32x4 *>(a.a2) + ((size_t)(row >> 5) * a.kt_a2) * 128 + rp : ap[i];
  }
  struct Frag {
    u32x4 a[TM][2], w[TN][2];
  };
  auto load = [&](int kt, Frag &f) __attribute__((always_inline)) {
    const int kc = min(kt, k1 - 1);
#pragma unroll
    for (int i = 0; i < TM; i++) {
      const u32x4 *p;
      if constexpr (EPI == kMmGate || EPI == kMmConv) {  // a convolution's taps: tap j reads row m + j of a padded operand
        const int tap = kc / a.taps_kt, ktd = kc - tap * a.taps_kt;
        const int row = m0 + i * 32 + r31 + tap;
        p = reinterpret_cast<const u32x4 *>(a.a) + z * a.sa + ((size_t)(row >> 5) * a.kt_a + ktd) * 128 + h * 32 +
            (row & 31);
      } else {
        p = kc < a.nk1 ? ap[i] + (size_t)kc * 128 : ap2[i] + (size_t)(kc - a.nk1) * 128;
      }
      f.a[i][0] = p[0];
      f.a[i][1] = p[64];
    }
#pragma unroll
    for (int i = 0; i < TN; i++) {
      const u32x4 *q = wp[i] + (size_t)kc * 128;
      f.w[i][0] = q[0];
      f.w[i][1] = q[64];
    }
  };
  floatx16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[i][j][e] = 0.0f;
  auto mma = [&](const Frag &f) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < 3; p++)
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
          acc[i][j] = ITTS_MFMA16(__builtin_bit_cast(f16x8, f.a[i][p == 2]), __builtin_bit_cast(f16x8, f.w[j][p == 1]),
                                  acc[i][j], 0, 0, 0);
  };
  // The old rows that the epilogue adds to, loaded ahead of the K loop where a thread has few
  // items (otherwise a memory round trip follows the product).
  constexpr int ITEMS = BM * (BN / 8), IT = ITEMS / NT;
  constexpr bool kOld = (EPI == kMmPlain || EPI == kMmResSkip) && IT <= 2 && ITEMS % NT == 0;
  float4 old[kOld ? IT : 1][2];
  auto item = [&](int q, int &row, int &col) __attribute__((always_inline)) {
    row = (q >> 3) % BM;
    col = ((q >> 3) / BM * 8 + (q & 7)) * 8;
  };
  if constexpr (kOld) {
#pragma unroll
    for (int i = 0; i < IT; i++) {
      int row, col;
      item(i * NT + tid, row, col);
      const int r = min(m0 + row, a.M - 1), n = n0 + col;
      const float *p = a.yr && a.vec && n + 8 <= a.N ? a.yr + (size_t)z * a.sy + (size_t)r * a.ldy + n : nullptr;
      if constexpr (EPI == kMmResSkip) {
        const int d = a.ldy;
        p = n < a.N - d ? a.y + (size_t)r * d + n : n < a.N && !a.first ? a.y2 + (size_t)r * d + n - (a.N - d) : nullptr;
      }
      old[i][0] = old[i][1] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (p) {
        old[i][0] = reinterpret_cast<const float4 *>(p)[0];
        old[i][1] = reinterpret_cast<const float4 *>(p)[1];
      }
    }
  }
  if (k0 < k1) {
    Frag f[AH];
#pragma unroll
    for (int s = 0; s < AH; s++) load(k0 + s, f[s]);
    int kt = k0;
    for (; kt + AH < k1; kt += AH) {
#pragma unroll
      for (int s = 0; s < AH; s++) {
        mma(f[s]);
        load(kt + s + AH, f[s]);
      }
    }
#pragma unroll
    for (int s = 0; s < AH; s++)
      if (kt + s < k1) mma(f[s]);
  }

  // (with four parts of K two tiles of LDS do: four blocks of 64 x 64 to a compute unit, not two)
  constexpr int KL = C::KL;
  parts_to_lds<TM, TN, KS, KL, BM, LD>(red, acc, kq, h, r31);
  auto tile8 = [&](int row, int col, float v[8]) __attribute__((always_inline)) {
    parts_row8<KL, BM, LD>(red, row, col, v);
  };
  auto add8 = [&](const float *p, float v[8]) __attribute__((always_inline)) {
    const float4 x = *reinterpret_cast<const float4 *>(p), y = *reinterpret_cast<const float4 *>(p + 4);
    v[0] += x.x, v[1] += x.y, v[2] += x.z, v[3] += x.w, v[4] += y.x, v[5] += y.y, v[6] += y.z, v[7] += y.w;
  };
  auto put8 = [&](float *p, const float v[8]) __attribute__((always_inline)) {
    *reinterpret_cast<float4 *>(p) = make_float4(v[0], v[1], v[2], v[3]);
    *reinterpret_cast<float4 *>(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
  };
  auto put_frag = [&](u32x4 *o, long row, int k8, int nk, const float v[8]) __attribute__((always_inline)) {
    u32x4 hi, lo;
    split8(v, hi, lo);
    const size_t p = frag_piece(row, k8, nk);
    o[p] = hi;
    o[p + 64] = lo;
  };

  auto add_old = [&](int i, const float *p, float v[8]) __attribute__((always_inline)) {
    if constexpr (kOld) {
      const float4 x = old[i][0], y = old[i][1];
      v[0] += x.x, v[1] += x.y, v[2] += x.z, v[3] += x.w, v[4] += y.x, v[5] += y.y, v[6] += y.z, v[7] += y.w;
    } else {
      add8(p, v);
    }
  };

  if constexpr (EPI == kMmPlain || EPI == kMmConv) {
    // y = v + bias (+ yr), fp32 rows and / or fragment planes
#pragma unroll 2
    for (int i = 0; i < (ITEMS + NT - 1) / NT; i++) {
      const int q = i * NT + tid;
      int row, col;
      item(q, row, col);
      const int r = m0 + row, n = n0 + col;
      if (q >= ITEMS || r >= a.M || n >= a.N) continue;
      float v[8];
      tile8(row, col, v);
      const size_t o = (size_t)z * a.sy + (size_t)r * a.ldy + n;
      if (a.vec && n + 8 <= a.N) {
        if (a.bias) add8(a.bias + n, v);
        if (a.yr) add_old(i, a.yr + o, v);
        if (a.y) put8(a.y + o, v);
      } else {
        for (int k = 0; k < 8; k++) {
          if (n + k >= a.N) {
            v[k] = 0.0f;
            continue;
          }
          if (a.bias) v[k] += a.bias[n + k];
          if (a.yr) v[k] += a.yr[o + k];
          if (a.y) a.y[o + k] = v[k];
        }
      }
      if (a.o) {
        const int b = a.T ? r / a.T : z, rr = a.T ? r - b * a.T : r;
        put_frag(reinterpret_cast<u32x4 *>(a.o) + b * a.so, rr + a.o_row0, n >> 3, a.kt_o, v);
      }
    }
  } else if constexpr (EPI == kMmSwiglu || EPI == kMmGate) {
    // tile columns 0-31 and 32-63 of each 64 are the two halves' same 32 outputs
#pragma unroll 2
    for (int q = tid; q < BM * (BN / 16); q += NT) {
      const int c = q & 3, row = (q >> 2) % BM, grp = (q >> 2) / BM;
      const int r = m0 + row, n = ((n0 >> 6) + grp) * 32 + c * 8;  // output column
      if (r >= a.M || n >= a.N) continue;
      float x[8], y[8];
      tile8(row, grp * 64 + c * 8, x);
      tile8(row, grp * 64 + 32 + c * 8, y);
      if constexpr (EPI == kMmGate) {
        add8(a.bias + n, x);
        add8(a.bias + a.N + n, y);
        add8(a.g + (size_t)z * a.ld_g + n, x);
        add8(a.g + (size_t)z * a.ld_g + a.N + n, y);
#pragma unroll
        for (int k = 0; k < 8; k++) x[k] = tanhf(x[k]) * sigm(y[k]);
      } else {
#pragma unroll
        for (int k = 0; k < 8; k++) x[k] = silu(x[k]) * y[k];
      }
      put_frag(reinterpret_cast<u32x4 *>(a.o), (long)z * a.M + r, n >> 3, a.kt_o, x);
    }
  } else if constexpr (EPI == kMmResSkip) {
    // columns < d: h += v + bias (fp32 rows and the next convolution's padded planes);
    // columns d ..: out (+)= v + bias.  The last layer has only out's columns.
#pragma unroll 2
    for (int i = 0; i < (ITEMS + NT - 1) / NT; i++) {
      const int q = i * NT + tid;
      int row, col;
      item(q, row, col);
      const int r = m0 + row, n = n0 + col;
      if (q >= ITEMS || r >= a.M || n >= a.N) continue;
      float v[8];
      tile8(row, col, v);
      add8(a.bias + n, v);
      const int d = a.ldy;
      if (n < a.N - d) {
        float *hp = a.y + (size_t)r * d + n;
        add_old(i, hp, v);
        put8(hp, v);
        const int b = r / a.T;
        put_frag(reinterpret_cast<u32x4 *>(a.o) + b * a.so, r - b * a.T + a.o_row0, n >> 3, a.kt_o, v);
      } else {
        float *op = a.y2 + (size_t)r * d + n - (a.N - d);
        if (!a.first) add_old(i, op, v);
        put8(op, v);
      }
    }
  } else {
    // Q (rope, scaled by log2(e) / sqrt(64)) and K (rope) row fragments, V^T fragments with the
    // attention's key order; a 64-column group is one head of one of q, k, v.  Rows past M are
    // zeros to the end of the 32-row tile that holds row M - 1; a tile after it may stay unwritten
    // (the attention's blocks of four query tiles load such a Q tile and drop what comes of it).
    const int d = a.N / 3, H = d / kHd, Tt = (a.M + 63) / 64 * 2;  // 32-key tiles
    const float2 *tab = reinterpret_cast<const float2 *>(a.g);
#pragma unroll
    for (int grp = 0; grp < BN / 64; grp++) {
      const int nb = n0 + grp * 64;
      if (nb >= a.N) break;
      const int which = nb / d, head = (nb - which * d) / kHd;
      const size_t bh = (size_t)z * H + head;
      if (which < 2) {
#pragma unroll 2
        for (int q = tid; q < BM * 8; q += NT) {
          const int c = q & 7, row = q >> 3, t = m0 + row;
          if (t >= Tt * 32) continue;
          float v[8], o[8];
          tile8(row, grp * 64 + c * 8, v);
          const float4 *tr = reinterpret_cast<const float4 *>(tab + (size_t)min(t, a.M - 1) * (kHd / 2) + c * 4);
          const float4 x = tr[0], y = tr[1];
          const float cs[4] = {x.x, x.z, y.x, y.z}, sn[4] = {x.y, x.w, y.y, y.w};
          const float sc = t < a.M ? (which == 0 ? 0.125f * 1.4426950408889634f : 1.0f) : 0.0f;
#pragma unroll
          for (int j = 0; j < 4; j++) {
            o[2 * j] = t < a.M ? (v[2 * j] * cs[j] - v[2 * j + 1] * sn[j]) * sc : 0.0f;
            o[2 * j + 1] = t < a.M ? (v[2 * j] * sn[j] + v[2 * j + 1] * cs[j]) * sc : 0.0f;
          }
          u32x4 hi, lo;
          split8(o, hi, lo);
          u32x4 *dst;
          const int pc = (c & 1) * 32 + (t & 31);
          if (which == 0)
            dst = reinterpret_cast<u32x4 *>(a.o) + ((bh * Tt + (t >> 5)) * 4 + (c >> 1)) * 128 + pc;
          else
            dst = reinterpret_cast<u32x4 *>(a.o2) + (bh * Tt + (t >> 5)) * flash_tile_pieces(2) + (c >> 1) * 128 + pc;
          dst[0] = hi;
          dst[64] = lo;
        }
      } else {
        // item: dim e, eight key positions p8 of a 16-key step: keys 16 s + 4 hh + {0..3, 8..11}
#pragma unroll 2
        for (int q = tid; q < BM * 8; q += NT) {
          const int e = q & 63, k8 = q >> 6, rb = (k8 >> 1) * 16 + (k8 & 1) * 4, t = m0 + rb;
          if (t >= Tt * 32) continue;
          float v[8];
#pragma unroll
          for (int j = 0; j < 8; j++) {
            const int row = rb + (j >> 2) * 8 + (j & 3);
            float s = red[(size_t)row * LD + grp * 64 + e];
#pragma unroll
            for (int k = 1; k < KL; k++) s += red[((size_t)k * BM + row) * LD + grp * 64 + e];
            v[j] = m0 + row < a.M ? s : 0.0f;
          }
          u32x4 hi, lo;
          split8(v, hi, lo);
          u32x4 *dst = reinterpret_cast<u32x4 *>(a.o2) + (bh * Tt + (t >> 5)) * flash_tile_pieces(2) +
                       (4 + (e >> 5) * 2 + ((t >> 4) & 1)) * 128 + (k8 & 1) * 32 + (e & 31);
          dst[0] = hi;
          dst[64] = lo;
        }
      }
    }
  }
}

// The same fragments from fp32 rows qkv [B][T][3d] (forwards of under 64 rows, whose
// projections are fp32 products): thread = (b, head, q / k / v, row, chunk of 8), or for v
// (b, head, dim, 8 key positions).
__global__ __launch_bounds__(256) void qkv_frag_kernel(const float *qkv, const float2 *tab, int B, int T, int H,
                                                       u32x4 *qf, u32x4 *kvf) {
  const int Tt = (T + 63) / 64 * 2, d = H * kHd;
  const long per = (long)B * H * Tt * 32 * 8, i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= 3 * per) return;
  const int which = (int)(i / per);
  long j = i % per;
  const int c = (int)(j & 7);
  j >>= 3;
  const int t = (int)(j % (Tt * 32));
  const size_t bh = (size_t)(j / (Tt * 32));
  const int b = (int)(bh / H), head = (int)(bh % H);
  const float *base = qkv + (size_t)b * T * 3 * d + which * d + head * kHd;
  float o[8];
  u32x4 *dst;
  if (which < 2) {
    const float *p = base + (size_t)min(t, T - 1) * 3 * d + c * 8;
    const float2 *tr = tab + (size_t)min(t, T - 1) * (kHd / 2) + c * 4;
    const float sc = t < T ? (which == 0 ? 0.125f * 1.4426950408889634f : 1.0f) : 0.0f;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const float2 cs = tr[k];
      o[2 * k] = t < T ? (p[2 * k] * cs.x - p[2 * k + 1] * cs.y) * sc : 0.0f;
      o[2 * k + 1] = t < T ? (p[2 * k] * cs.y + p[2 * k + 1] * cs.x) * sc : 0.0f;
    }
    const int pc = (c & 1) * 32 + (t & 31);
    dst = which == 0 ? qf + ((bh * Tt + (t >> 5)) * 4 + (c >> 1)) * 128 + pc
                     : kvf + (bh * Tt + (t >> 5)) * flash_tile_pieces(2) + (c >> 1) * 128 + pc;
  } else {
    // (t, c) -> dim e, key positions 8 k8 .. +7 of the sequence's 16-key steps
    const int f = t * 8 + c, e = f & 63, k8 = f >> 6, t0 = (k8 >> 1) * 16 + (k8 & 1) * 4;
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const int tk = t0 + (k >> 2) * 8 + (k & 3);
      o[k] = tk < T ? base[(size_t)tk * 3 * d + e] : 0.0f;
    }
    dst = kvf + (bh * Tt + (t0 >> 5)) * flash_tile_pieces(2) + (4 + (e >> 5) * 2 + ((t0 >> 4) & 1)) * 128 +
          (k8 & 1) * 32 + (e & 31);
  }
  u32x4 hi, lo;
  split8(o, hi, lo);
  dst[0] = hi;
  dst[64] = lo;
}

// ---- attention (cfm.rs:274-289): non-causal over T positions ----------------------------
// Bound by the MFMA and VALU issue of its three fp16 products and exponentials: 24.2 us at
// 2 x 1033 frames (541 TFLOP/s of fp16 products; 73 us before as LDS-staged tiles, a partial
// buffer and a combine pass) and 81.4 us at 2 x 2325 (815; 224 us before).
// Block: four waves, 32 WQ queries of one (batch, head), the key tiles split over WK = 4 / WQ
// wave groups.  Output rows b T + t as fragment planes [B T][d].
template <int WQ>
__global__ __launch_bounds__(256, 2) void attn_kernel(const u32x4 *qf, const u32x4 *kvf, int H, int T, int d,
                                                      u32x4 *out, float *out_f) {
  constexpr int WK = 4 / WQ;
  __shared__ float buf[WK > 1 ? 4 * 2112 : 1];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = wave % WK, wq = wave / WK;
  const int bh = blockIdx.x, b = bh / H, head = bh % H;
  const int Tt = (T + 63) / 64 * 2, nt = (T + 31) / 32;
  const int qt = blockIdx.y * WQ + wq;
  u32x4 q[4][2];
  const u32x4 *qp = qf + (((size_t)bh * Tt + min(qt, Tt - 1)) * 4) * 128 + lane;
#pragma unroll
  for (int kk = 0; kk < 4; kk++) {
    q[kk][0] = qp[kk * 128];
    q[kk][1] = qp[kk * 128 + 64];
  }
  FlashState st;
  flash_init(st);
  const int per = (nt + WK - 1) / WK, t0 = g * per, t1 = min(nt, t0 + per);
  auto mask = [&](int t, floatx16 &S) __attribute__((always_inline)) {
    if (t == nt - 1 && (T & 31)) {
#pragma unroll
      for (int i = 0; i < 16; i++)
        if (t * 32 + (i >> 2) * 8 + (lane >> 5) * 4 + (i & 3) >= T) S[i] = -INFINITY;
    }
  };
  flash_tiles<F16Pairs, 2>(kvf + (size_t)bh * Tt * flash_tile_pieces(2) + lane, t0, t1, q, mask, st);
  flash_merge<WK>(st, buf + wq * WK * 2112, g, lane);
  const int t = qt * 32 + (lane & 31);
  if (g != 0 || t >= T) return;
  const float inv = 1.0f / st.l;
  const long r = (long)b * T + t;
  if (out_f) {
    float4 *o = reinterpret_cast<float4 *>(out_f + (size_t)r * d + head * kHd) + (lane >> 5);
#pragma unroll
    for (int i = 0; i < 8; i++)
      o[(i >> 2) * 8 + (i & 3) * 2] = make_float4(st.O[i >> 2][(i & 3) * 4] * inv, st.O[i >> 2][(i & 3) * 4 + 1] * inv,
                                                  st.O[i >> 2][(i & 3) * 4 + 2] * inv, st.O[i >> 2][(i & 3) * 4 + 3] * inv);
    return;
  }
#pragma unroll
  for (int dt = 0; dt < 2; dt++)
#pragma unroll
    for (int a8 = 0; a8 < 4; a8++) {
      u32x2 hi, lo;
#pragma unroll
      for (int j = 0; j < 2; j++) {
        uint32_t hw, lw;
        split_f16x2(st.O[dt][a8 * 4 + 2 * j] * inv, st.O[dt][a8 * 4 + 2 * j + 1] * inv, hw, lw);
        hi[j] = hw;
        lo[j] = lw;
      }
      // dims 8 a8 + 4 (lane >> 5) .. +3: half of a piece
      u32x2 *p = reinterpret_cast<u32x2 *>(out + frag_piece(r, head * 8 + dt * 4 + a8, d / 16)) + (lane >> 5);
      p[0] = hi;
      p[128] = lo;
    }
}

template <int EPI>
int mm_cols(const CfmMm &a) {  // columns of the product (interleaved halves count both)
  return EPI == kMmSwiglu || EPI == kMmGate ? (a.N + 31) / 32 * 64 : a.N;
}

template <class C, int EPI>
hipError_t mm_run(CfmMm a, int batch, hipStream_t s) {
  a.nM = (a.M + C::BM - 1) / C::BM;
  a.nN = (mm_cols<EPI>(a) + C::BN - 1) / C::BN;
  a.nz = batch;
  a.gm = xcd_rows(a.nM * batch, a.nN, (double)C::BM * (EPI == kMmGate || EPI == kMmConv ? a.taps_kt : a.nk) * 64,
                  (double)C::BN * a.nk * 64);
  const int gn = 8 / a.gm, blocks = 8 * ((a.nM * batch + a.gm - 1) / a.gm) * ((a.nN + gn - 1) / gn);
  hipLaunchKernelGGL((mm_kernel<C, EPI>), dim3(blocks), dim3(C::NT), C::LDS, s, a);
  return hipGetLastError();
}

template <class C, int EPI>
hipError_t mm_set() {
  return hipFuncSetAttribute(reinterpret_cast<const void *>(mm_kernel<C, EPI>),
                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)C::LDS);
}

// 64 x 64 tiles by four waves that split K; where those would be few and K short (the
// estimator's d-wide outputs), 32 x 64 tiles by two waves, or by four while those do not fill
// the chip once.  M x N x K in us, 64 x 64 by four / 32 x 64 by two / by four: 374 x 512 x 512
// 6.8 / 5.1 / 4.9, 2066 x 512 x 512 10.0 / 8.8 / 9.9, 2066 x 512 x 1536 20.0 / 19.8 / 21.8, 2066 x
// 1536 x 512 17.5 / 19.2 / 19.5, 2066 x 3072 x 512 29.2 / 32.9 / 33.8, 4650 x 1024 x 2560 78.7
// (310 TFLOP/s, 930 of fp16 products) / 100 / 106; 128-row and 128-column tiles lose throughout.
using MmLarge = MmCfg<2, 2, 4, 2>;
using MmSmall2 = MmCfg<1, 2, 2, 4>;
using MmSmall4 = MmCfg<1, 2, 4, 4>;

template <int EPI>
hipError_t mm_attr() {
  hipError_t e = mm_set<MmLarge, EPI>();
  if (e == hipSuccess) e = mm_set<MmSmall2, EPI>();
  if (e == hipSuccess) e = mm_set<MmSmall4, EPI>();
  return e;
}

template <int EPI>
hipError_t mm_pick(const CfmMm &a, int batch, int n_cu, hipStream_t s) {
  const long tn = (mm_cols<EPI>(a) + 63) / 64 * batch;
  const long t64 = (a.M + 63) / 64 * tn, t32 = (a.M + 31) / 32 * tn;
  if (t32 <= n_cu) return mm_run<MmSmall4, EPI>(a, batch, s);
  if (2 * t64 <= 5L * n_cu && a.nk <= 96) return mm_run<MmSmall2, EPI>(a, batch, s);
  return mm_run<MmLarge, EPI>(a, batch, s);
}
inline unsigned nblk(long n, int t = 256) { return (unsigned)((n + t - 1) / t); }

}  // namespace

size_t cfm_frag_pieces(long rows, int nk) { return (size_t)((rows + 127) / 128 * 4) * nk * 128; }

hipError_t cfm_weight_frag(const float *W, int ldw, int N, int K, int kt0, int nk, int ilv, uint4 *out,
                           hipStream_t s) {
  if (N < 1 || K < 1 || (ilv && N != 2 * ilv)) return hipErrorInvalidValue;
  const int cols = ilv ? (ilv + 31) / 32 * 64 : N, rows = (cols + 127) / 128 * 128, kts = (K + 15) / 16;
  if (kt0 + kts > nk) return hipErrorInvalidValue;
  hipLaunchKernelGGL(weight_frag_kernel, dim3(nblk((long)rows * kts * 2)), dim3(256), 0, s, W, ldw, N, K, rows, kt0,
                     kts, nk, ilv, reinterpret_cast<u32x4 *>(out));
  return hipGetLastError();
}

hipError_t cfm_rows_frag(const float *X, int ld, int R, int K, int nk, int row0, uint4 *out, hipStream_t s) {
  if (R < 1 || K < 1 || K > 16 * nk) return hipErrorInvalidValue;
  hipLaunchKernelGGL(rows_frag_kernel, dim3((R + 31) / 32, (2 * nk + 7) / 8), dim3(256), 0, s, X, ld, R, K, nk, row0,
                     reinterpret_cast<u32x4 *>(out));
  return hipGetLastError();
}

hipError_t cfm_norm_frag(const float *x, int R, int T, int d, const float *mod, int ld_mod, const float *norm_w,
                         bool final_norm, uint4 *out, hipStream_t s) {
  const dim3 grid((R + 3) / 4), blk(64);
  u32x4 *o = reinterpret_cast<u32x4 *>(out);
#define NORM(NJ, F) hipLaunchKernelGGL((norm_frag_kernel<NJ, F>), grid, blk, 0, s, x, R, T, d, mod, ld_mod, norm_w, o)
  if (final_norm) {
    if (d == 512) NORM(4, true);
    else NORM(0, true);
  } else {
    if (d == 512) NORM(4, false);
    else NORM(0, false);
  }
#undef NORM
  return hipGetLastError();
}

hipError_t cfm_mm_init() {
  for (hipError_t (*f)() : {mm_attr<kMmPlain>, mm_attr<kMmConv>, mm_attr<kMmGate>, mm_attr<kMmSwiglu>,
                            mm_attr<kMmResSkip>, mm_attr<kMmQkv>})
    if (hipError_t e = f()) return e;
  return hipSuccess;
}

hipError_t cfm_mm(CfmMm a, int epi, int batch, int n_cu, hipStream_t s) {
  if (batch < 1 || a.M < 1 || a.N < 1 || a.nk < 1 || !a.a || !a.w) return hipErrorInvalidValue;
  if (!a.a2) a.nk1 = a.nk;
  const uintptr_t al = reinterpret_cast<uintptr_t>(a.y) | reinterpret_cast<uintptr_t>(a.yr) |
                       reinterpret_cast<uintptr_t>(a.bias);
  a.vec = al % 16 == 0 && a.ldy % 4 == 0 && a.sy % 4 == 0;
  switch (epi) {
    case kMmConv: return a.taps_kt > 0 ? mm_pick<kMmConv>(a, batch, n_cu, s) : hipErrorInvalidValue;
    case kMmPlain: return mm_pick<kMmPlain>(a, batch, n_cu, s);
    case kMmSwiglu: return mm_pick<kMmSwiglu>(a, batch, n_cu, s);
    case kMmGate: return a.taps_kt > 0 ? mm_pick<kMmGate>(a, batch, n_cu, s) : hipErrorInvalidValue;
    case kMmResSkip: return mm_pick<kMmResSkip>(a, batch, n_cu, s);
    case kMmQkv: return a.N % 192 == 0 ? mm_pick<kMmQkv>(a, batch, n_cu, s) : hipErrorInvalidValue;
  }
  return hipErrorInvalidValue;
}

size_t cfm_q_pieces(int B, int T, int H) { return (size_t)B * H * ((T + 63) / 64 * 2) * 4 * 128; }
size_t cfm_kv_pieces(int B, int T, int H) { return (size_t)B * H * ((T + 63) / 64 * 2) * flash_tile_pieces(2); }

hipError_t cfm_qkv_frag(const float *qkv, const float *rope_tab, int B, int T, int H, uint4 *qf, uint4 *kvf,
                        hipStream_t s) {
  const long n = 3L * B * H * ((T + 63) / 64 * 64) * 8;
  hipLaunchKernelGGL(qkv_frag_kernel, dim3(nblk(n)), dim3(256), 0, s, qkv, reinterpret_cast<const float2 *>(rope_tab),
                     B, T, H, reinterpret_cast<u32x4 *>(qf), reinterpret_cast<u32x4 *>(kvf));
  return hipGetLastError();
}

hipError_t cfm_attn_frag(const uint4 *qf, const uint4 *kvf, int B, int T, int H, uint4 *out, float *out_f, int n_cu,
                         hipStream_t s) {
  if (B < 1 || T < 1 || H < 1) return hipErrorInvalidValue;
  const int nt = (T + 31) / 32, bh = B * H;
  // One query tile a block, its four waves on a quarter of the keys each; or four query tiles,
  // one a wave, where those blocks cover the chip about once: the waves then share the key
  // tiles' loads (2 x 1033 frames: solve 58.6 against 59.3 ms; 2 x 2325: 114.0 against 108.3).
  const long b4 = (long)bh * ((nt + 3) / 4);
  const int wq = 2 * b4 > n_cu && b4 <= n_cu ? 4 : 1;
  const dim3 grid(bh, (nt + wq - 1) / wq), blk(256);
  const u32x4 *q = reinterpret_cast<const u32x4 *>(qf), *kv = reinterpret_cast<const u32x4 *>(kvf);
  u32x4 *o = reinterpret_cast<u32x4 *>(out);
  if (wq == 1) hipLaunchKernelGGL(attn_kernel<1>, grid, blk, 0, s, q, kv, H, T, H * kHd, o, out_f);
  else hipLaunchKernelGGL(attn_kernel<4>, grid, blk, 0, s, q, kv, H, T, H * kHd, o, out_f);
  return hipGetLastError();
}

}  // namespace itts
