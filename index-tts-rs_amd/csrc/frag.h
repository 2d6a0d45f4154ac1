// Operands of v_mfma_f32_32x32x16_{f16, bf16} kept in memory in fragment order, and the
// attention loop that runs on them (gfx950, wave64).
//
// A matrix X [rows][K] that a product reads as an MFMA operand is stored as planes of 16-bit
// values in blocks of 32 rows x 16 K: lane l of the operand holds row (l & 31), K values
// 8 (l >> 5) .. +7, so a block's plane is 64 pieces of 16 bytes in lane order (1 KiB) and
// an operand load is one fully coalesced 16-byte load per lane straight into registers: no
// LDS staging, no barrier, and any number of K steps in flight.
//
// Planes: fp16 hi/lo pairs (~22 bits, magnitudes below 131008, an absolute 2^-25 at the small
// end), or bf16 triples, which hold an fp32 value's 24 bits over its whole range.
#pragma once

#include <algorithm>

#include "common.h"

namespace itts {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2v __attribute__((ext_vector_type(2)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

#define ITTS_MFMA16 __builtin_amdgcn_mfma_f32_32x32x16_f16
#define ITTS_MFMABF __builtin_amdgcn_mfma_f32_32x32x16_bf16

// 16-byte piece of (row, 8-value chunk k8 of K), hi plane; the lo plane's is 64 pieces on.
// nk: K steps of 16 that a row block holds.
__host__ __device__ inline size_t frag_piece(long row, int k8, int nk) {
  return (((size_t)(row >> 5) * nk + (k8 >> 1)) * 2) * 64 + (size_t)((k8 & 1) * 32 + (row & 31));
}

__device__ __forceinline__ void split8(const float v[8], u32x4 &hi, u32x4 &lo) {
#pragma unroll
  for (int j = 0; j < 4; j++) {
    uint32_t h, l;
    split_f16x2(v[2 * j], v[2 * j + 1], h, l);
    hi[j] = h;
    lo[j] = l;
  }
}

// v = p[0] + p[1] + p[2] (each plane the rounding of what the planes before it leave).  An
// infinity or NaN stays one in plane 0.
__device__ __forceinline__ void split8_bf16(const float v[8], u32x4 (&p)[3]) {
#pragma unroll
  for (int j = 0; j < 4; j++) {
    f32x2e a = {v[2 * j], v[2 * j + 1]};
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const bf16x2v h = __builtin_convertvector(a, bf16x2v);
      p[i][j] = __builtin_bit_cast(uint32_t, h);
      a -= __builtin_convertvector(h, f32x2e);
    }
  }
}

// The two operand forms: planes of an activation operand, its split, one MFMA of two planes.
struct F16Pairs {
  typedef f16x8 V;
  static constexpr int N = 2;
  static __device__ __forceinline__ floatx16 mma(V a, V b, floatx16 c) { return ITTS_MFMA16(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ void split(const float v[8], u32x4 (&p)[N]) { split8(v, p[0], p[1]); }
};
struct Bf16Triples {
  typedef bf16x8 V;
  static constexpr int N = 3;
  static __device__ __forceinline__ floatx16 mma(V a, V b, floatx16 c) { return ITTS_MFMABF(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ void split(const float v[8], u32x4 (&p)[N]) { split8_bf16(v, p); }
};
// c + a b over operands of NA and T::N planes: the products of planes whose orders add up to
// less than T::N (the others lie below the last plane's rounding).  Of triples the small products
// come first, so that a sum that starts at zero rounds them at their own magnitude.
template <class T, int NA>
__device__ __forceinline__ floatx16 mma_planes(const u32x4 (&a)[NA], const u32x4 (&b)[T::N], floatx16 c) {
  auto mma = [&](int i, int j) __attribute__((always_inline)) {
    c = T::mma(__builtin_bit_cast(typename T::V, a[i]), __builtin_bit_cast(typename T::V, b[j]), c);
  };
  if constexpr (T::N == 2) {
#pragma unroll
    for (int i = 0; i < NA; i++)
#pragma unroll
      for (int j = 0; j < 2 - i; j++) mma(i, j);
  } else {
#pragma unroll
    for (int o = T::N - 1; o >= 0; o--)
#pragma unroll
      for (int i = 0; i < NA && i <= o; i++) mma(i, o - i);
  }
  return c;
}

// Exchanges v with lane ^ 32 (one VALU swap, no LDS round trip).
__device__ __forceinline__ float other_half(float v, int lane) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(lane < 32 ? r[1] : r[0]);
}

// ---- a product block's partial tiles ------------------------------------------------------
// Row parts (of 8 = rows x columns) the XCDs divide the tile grid into: the split whose XCDs
// read the fewest operand bytes.  A part whose operands fit its L2 reads them once; a larger
// one reads, for every ~64 tiles in flight, the row tiles and the column tiles they span.
// (4650 x 1024 x 2560: 78 us at 2 x 4, 84 at 8 x 1; 2066 x 512 x 512: 10.6 at 4 x 2, 12.6 at
// 1 x 8, which the plain tile order amounts to.)
inline int xcd_rows(int nM, int nN, double a_tile, double w_tile) {
  int best = 1;
  double least = 1e300;
  for (int gm = 1; gm <= 8; gm *= 2) {
    const int gn = 8 / gm, pm = (nM + gm - 1) / gm, pn = (nN + gn - 1) / gn;
    double bytes = pm * a_tile + pn * w_tile;
    if (bytes > 3e6)
      bytes = std::max(bytes, pm * pn / 64.0 * (std::max(1.0, 64.0 / pn) * a_tile + std::min(pn, 64) * w_tile));
    if (bytes < least) least = bytes, best = gm;
  }
  return best;
}

// The TM x TN MFMA tiles of wave kq of KS that split K go to LDS (red: KL tiles of BM rows, LD
// floats apart): with KS > KL the upper half of the waves first, then the lower half adds its own
// to what it finds, so that half the tiles' LDS does.  h = lane >> 5, r31 = lane & 31.
template <int TM, int TN, int KS, int KL, int BM, int LD>
__device__ __forceinline__ void parts_to_lds(float *red, const floatx16 (&acc)[TM][TN], int kq, int h, int r31) {
  auto part = [&](int k) __attribute__((always_inline)) { return red + (size_t)k * BM * LD; };
  auto place = [&](int i, int j, int e) __attribute__((always_inline)) {
    return (i * 32 + (e >> 2) * 8 + h * 4 + (e & 3)) * LD + j * 32 + r31;
  };
  if constexpr (KS > KL) {
    if (kq >= KL) {
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
          for (int e = 0; e < 16; e++) part(kq - KL)[place(i, j, e)] = acc[i][j][e];
    }
    __syncthreads();
  }
  if (kq < KL) {
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int e = 0; e < 16; e++) {
          float *t = part(kq) + place(i, j, e);
          *t = KS > KL ? acc[i][j][e] + *t : acc[i][j][e];
        }
  }
  __syncthreads();
}

// Eight columns of a tile row, the parts added in order.
template <int KL, int BM, int LD>
__device__ __forceinline__ void parts_row8(const float *red, int row, int col, float v[8]) {
#pragma unroll
  for (int q = 0; q < 2; q++) {
    float4 s = *reinterpret_cast<const float4 *>(red + (size_t)row * LD + col + 4 * q);
#pragma unroll
    for (int k = 1; k < KL; k++) {
      const float4 p = *reinterpret_cast<const float4 *>(red + ((size_t)k * BM + row) * LD + col + 4 * q);
      s.x += p.x, s.y += p.y, s.z += p.z, s.w += p.w;
    }
    v[4 * q] = s.x, v[4 * q + 1] = s.y, v[4 * q + 2] = s.z, v[4 * q + 3] = s.w;
  }
}

// ---- attention over key tiles of 32, one wave for 32 queries ----------------------------
// The scores are formed transposed, S^T = K Q^T: a lane then holds 16 keys of one query, so
// the softmax needs no cross-lane reduction but one exchange between the wave's halves, and
// the probabilities are already the B operand of O^T = V^T P^T (registers 8 kk .. 8 kk + 7
// are the keys of K step kk) with no LDS round trip.  V^T's fragments hold their keys in that
// order: position 8 h + 4 j2 + b of a 16-key step is key 8 j2 + 4 h + b.
//
// A key tile holds 8 fragments (4 K steps of K rows over the 64 dims; 2 dim tiles x 2 key
// steps of V^T) of NP planes each: kFlashFrags * NP KiB, contiguous.  Pairs have two planes;
// triples three, or one where the rows are bf16 (the plane is the value itself, whatever its
// magnitude, infinities and NaN with it).
constexpr int kFlashFrags = 8;
__host__ __device__ inline size_t flash_tile_pieces(int np) { return (size_t)kFlashFrags * np * 64; }
// position of key t (mod 16) within V^T's 16-key step
__host__ __device__ inline int flash_key_pos(int t) { return ((t >> 2) & 1) * 8 + ((t >> 3) & 1) * 4 + (t & 3); }

struct FlashState {
  float m, l;      // reference exponent and this lane's share (its half's keys) of the denominator
  floatx16 O[2];   // O^T: column = query (lane & 31), rows 8 (i >> 2) + 4 (lane >> 5) + (i & 3) of each 32 dims
};

__device__ __forceinline__ void flash_init(FlashState &st) {
  st.m = -3.0e38f;
  st.l = 0.0f;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    st.O[0][i] = 0.0f;
    st.O[1][i] = 0.0f;
  }
}

// Key tiles [t0, t1) at kv (piece index of tile 0 of this head, lane added); q is scaled so
// that a score's exponential is 2^s.  mask(tile, S) sets scores of masked keys to -inf.  The
// exponent reference m is raised only when some score passes it by more than 2^8: until then
// probabilities up to 2^8 are carried, in the same relative precision, and the rescaling of
// O is skipped.  (A masked key's V row still meets a probability of zero: if it is not finite,
// the rows that share its tile become NaN too.)
template <class T, int NP, class Mask>
__device__ __forceinline__ void flash_tiles(const u32x4 *kv, int t0, int t1, const u32x4 (&q)[4][T::N], Mask mask,
                                            FlashState &st) {
  if (t0 >= t1) return;
  u32x4 kf[4][NP], vf[4][NP];
  auto load_k = [&](int t) __attribute__((always_inline)) {
    const u32x4 *p = kv + (size_t)t * flash_tile_pieces(NP);
#pragma unroll
    for (int f = 0; f < 4; f++)
#pragma unroll
      for (int pl = 0; pl < NP; pl++) kf[f][pl] = p[(f * NP + pl) * 64];
  };
  auto load_v = [&](int t) __attribute__((always_inline)) {
    const u32x4 *p = kv + (size_t)t * flash_tile_pieces(NP) + 4 * NP * 64;
#pragma unroll
    for (int f = 0; f < 4; f++)
#pragma unroll
      for (int pl = 0; pl < NP; pl++) vf[f][pl] = p[(f * NP + pl) * 64];
  };
  load_k(t0);
  load_v(t0);
  for (int t = t0; t < t1; t++) {
    floatx16 S;
#pragma unroll
    for (int i = 0; i < 16; i++) S[i] = 0.0f;
#pragma unroll
    for (int kk = 0; kk < 4; kk++) S = mma_planes<T, NP>(kf[kk], q[kk], S);
    // the next tile's K into the registers just read (the last tile's again at the end)
    load_k(min(t + 1, t1 - 1));
    mask(t, S);
    float tmax = fmaxf(S[0], S[1]);
#pragma unroll
    for (int i = 2; i < 16; i++) tmax = fmaxf(tmax, S[i]);
    if (__any(tmax > st.m + 8.0f)) {
      const float mn = fmaxf(st.m, fmaxf(tmax, other_half(tmax, threadIdx.x & 63)));
      const float corr = __builtin_amdgcn_exp2f(st.m - mn);
      st.m = mn;
      st.l *= corr;
#pragma unroll
      for (int i = 0; i < 16; i++) {
        st.O[0][i] *= corr;
        st.O[1][i] *= corr;
      }
    }
    float p[16];
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; i++) {
      p[i] = __builtin_amdgcn_exp2f(S[i] - st.m);
      sum += p[i];
    }
    st.l += sum;
#pragma unroll
    for (int kk = 0; kk < 2; kk++) {
      u32x4 pp[T::N];
      T::split(p + 8 * kk, pp);
#pragma unroll
      for (int dt = 0; dt < 2; dt++) st.O[dt] = mma_planes<T, NP>(vf[dt * 2 + kk], pp, st.O[dt]);
    }
    load_v(min(t + 1, t1 - 1));
  }
}

// The waves of a block that share queries (wave g of WK took the keys' part g) merge their
// states through LDS (buf: WK x 2112 floats per query tile); wave 0 of the group returns
// with O and the full denominator.  Every thread of the block calls it.
template <int WK>
__device__ __forceinline__ void flash_merge(FlashState &st, float *buf, int g, int lane) {
  st.l += other_half(st.l, lane);
  if constexpr (WK > 1) {
    float *mine = buf + g * 2112;
    if (g > 0) {
#pragma unroll
      for (int i = 0; i < 16; i++) {
        mine[i * 64 + lane] = st.O[0][i];
        mine[(16 + i) * 64 + lane] = st.O[1][i];
      }
      if (lane < 32) {
        mine[2048 + lane] = st.m;
        mine[2080 + lane] = st.l;
      }
    }
    __syncthreads();
    if (g == 0) {
      float mg[WK], M = st.m;
#pragma unroll
      for (int j = 1; j < WK; j++) {
        mg[j] = buf[j * 2112 + 2048 + (lane & 31)];
        M = fmaxf(M, mg[j]);
      }
      const float f0 = __builtin_amdgcn_exp2f(st.m - M);
      st.l *= f0;
#pragma unroll
      for (int i = 0; i < 16; i++) {
        st.O[0][i] *= f0;
        st.O[1][i] *= f0;
      }
#pragma unroll
      for (int j = 1; j < WK; j++) {
        const float *o = buf + j * 2112;
        const float f = __builtin_amdgcn_exp2f(mg[j] - M);
        st.l += o[2080 + (lane & 31)] * f;
#pragma unroll
        for (int i = 0; i < 16; i++) {
          st.O[0][i] += o[i * 64 + lane] * f;
          st.O[1][i] += o[(16 + i) * 64 + lane] * f;
        }
      }
      st.m = M;
    }
  }
}

}  // namespace itts
