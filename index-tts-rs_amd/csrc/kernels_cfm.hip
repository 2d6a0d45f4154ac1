// Stage-2 CFM DiT estimator kernels for gfx950 (crates/core/src/models/cfm.rs) other than its
// MFMA products: the few-row fp32 FMA product (one wave per output column) for the per-batch
// conditioning projections and forwards of under 64 rows, the timestep frequency embedding, the
// row and elementwise kernels of those small forwards, and the Euler / classifier-free-guidance
// update.  Activations are [B][T][C] row-major fp32.
#include "kernels.h"

namespace itts {

namespace {

constexpr int kHd = 64;          // head dimension (cfm.rs:42)
constexpr int kFreqHalf = 128;   // TimestepEmbedder: 128 frequencies (cfm.rs:115-121)

__device__ inline float silu(float x) { return x / (1.0f + expf(-x)); }
__device__ inline float sigm(float x) { return 1.0f / (1.0f + expf(-x)); }

// Rope inverse frequency of pair k (compute_rope_freqs, cfm.rs:88-92).
__device__ inline float rope_inv(int k) { return 1.0f / powf(10000.0f, (float)(2 * k) / (float)kHd); }

// Block sum over 256 threads; red holds 8 floats.
__device__ inline float block_sum256(float v, float *red) {
  v = wave64_sum_dpp(v);
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[w] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

// emb[b] = [cos(t_b f_k), sin(t_b f_k)], f_k = 1000 exp(-ln(10000) k / 128) (cfm.rs:141-146)
__global__ void temb_kernel(const float *t, int B, float *emb) {
  const int b = blockIdx.x, k = threadIdx.x;
  if (b >= B || k >= kFreqHalf) return;
  const float f = 1000.0f * expf(-logf(10000.0f) * (float)k / (float)kFreqHalf);
  const float a = t[b] * f;
  emb[b * 2 * kFreqHalf + k] = cosf(a);
  emb[b * 2 * kFreqHalf + kFreqHalf + k] = sinf(a);
}

__global__ void silu_kernel(const float *x, float *y, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = silu(x[i]);
}

// C[r][c] = bias[c] for r < rows, c < cols (rows ldc apart)
__global__ void bias_rows_kernel(float *C, int ldc, const float *bias, int rows, int cols) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long)rows * cols) return;
  const int r = (int)(i / cols), c = (int)(i % cols);
  C[(size_t)r * ldc + c] = bias[c];
}

// AdaLn::forward (cfm.rs:173-182) on row r = b*T + t: y = w_b * (x * rsqrt(mean(x^2) + 1e-5)
// * norm_w) + b_b, (w_b, b_b) = mod[b][0..d), mod[b][d..2d).  One 256-thread block per row.
__global__ __launch_bounds__(256) void adaln_kernel(const float *x, float *y, int T, int d, const float *mod,
                                                    int ld_mod, const float *norm_w) {
  __shared__ float red[8];
  const int r = blockIdx.x, b = r / T;
  const float *xr = x + (size_t)r * d;
  float s = 0.0f;
  for (int i = threadIdx.x; i < d; i += 256) s += xr[i] * xr[i];
  s = block_sum256(s, red);
  const float rs = 1.0f / sqrtf(s / (float)d + 1e-5f);
  const float *w = mod + (size_t)b * ld_mod, *bb = w + d;
  for (int i = threadIdx.x; i < d; i += 256) y[(size_t)r * d + i] = w[i] * (xr[i] * rs * norm_w[i]) + bb[i];
}

// adaln_kernel with one wave per row for d = 256 * NV: lane l holds columns 256 j + 4 l ..
// + 3 of pass j in registers, the mean square is a DPP wave sum (no LDS, no barrier).
template <int NV>
__global__ __launch_bounds__(256) void adaln_wave_kernel(const float *x, float *y, int R, int T, int d,
                                                         const float *mod, int ld_mod, const float *norm_w) {
  const int lane = threadIdx.x & 63, r = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= R) return;  // whole waves leave together
  const int b = r / T;
  const float4 *xr = reinterpret_cast<const float4 *>(x + (size_t)r * d);
  const float4 *w = reinterpret_cast<const float4 *>(mod + (size_t)b * ld_mod);
  const float4 *bb = reinterpret_cast<const float4 *>(mod + (size_t)b * ld_mod + d);
  const float4 *nw = reinterpret_cast<const float4 *>(norm_w);
  // the row, its batch's modulation and the norm weight all loaded before the reduction
  // (one memory round trip, not two)
  float4 v[NV], wv[NV], bv[NV], nv[NV];
#pragma unroll
  for (int j = 0; j < NV; j++) {
    const int c = 64 * j + lane;
    v[j] = xr[c];
    wv[j] = w[c];
    bv[j] = bb[c];
    nv[j] = nw[c];
  }
  float s = 0.0f;
#pragma unroll
  for (int j = 0; j < NV; j++) s += (v[j].x * v[j].x + v[j].y * v[j].y) + (v[j].z * v[j].z + v[j].w * v[j].w);
  const float rs = 1.0f / sqrtf(wave64_sum_dpp(s) / (float)d + 1e-5f);
  float4 *yr = reinterpret_cast<float4 *>(y + (size_t)r * d);
#pragma unroll
  for (int j = 0; j < NV; j++) {
    const int c = 64 * j + lane;
    const float4 wj = wv[j], bj = bv[j], nj = nv[j];
    yr[c] = make_float4(wj.x * (v[j].x * rs * nj.x) + bj.x, wj.y * (v[j].y * rs * nj.y) + bj.y,
                        wj.z * (v[j].z * rs * nj.z) + bj.z, wj.w * (v[j].w * rs * nj.w) + bj.w);
  }
}

// FinalLayer norm (cfm.rs:605-609): layer_norm(h, eps 1e-6, no affine) * (1 + scale_b) +
// shift_b, (shift_b, scale_b) = mod[b][0..d), mod[b][d..2d).
__global__ __launch_bounds__(256) void final_norm_kernel(const float *x, float *y, int T, int d, const float *mod) {
  __shared__ float red[8];
  const int r = blockIdx.x, b = r / T;
  const float *xr = x + (size_t)r * d;
  float s = 0.0f;
  for (int i = threadIdx.x; i < d; i += 256) s += xr[i];
  const float mean = block_sum256(s, red) / (float)d;
  float q = 0.0f;
  for (int i = threadIdx.x; i < d; i += 256) {
    const float v = xr[i] - mean;
    q += v * v;
  }
  q = block_sum256(q, red);
  const float rstd = 1.0f / sqrtf(q / (float)d + 1e-6f);
  const float *shift = mod + (size_t)b * 2 * d, *scale = shift + d;
  for (int i = threadIdx.x; i < d; i += 256)
    y[(size_t)r * d + i] = ((xr[i] - mean) * rstd) * (1.0f + scale[i]) + shift[i];
}

// Rope table (compute_rope_freqs, cfm.rs:73-101): tab[t][k] = (cos, sin) of t * inv_freq(k),
// k < 32, computed once per sequence length.
__global__ void rope_table_kernel(int T, float2 *tab) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= T * (kHd / 2)) return;
  const int t = i / (kHd / 2), k = i % (kHd / 2);
  const float a = (float)t * rope_inv(k);
  tab[i] = make_float2(cosf(a), sinf(a));
}

// SwiGLU (cfm.rs:306-311): out[r][i] = silu(gu[r][i]) * gu[r][F + i]
__global__ void swiglu_kernel(const float *gu, int R, int F, float *out) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long)R * F) return;
  const int r = (int)(i / F), c = (int)(i % F);
  out[i] = silu(gu[(size_t)r * 2 * F + c]) * gu[(size_t)r * 2 * F + F + c];
}

// WaveNet gated activation (cfm.rs:379-391): acts = conv + in_b + g_b; act = tanh(acts[:d]) *
// sigmoid(acts[d:]); g rows ld_g apart per batch.
__global__ void gate_kernel(const float *acts, const float *in_b, const float *g, int ld_g, int R, int T, int d,
                            float *act) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long)R * d) return;
  const int r = (int)(i / d), c = (int)(i % d), b = r / T;
  const float *ar = acts + (size_t)r * 2 * d, *gb = g + (size_t)b * ld_g;
  const float a = ar[c] + in_b[c] + gb[c];
  const float s = ar[d + c] + in_b[d + c] + gb[d + c];
  act[i] = tanhf(a) * sigm(s);
}

// WaveNet residual / skip (cfm.rs:392-405): rs rows of width rso (+ rs_b); not last: h +=
// rs[:d], out += rs[d:]; last: out += rs (first: out = rs).
__global__ void res_skip_kernel(const float *rs, const float *rs_b, int last, int first, int R, int d, float *h,
                                float *out) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long)R * d) return;
  const int r = (int)(i / d), c = (int)(i % d);
  const float old = first ? 0.0f : out[i];
  if (last) {
    out[i] = old + (rs[(size_t)r * d + c] + rs_b[c]);
  } else {
    h[i] += rs[(size_t)r * 2 * d + c] + rs_b[c];
    out[i] = old + (rs[(size_t)r * 2 * d + d + c] + rs_b[d + c]);
  }
}

// Euler step input (cfm.rs:727-731): x = x * mask (zero over the first T_ref frames); x_t =
// [x, x] transposed to [2][T][C], also the first C columns of both merged rows.
__global__ void euler_prep_kernel(float *x, int C, int T, int T_ref, float *xt, float *merged, int MD) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long)C * T) return;
  const int c = (int)(i / T), t = (int)(i % T);
  float v = x[i];
  if (t < T_ref) {
    v = v * 0.0f;
    x[i] = v;
  }
  for (int b = 0; b < 2; b++) {
    xt[((size_t)b * T + t) * C + c] = v;
    merged[((size_t)b * T + t) * MD + c] = v;
  }
}

// Euler update with guidance (cfm.rs:735-745): x += dt * (pos * (1 + cfg) - neg * cfg), or dt *
// pos when cfg <= 0; v [2][T][C].
__global__ void euler_update_kernel(float *x, const float *v, int C, int T, float dt, float cfg) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long)C * T) return;
  const int c = (int)(i / T), t = (int)(i % T);
  const float pos = v[(size_t)t * C + c], neg = v[((size_t)T + t) * C + c];
  const float g = cfg > 0.0f ? pos * (1.0f + cfg) - neg * cfg : pos;
  x[i] = x[i] + g * dt;
}

// Static CFG tail of the merged input (cfm.rs:682-711): columns [C, 2C) = prompt mel (row 0,
// frames < T_ref), [2C + d, 2C + d + S) = style (row 0); zeros elsewhere (pre-cleared).
__global__ void static_tail_kernel(float *merged, int MD, int C, int d, int S, int T, const float *ref_mel, int T_ref,
                                   const float *style) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long)T * (C + S)) return;
  const int t = (int)(i / (C + S)), j = (int)(i % (C + S));
  float *row = merged + (size_t)t * MD;  // batch row 0
  if (j < C) {
    if (t < T_ref) row[C + j] = ref_mel[(size_t)j * T_ref + t];
  } else {
    row[2 * C + d + (j - C)] = style[j - C];
  }
}

// v [B][T][C] -> out [B][C][T]
__global__ void transpose_tc_kernel(const float *v, int B, int T, int C, float *out) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long)B * T * C) return;
  const int b = (int)(i / ((long)T * C)), rem = (int)(i % ((long)T * C)), t = rem / C, c = rem % C;
  out[((size_t)b * C + c) * T + t] = v[i];
}

// Few-row product y[z][m][n] = sum_k A[z][m][k] W[z][n][k] + beta y[z][m][n] in fp32 FMAs:
// the per-batch timestep / AdaLN / WaveNet-conditioning projections (2 rows, the CFG pair)
// and forwards of fewer than 64 rows.  One wave per output column n streams W's row n once
// (coalesced, VEC floats per lane) against MT rows of A (L2-resident); lane partial sums
// meet in a DPP reduction.  Block: 4 waves = 4 columns; grid (N/4, M/MT, batch).
template <int MT, int VEC>
__global__ __launch_bounds__(256) void rows_gemm_kernel(const float *__restrict__ A, int lda, long sa,
                                                        const float *__restrict__ W, int ldw, long sw, float *y,
                                                        int ldy, long sy, int M, int N, int K, float beta,
                                                        const float *bias) {
  const int lane = threadIdx.x & 63;
  const int n = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (n >= N) return;
  const int m0 = blockIdx.y * MT, z = blockIdx.z;
  const float *w = W + z * sw + (size_t)n * ldw;
  const float *a[MT];
#pragma unroll
  for (int j = 0; j < MT; j++) a[j] = A + z * sa + (size_t)(m0 + j < M ? m0 + j : m0) * lda;
  float acc[MT];
#pragma unroll
  for (int j = 0; j < MT; j++) acc[j] = 0.0f;
  if constexpr (VEC == 4) {
    for (int k = 4 * lane; k < K; k += 256) {
      const float4 wv = *reinterpret_cast<const float4 *>(w + k);
#pragma unroll
      for (int j = 0; j < MT; j++) {
        const float4 av = *reinterpret_cast<const float4 *>(a[j] + k);
        acc[j] = fmaf(av.x, wv.x, acc[j]);
        acc[j] = fmaf(av.y, wv.y, acc[j]);
        acc[j] = fmaf(av.z, wv.z, acc[j]);
        acc[j] = fmaf(av.w, wv.w, acc[j]);
      }
    }
  } else {
    for (int k = lane; k < K; k += 64) {
      const float wv = w[k];
#pragma unroll
      for (int j = 0; j < MT; j++) acc[j] = fmaf(a[j][k], wv, acc[j]);
    }
  }
#pragma unroll
  for (int j = 0; j < MT; j++) acc[j] = wave64_sum_dpp(acc[j]);
  if (lane < MT && m0 + lane < M) {
    float v = acc[0];
#pragma unroll
    for (int j = 1; j < MT; j++)
      if (lane == j) v = acc[j];
    float *dst = y + z * sy + (size_t)(m0 + lane) * ldy + n;
    if (bias) v = v + bias[n];
    *dst = beta != 0.0f ? v + beta * *dst : v;
  }
}

__global__ void fill_kernel(float *p, int n, float v) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

inline unsigned nblk(long n, int t = 256) { return (unsigned)((n + t - 1) / t); }

}  // namespace

hipError_t cfm_temb(const float *t, int B, float *emb, hipStream_t s) {
  hipLaunchKernelGGL(temb_kernel, dim3(B), dim3(kFreqHalf), 0, s, t, B, emb);
  return hipGetLastError();
}
hipError_t cfm_silu(const float *x, float *y, int n, hipStream_t s) {
  hipLaunchKernelGGL(silu_kernel, dim3(nblk(n)), dim3(256), 0, s, x, y, n);
  return hipGetLastError();
}
hipError_t cfm_bias_rows(float *C, int ldc, const float *bias, int rows, int cols, hipStream_t s) {
  hipLaunchKernelGGL(bias_rows_kernel, dim3(nblk((long)rows * cols)), dim3(256), 0, s, C, ldc, bias, rows, cols);
  return hipGetLastError();
}
hipError_t cfm_adaln(const float *x, float *y, int R, int T, int d, const float *mod, int ld_mod, const float *norm_w,
                     hipStream_t s) {
  // one wave per row when d = 256 or 512 and the modulation rows keep 16-byte alignment
  const bool wave = (d == 256 || d == 512) && ld_mod % 4 == 0;
  if (wave && d == 512)
    hipLaunchKernelGGL(adaln_wave_kernel<2>, dim3((R + 3) / 4), dim3(256), 0, s, x, y, R, T, d, mod, ld_mod, norm_w);
  else if (wave)
    hipLaunchKernelGGL(adaln_wave_kernel<1>, dim3((R + 3) / 4), dim3(256), 0, s, x, y, R, T, d, mod, ld_mod, norm_w);
  else
    hipLaunchKernelGGL(adaln_kernel, dim3(R), dim3(256), 0, s, x, y, T, d, mod, ld_mod, norm_w);
  return hipGetLastError();
}
hipError_t cfm_final_norm(const float *x, float *y, int R, int T, int d, const float *mod, hipStream_t s) {
  hipLaunchKernelGGL(final_norm_kernel, dim3(R), dim3(256), 0, s, x, y, T, d, mod);
  return hipGetLastError();
}
hipError_t cfm_rope_table(int T, float *tab, hipStream_t s) {
  hipLaunchKernelGGL(rope_table_kernel, dim3(nblk((long)T * (kHd / 2))), dim3(256), 0, s, T,
                     reinterpret_cast<float2 *>(tab));
  return hipGetLastError();
}
hipError_t cfm_rows_gemm(int batch, int M, int N, int K, const float *A, int lda, long sa, const float *W, int ldw,
                         long sw, float *y, int ldy, long sy, float beta, hipStream_t s, const float *bias) {
  if (batch < 1 || M < 1 || N < 1 || K < 1 || lda < K || ldw < K || ldy < N) return hipErrorInvalidValue;
  const bool v4 = K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && sa % 4 == 0 && sw % 4 == 0 &&
                  (reinterpret_cast<uintptr_t>(A) & 15) == 0 && (reinterpret_cast<uintptr_t>(W) & 15) == 0;
  const int mt = M <= 1 ? 1 : M <= 2 ? 2 : M <= 4 ? 4 : 8;
  const dim3 grid((N + 3) / 4, (M + mt - 1) / mt, batch);
#define ROWS_GEMM(MT, VEC)                                                                                        hipLaunchKernelGGL((rows_gemm_kernel<MT, VEC>), grid, dim3(256), 0, s, A, lda, sa, W, ldw, sw, y, ldy, sy, M, N,                      K, beta, bias)
  if (v4) {
    if (mt == 1) ROWS_GEMM(1, 4);
    else if (mt == 2) ROWS_GEMM(2, 4);
    else if (mt == 4) ROWS_GEMM(4, 4);
    else ROWS_GEMM(8, 4);
  } else {
    if (mt == 1) ROWS_GEMM(1, 1);
    else if (mt == 2) ROWS_GEMM(2, 1);
    else if (mt == 4) ROWS_GEMM(4, 1);
    else ROWS_GEMM(8, 1);
  }
#undef ROWS_GEMM
  return hipGetLastError();
}
hipError_t cfm_swiglu(const float *gu, int R, int F, float *out, hipStream_t s) {
  hipLaunchKernelGGL(swiglu_kernel, dim3(nblk((long)R * F)), dim3(256), 0, s, gu, R, F, out);
  return hipGetLastError();
}
hipError_t cfm_gate(const float *acts, const float *in_b, const float *g, int ld_g, int R, int T, int d, float *act,
                    hipStream_t s) {
  hipLaunchKernelGGL(gate_kernel, dim3(nblk((long)R * d)), dim3(256), 0, s, acts, in_b, g, ld_g, R, T, d, act);
  return hipGetLastError();
}
hipError_t cfm_res_skip(const float *rs, const float *rs_b, int last, int first, int R, int d, float *h, float *out,
                        hipStream_t s) {
  hipLaunchKernelGGL(res_skip_kernel, dim3(nblk((long)R * d)), dim3(256), 0, s, rs, rs_b, last, first, R, d, h, out);
  return hipGetLastError();
}
hipError_t cfm_euler_prep(float *x, int C, int T, int T_ref, float *xt, float *merged, int MD, hipStream_t s) {
  hipLaunchKernelGGL(euler_prep_kernel, dim3(nblk((long)C * T)), dim3(256), 0, s, x, C, T, T_ref, xt, merged, MD);
  return hipGetLastError();
}
hipError_t cfm_euler_update(float *x, const float *v, int C, int T, float dt, float cfg, hipStream_t s) {
  hipLaunchKernelGGL(euler_update_kernel, dim3(nblk((long)C * T)), dim3(256), 0, s, x, v, C, T, dt, cfg);
  return hipGetLastError();
}
hipError_t cfm_static_tail(float *merged, int MD, int C, int d, int S, int T, const float *ref_mel, int T_ref,
                           const float *style, hipStream_t s) {
  hipLaunchKernelGGL(static_tail_kernel, dim3(nblk((long)T * (C + S))), dim3(256), 0, s, merged, MD, C, d, S, T,
                     ref_mel, T_ref, style);
  return hipGetLastError();
}
hipError_t cfm_transpose_tc(const float *v, int B, int T, int C, float *out, hipStream_t s) {
  hipLaunchKernelGGL(transpose_tc_kernel, dim3(nblk((long)B * T * C)), dim3(256), 0, s, v, B, T, C, out);
  return hipGetLastError();
}
hipError_t cfm_fill(float *p, int n, float v, hipStream_t s) {
  hipLaunchKernelGGL(fill_kernel, dim3(nblk(n)), dim3(256), 0, s, p, n, v);
  return hipGetLastError();
}

}  // namespace itts
