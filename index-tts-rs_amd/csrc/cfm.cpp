// libitts_hip: the Stage-2 CFM DiT estimator and its Euler / classifier-free-guidance solver
// (crates/core/src/models/cfm.rs), the itts_cfm_* entry points of include/itts_hip.h.
//
// CfmDit::from_weights -> itts_cfm_create (tensors by checkpoint name, checked by element
// count), forward_merged -> itts_cfm_forward, solve_euler -> itts_cfm_solve_euler.  Forwards of
// 64 rows and more keep the residual stream in fp32 and hand every product its operands as
// fp16 hi/lo planes in MFMA fragment order (kernels_cfm_mm.hip); smaller ones, and operands
// whose widths are not multiples of 4, run the linears as fp32 FMA products
// (kernels_cfm.hip).  Layout: activations [B][T][C] row-major, the CFG pair as batch rows 0
// (conditioned) and 1 (unconditioned).
#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <utility>
#include <vector>

#include "../../include/itts_hip.h"
#include "kernels.h"

namespace itts {
itts_status set_error_text(itts_status st, const char *msg);  // runtime.cpp
}

namespace {

using namespace itts;

itts_status cerr(itts_status st, const char *fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  return set_error_text(st, buf);
}

#define CK(expr)                                                                                       \
  do {                                                                                                 \
    hipError_t e_ = (expr);                                                                            \
    if (e_ != hipSuccess) return cerr(ITTS_E_DEVICE, "HIP error %s at %s:%d", hipGetErrorName(e_), __FILE__, __LINE__); \
  } while (0)

constexpr int kFreqDim = 256;

struct Buf {
  float *p = nullptr;
  size_t n = 0;
  // the shape whose table or zero rows the buffer holds ((0, 0): none); lost with the memory
  std::pair<int, int> holds{0, 0};
  Buf() = default;
  Buf(const Buf &) = delete;
  Buf &operator=(const Buf &) = delete;
  Buf(Buf &&o) noexcept : p(o.p), n(o.n), holds(o.holds) { o.p = nullptr, o.n = 0, o.holds = {0, 0}; }
  ~Buf() {
    if (p) (void)hipFree(p);
  }
  hipError_t ensure(size_t count) {
    if (count <= n) return hipSuccess;
    holds = {0, 0};
    if (p) {
      hipError_t e = hipFree(p);
      p = nullptr;
      n = 0;
      if (e != hipSuccess) return e;
    }
    hipError_t e = hipMalloc(&p, count * sizeof(float));
    if (e == hipSuccess) n = count;
    return e;
  }
};

struct Block {
  const float *wqkv, *wo, *w13, *w2, *skip_w, *skip_b, *an_w, *fn_w;
};
struct WnLayer {
  const float *in_w, *in_b, *rs_w, *rs_b;
};

}  // namespace

struct itts_cfm {
  itts_cfm_config c{};
  hipStream_t s = nullptr;
  float *arena = nullptr;
  const float *cond_w, *cond_b, *merge_w, *merge_b;
  const float *te_w0[2], *te_b0[2], *te_w2[2], *te_b2[2];
  const float *ada_w, *ada_b, *tn_w;  // AdaLN projections packed [(2L+1)*2d][d]: layer i attn 2i, ffn 2i+1, final 2L
  const float *skl_w, *skl_b, *c1_w, *c1_b, *rp_w, *rp_b, *wc_w, *wc_b, *fa_w, *fa_b, *fl_w, *fl_b, *c2_w, *c2_b;
  std::vector<Block> L;
  std::vector<WnLayer> wn;
  // per-forward workspace (sized for R = B*T rows)
  Buf emb, th, t1, t2, st, mods, wng, fmod, tdev;
  Buf hA, hB, n, qkv, att, gu, act, xres, hw, acts, rs, oacc, v, rope;
  // fragment planes (16-byte pieces): norm / attention / FFN outputs, the block output a
  // long skip joins, the skips, merged and x_t inputs, x_res, WaveNet's padded input, Q, K / V
  Buf nP, attP, actP, curP, mP, xtP, xresP, hpP, qF, kvF;
  std::vector<Buf> skipP, skips;
  int n_cu = 0;  // compute units of the device (the launch rules' parameter)
  // solve / API staging
  Buf x, xt, merged, catc, refm, sty, io_a, io_b;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  float last_ms = -1.0f;
  // the weights' fragment planes, laid out at their first use, by (first row, halves
  // interleaved)
  std::map<std::pair<const float *, int>, uint4 *> wfrag;
  ~itts_cfm() {
    for (auto &kv : wfrag) (void)hipFree(kv.second);
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    if (arena) (void)hipFree(arena);
    if (s) (void)hipStreamDestroy(s);
  }
};

namespace {

constexpr int kMfmaRows = 64;  // forwards of fewer rows run their linears as fp32 FMA products

int steps16(int K) { return (K + 15) / 16; }
int round32(int n) { return (n + 31) / 32 * 32; }
uint4 *pieces(const Buf &b) { return reinterpret_cast<uint4 *>(b.p); }
size_t piece_floats(size_t n) { return 4 * n; }

// The fragment planes of weight W [N][ldw] (K values, plus K2 more at W + off2 as further K
// steps; halves interleaved when ilv > 0), made on the estimator's stream at their first use
// (the weights are constant while the estimator lives); nullptr on failure.
const uint4 *weight_frag(itts_cfm *m, const float *W, int ldw, int N, int K, int ilv = 0, int off2 = 0, int K2 = 0) {
  const auto key = std::make_pair(W, ilv);
  auto it = m->wfrag.find(key);
  if (it != m->wfrag.end()) return it->second;
  const int nk = steps16(K) + (K2 ? steps16(K2) : 0);
  const size_t bytes = cfm_frag_pieces(ilv ? 64L * ((ilv + 31) / 32) : N, nk) * sizeof(uint4);
  uint4 *p = nullptr;
  if (hipMalloc(&p, bytes) != hipSuccess) return nullptr;
  if (hipMemsetAsync(p, 0, bytes, m->s) != hipSuccess ||
      cfm_weight_frag(W, ldw, N, K, 0, nk, ilv, p, m->s) != hipSuccess ||
      (K2 && cfm_weight_frag(W + off2, ldw, N, K2, steps16(K), nk, ilv, p, m->s) != hipSuccess)) {
    (void)hipFree(p);
    return nullptr;
  }
  m->wfrag.emplace(key, p);
  return p;
}

// y[M][N] = A[M][K] W[N][K]^T (+ bias[n]) + beta y (row-major; W rows ldw apart) in fp32 FMAs
// on the estimator's stream: the per-batch timestep, AdaLN and WaveNet-conditioning
// projections, forwards of under kMfmaRows rows, and widths that are not multiples of 4.
hipError_t gemm(itts_cfm *m, int M, int N, int K, const float *A, int lda, const float *W, int ldw, float *y,
                int ldy, float beta, const float *bias = nullptr) {
  return itts::cfm_rows_gemm(1, M, N, K, A, lda, 0, W, ldw, 0, y, ldy, 0, beta, m->s, bias);
}

// A product over fragment planes: M rows of `a` (K values, ka K steps) by the planes w.
CfmMm mm_args(const uint4 *a, int K, const uint4 *w, int M, int N) {
  CfmMm g{};
  g.a = a;
  g.kt_a = g.nk = steps16(K);
  g.w = w;
  g.M = M;
  g.N = N;
  return g;
}

itts_status check_config(const itts_cfm_config &c) {
  if (c.n_heads < 1 || c.dim != 64 * c.n_heads || c.n_layers < 1 || c.inter < 1 || c.in_ch < 1 || c.style_dim < 0 ||
      c.wn_layers < 1 || c.wn_kernel < 1 || c.wn_kernel % 2 == 0 || c.dim > 8192 || c.inter > 65536)
    return cerr(ITTS_E_VALIDATION, "cfm config: unsupported shape (dim must be 64 * n_heads, wn_kernel odd)");
  return ITTS_OK;
}

// Pieces of one batch entry of WaveNet's padded input: the rows whole tiles of T read at every tap.
size_t hp_pieces(const itts_cfm_config &c, int T) {
  return cfm_frag_pieces((T + 127) / 128 * 128 + c.wn_kernel, c.dim / 16);
}
// The skip / merge products whose fp32 rows are not 16-byte aligned stay fp32 FMA products.
bool unaligned_skip(const itts_cfm_config &c) { return c.in_ch % 4 != 0 || (c.dim + c.in_ch) % 4 != 0; }
bool unaligned_merge(const itts_cfm_config &c) { return (2 * c.in_ch + c.dim + c.style_dim) % 4 != 0; }

itts_status ensure_rows(itts_cfm *m, int B, int T) {
  const itts_cfm_config &c = m->c;
  const size_t R = (size_t)B * T, d = c.dim, F = c.inter, NL = c.wn_layers;
  const size_t na = 2 * (size_t)c.n_layers + 1;
  CK(m->emb.ensure(B * kFreqDim));
  CK(m->th.ensure(B * d));
  CK(m->t1.ensure(B * d));
  CK(m->t2.ensure(B * d));
  CK(m->st.ensure(B * d));
  CK(m->mods.ensure(B * na * 2 * d));
  CK(m->wng.ensure(B * 2 * d * NL));
  CK(m->fmod.ensure(B * 2 * d));
  CK(m->tdev.ensure(B));
  CK(m->hA.ensure(R * d));
  CK(m->hB.ensure(R * d));
  CK(m->hw.ensure(R * d));
  CK(m->oacc.ensure(R * d));
  CK(m->v.ensure(R * c.in_ch));
  const int dk = (int)d / 16;
  CK(m->actP.ensure(piece_floats(cfm_frag_pieces(R, round32(F > d ? F : d) / 16))));
  CK(m->qF.ensure(piece_floats(cfm_q_pieces(B, T, c.n_heads))));
  CK(m->kvF.ensure(piece_floats(cfm_kv_pieces(B, T, c.n_heads))));
  const size_t hp = hp_pieces(c, T);
  CK(m->hpP.ensure(piece_floats(B * hp)));
  if (m->hpP.holds != std::make_pair(B, T)) {  // the convolution's padding rows, zero from here on
    m->hpP.holds = {0, 0};
    CK(hipMemsetAsync(m->hpP.p, 0, sizeof(uint4) * B * hp, m->s));
    m->hpP.holds = {B, T};
  }
  const bool few = R < kMfmaRows;
  if (few || unaligned_skip(c)) {
    CK(m->n.ensure(R * d));
    CK(m->xres.ensure(R * d));
  }
  if (few) {
    CK(m->qkv.ensure(R * 3 * d));
    CK(m->att.ensure(R * d));
    CK(m->gu.ensure(R * 2 * F));
    CK(m->act.ensure(R * (F > d ? F : d)));
    CK(m->acts.ensure(R * 2 * d));
    CK(m->rs.ensure(R * 2 * d));
    for (auto &b : m->skips) CK(b.ensure(R * d));
  } else {
    const size_t rows = piece_floats(cfm_frag_pieces(R, dk));
    // (a tile over one batch entry's rows reads up to 127 rows past them)
    CK(m->nP.ensure(piece_floats(cfm_frag_pieces(R + 128, dk))));
    for (Buf *b : {&m->attP, &m->curP, &m->xresP}) CK(b->ensure(rows));
    for (auto &b : m->skipP) CK(b.ensure(rows));
    CK(m->mP.ensure(piece_floats(cfm_frag_pieces(R, steps16(2 * c.in_ch + c.dim + c.style_dim)))));
    CK(m->xtP.ensure(piece_floats(cfm_frag_pieces(R, steps16(c.in_ch)))));
  }
  CK(m->rope.ensure((size_t)T * 64));
  if (m->rope.holds != std::make_pair(1, T)) {
    m->rope.holds = {0, 0};
    CK(cfm_rope_table(T, m->rope.p, m->s));
    m->rope.holds = {1, T};
  }
  return ITTS_OK;
}

// TimestepEmbedder::forward (cfm.rs:141-146) for embedder e on the device t [B] -> out [B][d]
itts_status timestep(itts_cfm *m, int e, int B, float *out) {
  const int d = m->c.dim;
  hipStream_t s = m->s;
  CK(cfm_temb(m->tdev.p, B, m->emb.p, s));
  CK(gemm(m, B, d, kFreqDim, m->emb.p, kFreqDim, m->te_w0[e], kFreqDim, m->th.p, d, 0.0f, m->te_b0[e]));
  CK(cfm_silu(m->th.p, m->th.p, B * d, s));
  CK(gemm(m, B, d, d, m->th.p, d, m->te_w2[e], d, out, d, 0.0f, m->te_b2[e]));
  return ITTS_OK;
}

// The U-ViT blocks, skip_linear and conv1 (cfm.rs:553-585) of at least kMfmaRows rows: residual
// stream fp32 in hA / hB, every product's operand as fragment planes; leaves x_res in xresP,
// WaveNet's input in hw (fp32) and hpP.
itts_status blocks_mfma(itts_cfm *m, const float *x_t, const float *merged, int B, int T) {
  const itts_cfm_config &c = m->c;
  const int d = c.dim, C = c.in_ch, MD = 2 * C + d + c.style_dim, R = B * T, Lc = c.n_layers, split = Lc / 2;
  const int na2 = (2 * Lc + 1) * 2 * d, dk = d / 16, F32 = round32(c.inter), pad = c.wn_kernel / 2;
  hipStream_t s = m->s;
#define WF(var, ...)                                                                                  \
  const uint4 *var = weight_frag(m, __VA_ARGS__);                                                     \
  if (!var) return cerr(ITTS_E_DEVICE, "out of device memory for the weights' operand planes")
  auto mm = [&](const CfmMm &g, int epi, int batch) { return cfm_mm(g, epi, batch, m->n_cu, s); };
  float *cur = m->hA.p, *oth = m->hB.p;
  if (unaligned_merge(c)) {
    CK(gemm(m, R, d, MD, merged, MD, m->merge_w, MD, cur, d, 0.0f, m->merge_b));
  } else {
    WF(w, m->merge_w, MD, d, MD);
    CK(cfm_rows_frag(merged, MD, R, MD, steps16(MD), 0, pieces(m->mP), s));
    CfmMm g = mm_args(pieces(m->mP), MD, w, R, d);
    g.bias = m->merge_b;
    g.y = cur;
    g.ldy = d;
    CK(mm(g, kMmPlain, 1));
  }
  int nsk = 0;
  for (int i = 0; i < Lc; i++) {
    const Block &b = m->L[i];
    if (i > split && nsk > 0) {  // skip_in_linear([h, skip]): two operands along K
      WF(w, b.skip_w, 2 * d, d, 2 * d);
      CfmMm g = mm_args(pieces(m->curP), d, w, R, d);
      g.a2 = pieces(m->skipP[--nsk]);
      g.kt_a2 = g.nk1 = dk;
      g.nk = 2 * dk;
      g.bias = b.skip_b;
      g.y = oth;
      g.ldy = d;
      CK(mm(g, kMmPlain, 1));
      std::swap(cur, oth);
    }
    const float *mod_a = m->mods.p + (size_t)(2 * i) * 2 * d, *mod_f = m->mods.p + (size_t)(2 * i + 1) * 2 * d;
    CK(cfm_norm_frag(cur, R, T, d, mod_a, na2, b.an_w, false, pieces(m->nP), s));
    {
      WF(w, b.wqkv, d, 3 * d, d);
      CfmMm g = mm_args(pieces(m->nP), d, w, T, 3 * d);
      g.zr = T;
      g.o = pieces(m->qF);
      g.o2 = pieces(m->kvF);
      g.g = m->rope.p;
      CK(mm(g, kMmQkv, B));
    }
    CK(cfm_attn_frag(pieces(m->qF), pieces(m->kvF), B, T, c.n_heads, pieces(m->attP), nullptr, m->n_cu, s));
    {
      WF(w, b.wo, d, d, d);
      CfmMm g = mm_args(pieces(m->attP), d, w, R, d);
      g.y = cur;
      g.yr = cur;
      g.ldy = d;
      CK(mm(g, kMmPlain, 1));
    }
    CK(cfm_norm_frag(cur, R, T, d, mod_f, na2, b.fn_w, false, pieces(m->nP), s));
    {
      WF(w, b.w13, d, 2 * c.inter, d, c.inter);
      CfmMm g = mm_args(pieces(m->nP), d, w, R, F32);
      g.o = pieces(m->actP);
      g.kt_o = F32 / 16;
      CK(mm(g, kMmSwiglu, 1));
    }
    {  // hidden + ffn; the output's planes where a skip_in_linear reads them
      WF(w, b.w2, c.inter, d, c.inter);
      CfmMm g = mm_args(pieces(m->actP), c.inter, w, R, d);
      g.kt_a = F32 / 16;
      g.y = cur;
      g.yr = cur;
      g.ldy = d;
      if (i < split) g.o = pieces(m->skipP[nsk++]);
      else if (i + 1 < Lc && nsk > 0) g.o = pieces(m->curP);
      g.kt_o = dk;
      CK(mm(g, kMmPlain, 1));
    }
  }
  // transformer.norm, x_res = skip_linear([h, x_t]), h = conv1(x_res)
  const float *mod_n = m->mods.p + (size_t)(2 * Lc) * 2 * d;
  if (unaligned_skip(c)) {
    CK(cfm_adaln(cur, m->n.p, R, T, d, mod_n, na2, m->tn_w, s));
    CK(gemm(m, R, d, d, m->n.p, d, m->skl_w, d + C, m->xres.p, d, 0.0f, m->skl_b));
    CK(gemm(m, R, d, C, x_t, C, m->skl_w + d, d + C, m->xres.p, d, 1.0f));
    CK(cfm_rows_frag(m->xres.p, d, R, d, dk, 0, pieces(m->xresP), s));
  } else {
    CK(cfm_norm_frag(cur, R, T, d, mod_n, na2, m->tn_w, false, pieces(m->nP), s));
    CK(cfm_rows_frag(x_t, C, R, C, steps16(C), 0, pieces(m->xtP), s));
    WF(w, m->skl_w, d + C, d, d, 0, d, C);
    CfmMm g = mm_args(pieces(m->nP), d, w, R, d);
    g.a2 = pieces(m->xtP);
    g.kt_a2 = steps16(C);
    g.nk1 = dk;
    g.nk = dk + g.kt_a2;
    g.bias = m->skl_b;
    g.o = pieces(m->xresP);
    g.kt_o = dk;
    CK(mm(g, kMmPlain, 1));
  }
  WF(w, m->c1_w, d, d, d);
  CfmMm g = mm_args(pieces(m->xresP), d, w, R, d);
  g.bias = m->c1_b;
  g.y = m->hw.p;
  g.ldy = d;
  g.T = T;
  g.o = pieces(m->hpP);
  g.so = (long)hp_pieces(c, T);
  g.o_row0 = pad;
  g.kt_o = dk;
  CK(mm(g, kMmPlain, 1));
  return ITTS_OK;
}

// The same of fewer rows: fp32 activations, fp32 FMA linears; x_res in xres, WaveNet's input in hw.
itts_status blocks_few(itts_cfm *m, const float *x_t, const float *merged, int B, int T) {
  const itts_cfm_config &c = m->c;
  const int d = c.dim, F = c.inter, C = c.in_ch, MD = 2 * C + d + c.style_dim, R = B * T, Lc = c.n_layers;
  const int split = Lc / 2, na2 = (2 * Lc + 1) * 2 * d;
  hipStream_t s = m->s;
  float *cur = m->hA.p, *oth = m->hB.p;
  CK(gemm(m, R, d, MD, merged, MD, m->merge_w, MD, cur, d, 0.0f, m->merge_b));
  int nsk = 0;
  for (int i = 0; i < Lc; i++) {
    const Block &b = m->L[i];
    if (i > split && nsk > 0) {  // skip_in_linear([h, skip]) as two accumulating products
      const float *sk = m->skips[--nsk].p;
      CK(gemm(m, R, d, d, cur, d, b.skip_w, 2 * d, oth, d, 0.0f, b.skip_b));
      CK(gemm(m, R, d, d, sk, d, b.skip_w + d, 2 * d, oth, d, 1.0f));
      std::swap(cur, oth);
    }
    const float *mod_a = m->mods.p + (size_t)(2 * i) * 2 * d, *mod_f = m->mods.p + (size_t)(2 * i + 1) * 2 * d;
    CK(cfm_adaln(cur, m->n.p, R, T, d, mod_a, na2, b.an_w, s));
    CK(gemm(m, R, 3 * d, d, m->n.p, d, b.wqkv, d, m->qkv.p, 3 * d, 0.0f));
    CK(cfm_qkv_frag(m->qkv.p, m->rope.p, B, T, c.n_heads, pieces(m->qF), pieces(m->kvF), s));
    CK(cfm_attn_frag(pieces(m->qF), pieces(m->kvF), B, T, c.n_heads, nullptr, m->att.p, m->n_cu, s));
    CK(gemm(m, R, d, d, m->att.p, d, b.wo, d, cur, d, 1.0f));
    CK(cfm_adaln(cur, m->n.p, R, T, d, mod_f, na2, b.fn_w, s));
    CK(gemm(m, R, 2 * F, d, m->n.p, d, b.w13, d, m->gu.p, 2 * F, 0.0f));
    CK(cfm_swiglu(m->gu.p, R, F, m->act.p, s));
    CK(gemm(m, R, d, F, m->act.p, F, b.w2, F, cur, d, 1.0f));  // hidden + ffn
    if (i < split) {
      CK(hipMemcpyAsync(m->skips[nsk++].p, cur, sizeof(float) * R * d, hipMemcpyDeviceToDevice, s));
    }
  }
  CK(cfm_adaln(cur, m->n.p, R, T, d, m->mods.p + (size_t)(2 * Lc) * 2 * d, na2, m->tn_w, s));
  CK(gemm(m, R, d, d, m->n.p, d, m->skl_w, d + C, m->xres.p, d, 0.0f, m->skl_b));
  CK(gemm(m, R, d, C, x_t, C, m->skl_w + d, d + C, m->xres.p, d, 1.0f));
  CK(gemm(m, R, d, d, m->xres.p, d, m->c1_w, d, m->hw.p, d, 0.0f, m->c1_b));
  return ITTS_OK;
}

// forward_merged (cfm.rs:545-617) on device inputs x_t [B][T][C], merged [B][T][MD] and the
// timesteps already in m->tdev; the velocity lands in m->v as [B][T][C].
itts_status forward(itts_cfm *m, const float *x_t, const float *merged, int B, int T) {
  const itts_cfm_config &c = m->c;
  const int d = c.dim, C = c.in_ch, NL = c.wn_layers, K = c.wn_kernel, pad = K / 2, R = B * T, Lc = c.n_layers;
  const int na2 = (2 * Lc + 1) * 2 * d, dk = d / 16;  // na2: packed AdaLN modulation width
  const bool few = R < kMfmaRows;
  hipStream_t s = m->s;
  if (itts_status st = ensure_rows(m, B, T)) return st;
  // conditioning vectors: t1, t2, every AdaLN's (w, b), WaveNet's per-layer g, FinalLayer's (shift, scale)
  if (itts_status st = timestep(m, 0, B, m->t1.p)) return st;
  if (itts_status st = timestep(m, 1, B, m->t2.p)) return st;
  CK(gemm(m, B, na2, d, m->t1.p, d, m->ada_w, d, m->mods.p, na2, 0.0f, m->ada_b));
  CK(gemm(m, B, 2 * d * NL, d, m->t2.p, d, m->wc_w, d, m->wng.p, 2 * d * NL, 0.0f, m->wc_b));
  CK(cfm_silu(m->t1.p, m->st.p, B * d, s));
  CK(gemm(m, B, 2 * d, d, m->st.p, d, m->fa_w, d, m->fmod.p, 2 * d, 0.0f, m->fa_b));
  if (itts_status st = few ? blocks_few(m, x_t, merged, B, T) : blocks_mfma(m, x_t, merged, B, T)) return st;
  auto mm = [&](const CfmMm &g, int epi, int batch) { return cfm_mm(g, epi, batch, m->n_cu, s); };
  // WaveNet (cfm.rs:373-408): h fp32 in hw, and as the convolutions' operand in rows pad ..
  // of the zero-padded planes; all taps are one product (K step kt reads row m + tap)
  const long hp = (long)hp_pieces(c, T);
  for (int l = 0; l < NL; l++) {
    const WnLayer &w = m->wn[l];
    const bool last = l + 1 == NL;
    const int rso = last ? d : 2 * d;
    if (few)
      for (int b = 0; b < B; b++)
        CK(cfm_rows_frag(m->hw.p + (size_t)b * T * d, d, T, d, dk, pad, pieces(m->hpP) + b * hp, s));
    WF(in_w, w.in_w, K * d, 2 * d, K * d, few ? 0 : d);
    CfmMm g = mm_args(pieces(m->hpP), K * d, in_w, T, d);
    g.sa = hp;
    g.kt_a = g.taps_kt = dk;
    if (few) {
      g.N = 2 * d;
      g.y = m->acts.p;
      g.ldy = 2 * d;
      g.sy = (long)T * 2 * d;
      CK(mm(g, kMmConv, B));
      CK(cfm_gate(m->acts.p, w.in_b, m->wng.p + (size_t)l * 2 * d, 2 * d * NL, R, T, d, m->act.p, s));
      CK(gemm(m, R, rso, d, m->act.p, d, w.rs_w, d, m->rs.p, rso, 0.0f));
      CK(cfm_res_skip(m->rs.p, w.rs_b, last ? 1 : 0, l == 0, R, d, m->hw.p, m->oacc.p, s));
      continue;
    }
    g.bias = w.in_b;
    g.g = m->wng.p + (size_t)l * 2 * d;
    g.ld_g = 2 * d * NL;
    g.o = pieces(m->actP);
    g.kt_o = dk;
    CK(mm(g, kMmGate, B));
    WF(rs_w, w.rs_w, d, rso, d);
    CfmMm r = mm_args(pieces(m->actP), d, rs_w, R, rso);
    r.T = T;
    r.bias = w.rs_b;
    r.y = m->hw.p;
    r.y2 = m->oacc.p;
    r.ldy = d;
    r.o = pieces(m->hpP);
    r.so = hp;
    r.o_row0 = pad;
    r.kt_o = dk;
    r.first = l == 0;
    CK(mm(r, kMmResSkip, 1));
  }
  // h = wavenet + res_projection(x_res); FinalLayer; conv2
  float *h = m->hA.p;
  if (few) {
    CK(gemm(m, R, d, d, m->xres.p, d, m->rp_w, d, m->oacc.p, d, 1.0f, m->rp_b));
    CK(cfm_final_norm(m->oacc.p, m->n.p, R, T, d, m->fmod.p, s));
    CK(gemm(m, R, d, d, m->n.p, d, m->fl_w, d, h, d, 0.0f, m->fl_b));
    CK(gemm(m, R, C, d, h, d, m->c2_w, d, m->v.p, C, 0.0f, m->c2_b));
    return ITTS_OK;
  }
  {
    WF(w, m->rp_w, d, d, d);
    CfmMm g = mm_args(pieces(m->xresP), d, w, R, d);
    g.bias = m->rp_b;
    g.y = m->oacc.p;
    g.yr = m->oacc.p;
    g.ldy = d;
    CK(mm(g, kMmPlain, 1));
  }
  CK(cfm_norm_frag(m->oacc.p, R, T, d, m->fmod.p, 2 * d, nullptr, true, pieces(m->nP), s));
  {
    WF(w, m->fl_w, d, d, d);
    CfmMm g = mm_args(pieces(m->nP), d, w, R, d);
    g.bias = m->fl_b;
    g.o = pieces(m->attP);
    g.kt_o = dk;
    CK(mm(g, kMmPlain, 1));
  }
  WF(w, m->c2_w, d, C, d);
  CfmMm g = mm_args(pieces(m->attP), d, w, R, C);
  g.bias = m->c2_b;
  g.y = m->v.p;
  g.ldy = C;
  CK(mm(g, kMmPlain, 1));
  return ITTS_OK;
#undef WF
}

}  // namespace

extern "C" {

itts_status itts_cfm_create(const itts_cfm_config *cfg, const char *const *names, const float *const *data,
                            const int64_t *numel, int32_t n, itts_cfm **out) {
  if (!cfg || !out || (n > 0 && (!names || !data || !numel))) return cerr(ITTS_E_VALIDATION, "cfm: null argument");
  *out = nullptr;
  if (itts_status st = check_config(*cfg)) return st;
  const itts_cfm_config c = *cfg;
  const size_t d = c.dim, F = c.inter, C = c.in_ch, NL = c.wn_layers, K = c.wn_kernel, Lc = c.n_layers;
  const size_t MD = 2 * C + d + c.style_dim;
  // arena slots: name -> (offset, count); AdaLN projections and w1/w3 packed as used
  struct Slot {
    size_t off, count;
  };
  std::map<std::string, Slot> slots;
  size_t top = 0;
  auto put = [&](const std::string &nm, size_t count) {
    slots[nm] = Slot{top, count};
    top += (count + 63) & ~size_t(63);
  };
  auto put_at = [&](const std::string &nm, size_t off, size_t count) { slots[nm] = Slot{off, count}; };
  put("cond_projection.weight", d * d);
  put("cond_projection.bias", d);
  put("cond_x_merge_linear.weight", d * MD);
  put("cond_x_merge_linear.bias", d);
  for (const char *p : {"t_embedder", "t_embedder2"}) {
    put(std::string(p) + ".mlp.layers.0.weight", d * kFreqDim);
    put(std::string(p) + ".mlp.layers.0.bias", d);
    put(std::string(p) + ".mlp.layers.2.weight", d * d);
    put(std::string(p) + ".mlp.layers.2.bias", d);
  }
  const size_t na = 2 * Lc + 1, ada_w = top;
  top += na * 2 * d * d;
  const size_t ada_b = top;
  top += (na * 2 * d + 63) & ~size_t(63);
  auto ada = [&](const std::string &p, size_t slot) {
    put_at(p + ".project_layer.weight", ada_w + slot * 2 * d * d, 2 * d * d);
    put_at(p + ".project_layer.bias", ada_b + slot * 2 * d, 2 * d);
    put(p + ".norm.weight", d);
  };
  for (size_t i = 0; i < Lc; i++) {
    const std::string p = "transformer.layers." + std::to_string(i);
    ada(p + ".attention_norm", 2 * i);
    ada(p + ".ffn_norm", 2 * i + 1);
    put(p + ".attention.wqkv.weight", 3 * d * d);
    put(p + ".attention.wo.weight", d * d);
    put_at(p + ".feed_forward.w1.weight", top, F * d);  // w3 right after w1: the packed [w1; w3]
    put_at(p + ".feed_forward.w3.weight", top + F * d, F * d);
    top += (2 * F * d + 63) & ~size_t(63);
    put(p + ".feed_forward.w2.weight", d * F);
    put(p + ".skip_in_linear.weight", d * 2 * d);
    put(p + ".skip_in_linear.bias", d);
  }
  ada("transformer.norm", 2 * Lc);
  put("skip_linear.weight", d * (d + C));
  put("skip_linear.bias", d);
  put("conv1.weight", d * d);
  put("conv1.bias", d);
  put("res_projection.weight", d * d);
  put("res_projection.bias", d);
  put("wavenet.cond_layer.weight", 2 * d * NL * d);
  put("wavenet.cond_layer.bias", 2 * d * NL);
  for (size_t i = 0; i < NL; i++) {
    const size_t rso = i + 1 == NL ? d : 2 * d;
    put("wavenet.in_layers." + std::to_string(i) + ".weight", 2 * d * K * d);
    put("wavenet.in_layers." + std::to_string(i) + ".bias", 2 * d);
    put("wavenet.res_skip_layers." + std::to_string(i) + ".weight", rso * d);
    put("wavenet.res_skip_layers." + std::to_string(i) + ".bias", rso);
  }
  put("final_layer.adaLN_modulation.layers.1.weight", 2 * d * d);
  put("final_layer.adaLN_modulation.layers.1.bias", 2 * d);
  put("final_layer.linear.weight", d * d);
  put("final_layer.linear.bias", d);
  put("conv2.weight", C * d);
  put("conv2.bias", C);
  // every required tensor exactly once, with the element count its name requires
  std::map<std::string, int> seen;
  for (int32_t i = 0; i < n; i++) {
    if (!names[i] || !data[i]) return cerr(ITTS_E_VALIDATION, "cfm: null tensor name or data at %d", i);
    auto it = slots.find(names[i]);
    if (it == slots.end()) continue;  // tensors the estimator does not use are ignored, as the filtered loader does
    if (numel[i] != (int64_t)it->second.count)
      return cerr(ITTS_E_WEIGHT, "weight load error in `%s`: %lld elements, expected %zu", names[i],
                  (long long)numel[i], it->second.count);
    if (seen.count(names[i])) return cerr(ITTS_E_WEIGHT, "weight load error in `%s`: given twice", names[i]);
    seen[names[i]] = i;
  }
  for (const auto &kv : slots)
    if (!seen.count(kv.first)) return cerr(ITTS_E_WEIGHT, "weight load error in `%s`: missing tensor", kv.first.c_str());
  auto *m = new itts_cfm();
  m->c = c;
  auto fail = [&](itts_status st) {
    delete m;
    return st;
  };
  if (hipStreamCreate(&m->s) != hipSuccess) return fail(cerr(ITTS_E_DEVICE, "hipStreamCreate failed"));
  {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&m->n_cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
      return fail(cerr(ITTS_E_DEVICE, "querying the device's compute units failed"));
  }
  if (cfm_mm_init() != hipSuccess) return fail(cerr(ITTS_E_DEVICE, "preparing the product kernels failed"));
  if (hipMalloc(&m->arena, top * sizeof(float)) != hipSuccess)
    return fail(cerr(ITTS_E_DEVICE, "out of device memory for the CFM weights (%zu bytes)", top * sizeof(float)));
  for (const auto &kv : seen) {
    const Slot &sl = slots[kv.first];
    if (hipMemcpy(m->arena + sl.off, data[kv.second], sl.count * sizeof(float), hipMemcpyHostToDevice) != hipSuccess)
      return fail(cerr(ITTS_E_DEVICE, "copying `%s` to the device failed", kv.first.c_str()));
  }
  auto at = [&](const std::string &nm) -> const float * { return m->arena + slots[nm].off; };
  m->cond_w = at("cond_projection.weight");
  m->cond_b = at("cond_projection.bias");
  m->merge_w = at("cond_x_merge_linear.weight");
  m->merge_b = at("cond_x_merge_linear.bias");
  const char *te[2] = {"t_embedder", "t_embedder2"};
  for (int e = 0; e < 2; e++) {
    m->te_w0[e] = at(std::string(te[e]) + ".mlp.layers.0.weight");
    m->te_b0[e] = at(std::string(te[e]) + ".mlp.layers.0.bias");
    m->te_w2[e] = at(std::string(te[e]) + ".mlp.layers.2.weight");
    m->te_b2[e] = at(std::string(te[e]) + ".mlp.layers.2.bias");
  }
  m->ada_w = m->arena + ada_w;
  m->ada_b = m->arena + ada_b;
  m->tn_w = at("transformer.norm.norm.weight");
  for (size_t i = 0; i < Lc; i++) {
    const std::string p = "transformer.layers." + std::to_string(i);
    m->L.push_back(Block{at(p + ".attention.wqkv.weight"), at(p + ".attention.wo.weight"),
                         at(p + ".feed_forward.w1.weight"), at(p + ".feed_forward.w2.weight"),
                         at(p + ".skip_in_linear.weight"), at(p + ".skip_in_linear.bias"),
                         at(p + ".attention_norm.norm.weight"), at(p + ".ffn_norm.norm.weight")});
  }
  m->skl_w = at("skip_linear.weight");
  m->skl_b = at("skip_linear.bias");
  m->c1_w = at("conv1.weight");
  m->c1_b = at("conv1.bias");
  m->rp_w = at("res_projection.weight");
  m->rp_b = at("res_projection.bias");
  m->wc_w = at("wavenet.cond_layer.weight");
  m->wc_b = at("wavenet.cond_layer.bias");
  for (size_t i = 0; i < NL; i++) {
    const std::string a = "wavenet.in_layers." + std::to_string(i), b = "wavenet.res_skip_layers." + std::to_string(i);
    m->wn.push_back(WnLayer{at(a + ".weight"), at(a + ".bias"), at(b + ".weight"), at(b + ".bias")});
  }
  m->fa_w = at("final_layer.adaLN_modulation.layers.1.weight");
  m->fa_b = at("final_layer.adaLN_modulation.layers.1.bias");
  m->fl_w = at("final_layer.linear.weight");
  m->fl_b = at("final_layer.linear.bias");
  m->c2_w = at("conv2.weight");
  m->c2_b = at("conv2.bias");
  m->skips.resize(Lc / 2);
  m->skipP.resize(Lc / 2);
  if (hipEventCreate(&m->e0) != hipSuccess || hipEventCreate(&m->e1) != hipSuccess)
    return fail(cerr(ITTS_E_DEVICE, "hipEventCreate failed"));
  *out = m;
  return ITTS_OK;
}

void itts_cfm_destroy(itts_cfm *cfm) { delete cfm; }

itts_status itts_cfm_forward(itts_cfm *m, const float *x_t, const float *x_merged, const float *t, int32_t B,
                             int32_t T, float *out) {
  if (!m || !x_t || !x_merged || !t || !out) return cerr(ITTS_E_VALIDATION, "cfm forward: null argument");
  if (B < 1 || T < 1) return cerr(ITTS_E_VALIDATION, "x_t: expected [B, T, %d] with B, T >= 1", m->c.in_ch);
  const itts_cfm_config &c = m->c;
  const size_t R = (size_t)B * T, C = c.in_ch, MD = 2 * C + c.dim + c.style_dim;
  CK(m->io_a.ensure(R * C));
  CK(m->io_b.ensure(R * MD));
  if (itts_status st = ensure_rows(m, B, T)) return st;
  CK(hipMemcpyAsync(m->io_a.p, x_t, sizeof(float) * R * C, hipMemcpyHostToDevice, m->s));
  CK(hipMemcpyAsync(m->io_b.p, x_merged, sizeof(float) * R * MD, hipMemcpyHostToDevice, m->s));
  CK(hipMemcpyAsync(m->tdev.p, t, sizeof(float) * B, hipMemcpyHostToDevice, m->s));
  if (itts_status st = forward(m, m->io_a.p, m->io_b.p, B, T)) return st;
  CK(m->xt.ensure(R * C));
  CK(cfm_transpose_tc(m->v.p, B, T, (int)C, m->xt.p, m->s));
  CK(hipMemcpyAsync(out, m->xt.p, sizeof(float) * R * C, hipMemcpyDeviceToHost, m->s));
  CK(hipStreamSynchronize(m->s));
  return ITTS_OK;
}

itts_status itts_cfm_solve_euler(itts_cfm *m, const float *cat_condition, int32_t T_total, const float *ref_mel,
                                 int32_t T_ref, const float *style, const float *noise_z, int32_t n_timesteps,
                                 float cfg_rate, float *mel_out) {
  if (!m || !cat_condition || !style || !noise_z || !mel_out || (T_ref > 0 && !ref_mel))
    return cerr(ITTS_E_VALIDATION, "cfm solve: null argument");
  if (n_timesteps < 1) return cerr(ITTS_E_VALIDATION, "n_timesteps: n_timesteps must be >= 1");
  if (T_total < 1) return cerr(ITTS_E_VALIDATION, "cat_condition: expected [1, T_total, %d], got T_total %d", m->c.dim, T_total);
  if (T_ref < 0 || T_ref >= T_total)
    return cerr(ITTS_E_VALIDATION,
                "ref_mel: ref_mel length (%d) must be strictly less than cat_condition length (%d)", T_ref, T_total);
  const itts_cfm_config &c = m->c;
  const int d = c.dim, C = c.in_ch, S = c.style_dim, T = T_total, MD = 2 * C + d + S;
  hipStream_t s = m->s;
  m->last_ms = -1.0f;
  CK(m->x.ensure((size_t)C * T));
  CK(m->xt.ensure((size_t)2 * T * C));
  CK(m->merged.ensure((size_t)2 * T * MD));
  CK(m->catc.ensure((size_t)T * d));
  CK(m->refm.ensure((size_t)C * (T_ref > 0 ? T_ref : 1)));
  CK(m->sty.ensure((size_t)(S > 0 ? S : 1)));
  if (itts_status st = ensure_rows(m, 2, T)) return st;
  CK(hipMemcpyAsync(m->catc.p, cat_condition, sizeof(float) * T * d, hipMemcpyHostToDevice, s));
  if (T_ref > 0) CK(hipMemcpyAsync(m->refm.p, ref_mel, sizeof(float) * C * T_ref, hipMemcpyHostToDevice, s));
  if (S > 0) CK(hipMemcpyAsync(m->sty.p, style, sizeof(float) * S, hipMemcpyHostToDevice, s));
  CK(hipMemcpyAsync(m->x.p, noise_z, sizeof(float) * C * T, hipMemcpyHostToDevice, s));
  // static CFG tail (cfm.rs:682-711): prompt mel and style in row 0, cond_projection of the
  // condition in row 0 and of zeros (= its bias) in row 1
  CK(hipMemsetAsync(m->merged.p, 0, sizeof(float) * 2 * T * MD, s));
  CK(cfm_static_tail(m->merged.p, MD, C, d, S, T, m->refm.p, T_ref, m->sty.p, s));
  CK(cfm_bias_rows(m->merged.p + 2 * C, MD, m->cond_b, 2 * T, d, s));
  if (T >= kMfmaRows) {  // (2 T rows: the planes' path, whose buffers are in place)
    const uint4 *w = weight_frag(m, m->cond_w, d, d, d);
    if (!w) return cerr(ITTS_E_DEVICE, "out of device memory for the weights' operand planes");
    CK(cfm_rows_frag(m->catc.p, d, T, d, d / 16, 0, pieces(m->nP), s));
    CfmMm g = mm_args(pieces(m->nP), d, w, T, d);
    g.y = m->merged.p + 2 * C;
    g.yr = g.y;
    g.ldy = MD;
    CK(cfm_mm(g, kMmPlain, 1, m->n_cu, s));
  } else {
    CK(gemm(m, T, d, d, m->catc.p, d, m->cond_w, d, m->merged.p + 2 * C, MD, 1.0f));
  }
  CK(hipEventRecord(m->e0, s));
  const float dt = 1.0f / (float)n_timesteps;
  for (int step = 0; step < n_timesteps; step++) {
    CK(cfm_fill(m->tdev.p, 2, (float)step * dt, s));
    CK(cfm_euler_prep(m->x.p, C, T, T_ref, m->xt.p, m->merged.p, MD, s));
    if (itts_status st = forward(m, m->xt.p, m->merged.p, 2, T)) return st;
    CK(cfm_euler_update(m->x.p, m->v.p, C, T, dt, cfg_rate, s));
  }
  CK(hipEventRecord(m->e1, s));
  const int G = T - T_ref;
  CK(hipMemcpy2DAsync(mel_out, sizeof(float) * G, m->x.p + T_ref, sizeof(float) * T, sizeof(float) * G, C,
                      hipMemcpyDeviceToHost, s));
  CK(hipStreamSynchronize(s));
  float ms = 0.0f;
  CK(hipEventElapsedTime(&ms, m->e0, m->e1));
  m->last_ms = ms;
  return ITTS_OK;
}

itts_status itts_cfm_last_solve_ms(itts_cfm *m, float *ms) {
  if (!m || !ms) return cerr(ITTS_E_VALIDATION, "cfm timing: null argument");
  if (m->last_ms < 0.0f) return cerr(ITTS_E_VALIDATION, "cfm timing: no completed solve_euler call");
  *ms = m->last_ms;
  return ITTS_OK;
}

}  // extern "C"
