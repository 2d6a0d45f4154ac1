// Host-side launchers of the gfx950 kernels.  Every launcher enqueues on `stream` and
// returns the launch status; shapes are validated by the caller (runtime.cpp).
#pragma once

#include <hip/hip_runtime.h>

#include "common.h"

namespace itts {

// kProEmbedLN: the input row is the step embedding mel_emb[ctl->tok] + mel_pos[ctl->pos]
// (block 0 stores it to x_out as the residual stream), then LayerNorm.
// kProAttn: the input row is the attention output, combined from the split partials of
// the decode attention (attn.part / attn.n_head / attn.max_splits, L from ctl).
enum Prologue : int { kProNone = 0, kProLN = 1, kProLNLN = 2, kProEmbedLN = 3, kProAttn = 4 };

struct AttnPartials {
  const float *part;  // [n_head][max_splits][66]: max, denominator, 64 outputs
  int n_head;
  int max_splits;
  int static_len;     // key count when ctl == nullptr
};
enum Epilogue : int { kEpiStore = 0, kEpiResid = 1, kEpiGelu = 2, kEpiQKV = 3 };

// Activations as the prefill GEMM reads them: x = hi + lo (fp16 planes, ~22 significant
// bits) and the row sums of each 64-column group (the MLX bias term needs sum_k x).
struct SplitAct {
  const uint16_t *hi, *lo;  // [M][K]
  const float *gs;          // [M][K/64]
};
struct SplitOut {
  uint16_t *hi, *lo;
  float *gs;
  SplitAct act() const { return SplitAct{hi, lo, gs}; }
};

// One sequence of a batched decode step: its control block, its cache bases (layer 0 of
// [layer][n_head][max_seq][64]) and its code output.
struct BatchSeq {
  DecodeCtl *ctl;
  void *k, *v;
  int32_t *codes;
};

// Where the QKV epilogue scatters: q -> q_out[M][d]; k, v -> this layer's cache
// [n_head][max_seq][64] at row pos0 (the GEMV).  launch_gemm's rows are those of a batched step:
// row m belongs to sequence m, its K/V row goes to seqs[m]'s cache at offset layer_off (elements)
// and position ctl->valid_len, and nothing is written for a finished sequence.
struct QkvDst {
  float *q_out;
  void *k_cache;
  void *v_cache;
  int max_seq;
  int pos0;
  int d_model;
  const BatchSeq *seqs;
  size_t layer_off;
};

struct GemvArgs {
  DevQL ql;
  const float *x;          // input row [K]
  const float *ln_w, *ln_b;    // LN (prologue kProLN / first LN of kProLNLN)
  const float *ln2_w, *ln2_b;  // second LN of kProLNLN
  float *y;                // output row [N] (store / gelu) or residual stream (resid)
  QkvDst qkv;
  const DecodeCtl *ctl;    // optional: early exit when done, cache row = valid_len
  const float *emb_tok, *emb_pos;  // kProEmbedLN tables (mel_emb, mel_pos)
  float *x_out;            // kProEmbedLN: residual stream written by block 0
  DecodeCtl *finish;       // optional: block 0 advances finish->valid_len after its rows
  AttnPartials attn;       // kProAttn
};

hipError_t launch_gemv(const GemvArgs &a, int bits, int ptype, int pro, int epi, int kvt,
                       hipStream_t s);

// Decode attention: q [n_head*64] against cache rows 0..L-1 with L = ctl->valid_len + 1
// (or static_len), 256 keys per split.  Each split writes its partial (max, denominator,
// 64 unnormalised outputs) to part [n_head][max_splits][66]; the consumer (the c_proj
// GEMV's kProAttn prologue) combines them.
int attn_decode_max_splits(int max_seq);
// Batched decode attention, one 16-wave block per (head, sequence), into the sequences'
// attention rows [B][d] in split form; finished sequences are skipped.
hipError_t launch_decode_batch_rows(const float *q, const BatchSeq *seqs, int B, size_t layer_off, int n_head,
                                    int max_seq, const SplitOut &out, int kvt, hipStream_t s);
// x[b] = mel_emb[tok_b] + mel_pos[pos_b] from the sequences' control blocks.
hipError_t launch_embed_batch(const BatchSeq *seqs, int B, const float *mel_emb, const float *mel_pos, int d, float *x,
                              hipStream_t s);
// valid_len += 1 for every sequence that is not finished.
hipError_t launch_advance_batch(const BatchSeq *seqs, int B, hipStream_t s);
hipError_t launch_attn_decode(const float *q, const void *kc, const void *vc, int n_head,
                              int max_seq, const DecodeCtl *ctl, int static_len, float *part,
                              int kvt, hipStream_t s);


// Row descriptors for the prefill embedding.
struct EmbedRow {
  int kind;  // 0 cond row, 1 text row, 2 Mel row
  int id;    // cond row index / token id
  int pos;   // positional index
};
hipError_t launch_embed_rows(const EmbedRow *rows, int T, const float *conds,
                             const float *text_emb, const float *lang_row,
                             const float *text_pos, const float *mel_emb,
                             const float *mel_pos, int d, float *x, hipStream_t s);

// LN of T rows [T][d] -> [T][d] in the GEMM's split form; with w2/b2 a second LN follows.
hipError_t launch_ln_rows(const float *x, const float *w, const float *b, int T, int d,
                          const SplitOut &y, hipStream_t s, const float *w2 = nullptr,
                          const float *b2 = nullptr);

// Attention probe: softmax probabilities of head `head` (none when < 0) for the query rows
// q0.. over the key columns [k0, k1): out [(rows - q0)][k1 - k0].
struct AttnProbe {
  int head, q0, k0, k1;
  float *out;
};
// Probe of M concatenated rows (row t attends to keys kstart[t]..t of the K/V
// [n_head][M][64]): writes only the probabilities, for rows p.q0..M-1.
hipError_t launch_attn_probe(const float *q, int M, const int *kstart, const void *kc, const void *vc, int n_head,
                             const AttnProbe &p, int kvt, hipStream_t s);
// out[r] = log_softmax(logits[r])[codes[r]] for R rows of V logits.
hipError_t launch_log_softmax_pick(const float *logits, int R, int V, const int *codes, float *out, hipStream_t s);

// Prefill GEMM: y = x[M][K] . Wdeq^T + bias with the same epilogues as the GEMV.
// A LayerNorm folded into the product that follows it (few-row products, K <= 2048,
// K % 256 == 0): the product runs on gamma * x straight from the fp32 rows x [M][K] and its
// epilogue applies each row's statistics, rstd (sum - mean G[n]) + c[n], with G = W gamma
// and c = W beta + bias (launch_ln_fold), in place of sum + bias.
struct FoldIn {
  const float *x, *gamma, *G, *c;
};

struct GemmArgs {
  DevQL ql;
  // few-row products: the codes in fragment order and the (scale, bias) words [K/64][ldn] (null:
  // kEpiStore reads ql's, the others take the tiles)
  const uint4 *fcodes;
  const void *fparams;
  int ldn;
  SplitAct x;       // [M][K] (unused with fold.x)
  FoldIn fold;      // fold.x set: the input is LayerNorm(x) by the fold above
  int M;
  float *y;         // [M][N] (store) or residual stream [M][N] (resid)
  SplitOut xo;      // gelu: the next GEMM's input [M][N] (N a multiple of 64)
  QkvDst qkv;
  // split-K partial tiles and per-tile arrival counters (zero between launches); split-K
  // is not used when they are absent or too small
  float *ws;
  size_t ws_floats;
  uint32_t *cnt;
  int cnt_words;
  int n_cu;         // compute units (grid sizing)
};
hipError_t launch_gemm(const GemmArgs &a, int bits, int ptype, int epi, int kvt, hipStream_t s);
// Sets the LDS attributes of every GEMM instantiation (before any graph capture).
hipError_t gemm_init();
size_t gemm_ws_floats(int n_cu);
constexpr int kGemmCounters = 4096;

// ---- multi-row forwards on operands in fragment order (kernels_rows.hip) ----
// kvt of rows_mm and rows_attn, beside KvType: fp32 rows whose attention operands are fp16 pairs
// (magnitudes below 131008, 22 bits, an absolute 2^-25 at the small end; kKvF32 holds all of them
// as they are).
constexpr int kRowsPairs = 2;
// Activation planes of M rows of K values (16-byte pieces; the group sums' last step must be
// zero-filled once), the attention's Q and K / V fragments, and a weight's codes in fragment
// order, scale table and bias planes (made once by rows_params).
size_t rows_planes_pieces(int M, int K);
size_t rows_q_pieces(int M, int H);
size_t rows_kv_pieces(int M, int H);
int rows_ldn(int N);
size_t rows_scale_floats(int N, int K);
size_t rows_bias_pieces(int N, int K);
size_t rows_codes_bytes(int N, int K, int bits);
// ... (codes, scales, bias planes; params: the (scale, bias) words [K/64][rows_ldn(N)])
hipError_t rows_params(const DevQL &ql, int bits, int ptype, uint4 *codes, float *scale, uint4 *bw, void *params,
                       hipStream_t s);
// LN (and a second one with w2; none without w) of M rows [M][d] as planes.
hipError_t rows_ln(const float *x, const float *w, const float *b, const float *w2, const float *b2, int M, int d,
                   uint4 *out, hipStream_t s);
// One product over planes x, with the epilogues of launch_gemm: store y [M][N]; residual y +=,
// and with `o` the next folded LayerNorm's input (planes of gamma x, group statistics so);
// GELU to planes o; QKV to the fragments qf / kvf, to the cache rows 0.. [n_head][max_seq][64]
// where kc / vc are set, and q to q_out [M][N / 3] where set.  st, fG, fc: folded LayerNorm input.
struct RowsMm {
  const uint4 *x, *codes;
  const float *scale;
  const uint4 *bw;
  const float *bias;
  int ldn, M, N, K;
  const float2 *st;
  const float *fG, *fc;
  float *y;
  uint4 *o;
  const float *gamma;
  float2 *so;
  uint4 *qf, *kvf;
  float *q_out;
  void *kc, *vc;
  int max_seq, n_cu;
  float *ws;       // partial tiles and counters of products whose K is split over blocks (as in GemmArgs)
  size_t ws_floats;
  uint32_t *cnt;
  int cnt_words;
  int nM, nN, gm, S;  // tile grid and K split, set at the launch
};
hipError_t rows_mm(const RowsMm &a, int bits, int epi, int kvt, hipStream_t s);
// Causal attention: row t attends to keys kstart[t] (or 0) .. t; order (optional) lists the
// ceil(M / 32) query tiles, most keys first.  Output as planes [M][64 H].
hipError_t rows_attn(const uint4 *qf, const uint4 *kvf, int M, int H, const int *kstart, const int *order, int kvt,
                     uint4 *out, hipStream_t s);

// fp32 rows [M][K] -> the GEMM's split form.
hipError_t launch_split_rows(const float *x, int M, int K, const SplitOut &o, hipStream_t s);

hipError_t launch_dequant(const DevQL &ql, int bits, int ptype, float *out, hipStream_t s);

// Persistent decode step (kernels_persist.hip): one launch of B blocks
// (one per CU) runs a whole decode step.  Exchange words are (epoch << 32 | fp32 bits).
constexpr int kCntStride = 32;  // one 128-byte line per head counter
struct PersistArgs {
  const DevLayer *layers;  // device array [n_layer]
  int n_layer, d, H, F, V, S, B;
  DevQL head;
  const float *ln_f_w, *ln_f_b, *fn_w, *fn_b;
  // LayerNorms folded into the QKV and c_fc products (ln_fold_layout): per layer
  // G = W.gamma and c = W.beta + bias of both products, fold_floats(d, F) floats a layer
  const float *fold;
  const float *mel_emb, *mel_pos;
  void *kc, *vc;           // cache bases [n_layer][H][max_seq][64], bf16 or f32 rows
  int max_seq;
  int kvt;                 // KvType of the rows
  DecodeCtl *ctl;
  // exchange arrays of 16-byte words (three values and an epoch), 16-byte aligned
  void *x_x, *x_qkv, *x_part, *x_attn, *x_mid, *x_f;
  uint32_t *cnt;           // [H * kCntStride] split counters (wrap at S; start at 0)
  uint32_t *err;           // nonzero after a timed-out wait
  float *logits;           // [V]
  uint32_t ep_stride;      // epochs per step: 8 * (n_layer + 1)
  // LDS region sizes (floats, multiples of 4): input row, normalised row (both long enough
  // for the dot products' padded layout: 4 floats after every 16-byte code chunk's
  // values), per-chunk partials, residual slice, row outputs, attention partials of one
  // head, one layer's staged parameters
  int xin_len, xn_len, part_len, own_len, out_len, pp_len, lp_len;
};
// A LayerNorm followed by a QuantizedLinear, y = W.((x - mu) * rstd * gamma + beta) + bias,
// equals rstd * (W.(gamma * x) - mu * G) + c with G = W.gamma and c = W.beta + bias, so
// the product can start on gamma * x before mu and rstd are known.  Per layer the fold
// buffer holds G and c of c_attn (ln_1) and of c_fc (ln_2):
//   [G_qkv 3d][c_qkv 3d][G_fc F][c_fc F]
__host__ __device__ inline size_t fold_floats(int d, int F) { return 6 * (size_t)d + 2 * (size_t)F; }
// G[o] = sum_k Wdeq[o][k] gamma[k] and c[o] = sum_k Wdeq[o][k] beta[k] + bias[o] for the N
// rows of ql (fp64 sums, rounded once), one wave per row.
hipError_t launch_ln_fold(const DevQL &ql, int bits, int ptype, const float *gamma, const float *beta, float *G,
                          float *c, hipStream_t s);
// Whether the persistent step supports this shape on B blocks; *S = attention splits.
// f32 rows also need persist_f32_v_floats() floats from the start of the block's LDS
// (input row, normalised row and partials: the host pads the partials to fit).
bool persist_supported(int d, int F, int V, int H, int n_layer, int max_seq, int B, int bits, int *S);
constexpr size_t kPersistMaxLds = 150 * 1024;
// LDS floats that f32 V rows of one attention split take: 512 per chunk of 8 keys.
inline int persist_f32_v_floats(int max_seq, int S) { return 512 * (((max_seq + S - 1) / S + 7) / 8); }
size_t persist_lds_bytes(const PersistArgs &a);
// 16-byte words of the exchange arrays x_x, x_qkv, x_part, x_attn, x_mid, x_f: total, and
// each array's offset in off[6].
size_t persist_exchange_words(int d, int F, int H, int S, int B, size_t off[6]);
// Whether one block of the persistent kernel with `lds` bytes of dynamic LDS fits a
// compute unit (threads, static + dynamic LDS).
hipError_t persist_fits(int bits, int ptype, int kvt, size_t lds, bool *fits);
hipError_t launch_decode_persist(PersistArgs a, int bits, int ptype, hipStream_t s);
// Raises the kernel's dynamic-LDS limit; once per process, outside stream capture.
hipError_t persist_init();

// Raises the sampler's dynamic-LDS limit; call once per process before any launch
// (never during stream capture).
hipError_t sampler_init();

// Device sampler (one block).  mode 0: API call on `logits` (penalised in place,
// token to *tok_out, rng advanced); mode 1: generate step driven by ctl.
hipError_t launch_sampler(float *logits, int n, const uint64_t *seen, DevSampling p,
                          uint64_t *rng, int32_t *tok_out, DecodeCtl *ctl, int32_t *codes,
                          int stop_tok, int mode, hipStream_t s);
// One sampler block per sequence of a batch: block b samples logits[b][n] with ps[b] into
// seqs[b]'s control block and codes (the generate loop's mode).  lds_top_k is the largest
// top_k of the batch (sets the LDS of the candidate sort).
hipError_t launch_sampler_batch(float *logits, int n, const DevSampling *ps, const BatchSeq *seqs, int B,
                                int stop_tok, int lds_top_k, bool any_sampled, hipStream_t s);

// Device ordinals the library accepts.
constexpr int kMaxDevices = 64;
// Staging area of the sampler's no-allocation entry point: a static device array (one per
// device, held until the process ends) with room for kStageMaxLogits logits, the seen-set
// words, the RNG state and the token.
constexpr int kStageMaxLogits = 9216;
struct SamplerStage {
  float *logits;   // [kStageMaxLogits]
  uint64_t *seen;  // [129]
  uint64_t *rng;
  int32_t *tok;
};
// Looks up the staging array's address on device dev, which must be the current device;
// later calls for the same device do nothing.
hipError_t sampler_stage_init(int dev);
// The staging area of device dev; false if sampler_stage_init has not run for it.
bool sampler_stage(int dev, SamplerStage *out);

// ---- Stage-2 CFM DiT estimator (kernels_cfm.hip); activations [B][T][C] fp32 ----
hipError_t cfm_temb(const float *t, int B, float *emb /*[B][256]*/, hipStream_t s);
hipError_t cfm_silu(const float *x, float *y, int n, hipStream_t s);
hipError_t cfm_bias_rows(float *C, int ldc, const float *bias, int rows, int cols, hipStream_t s);
hipError_t cfm_adaln(const float *x, float *y, int R, int T, int d, const float *mod, int ld_mod, const float *norm_w,
                     hipStream_t s);
hipError_t cfm_final_norm(const float *x, float *y, int R, int T, int d, const float *mod, hipStream_t s);
// rope (cos, sin) table [T][32][2] for positions 0..T-1
hipError_t cfm_rope_table(int T, float *tab, hipStream_t s);
// ---- products over fragment planes (kernels_cfm_mm.hip; layout in frag.h) ----
// 16-byte pieces of the planes of `rows` rows (whole 128-row tiles) with nk K steps of 16.
size_t cfm_frag_pieces(long rows, int nk);
// Weight rows W [N][ldw] -> K steps kt0 .. kt0 + ceil(K / 16) of `out` (cfm_frag_pieces(N, nk),
// zero-filled by the caller where K steps stay unwritten).  With ilv = F (N = 2F) the two
// halves' rows alternate per 32, as the SwiGLU and gate epilogues take them (cfm_frag_pieces of
// 64 ceil(F / 32) rows).
hipError_t cfm_weight_frag(const float *W, int ldw, int N, int K, int kt0, int nk, int ilv, uint4 *out, hipStream_t s);
// fp32 rows X [R][ld] (K values) -> rows row0 .. of the planes `out`, nk K steps, zeros past K.
hipError_t cfm_rows_frag(const float *X, int ld, int R, int K, int nk, int row0, uint4 *out, hipStream_t s);
// AdaLN (or, final_norm, the final layer's norm with mod = shift | scale) of x [R][d] as planes.
hipError_t cfm_norm_frag(const float *x, int R, int T, int d, const float *mod, int ld_mod, const float *norm_w,
                         bool final_norm, uint4 *out, hipStream_t s);
// One product y[z] = A[z] W^T, z < batch; the epilogue by kind:
//   Plain   (+ bias) (+ yr) to fp32 rows y (ldy, batch stride sy) and / or planes o (kt_o K
//           steps, batch stride so pieces, rows from o_row0)
//   Conv    Plain over a convolution's operand: K step kt reads row m + kt / taps_kt
//   Gate    Conv, tanh(first half) * sigmoid(second half) with bias + g rows, to planes o;
//           N output columns, W interleaved
//   Swiglu  silu(first) * second to planes o; N output columns, W interleaved
//   ResSkip rows r = b T + t: columns < N - ldy add to y [.][ldy] and go to planes o (batch
//           b, row t + o_row0); the last ldy columns add to (first: set) y2 [.][ldy]
//   Qkv     N = 3d: o = Q and o2 = K, V fragments of the attention, with rope (g = the table)
enum CfmEpi : int { kMmPlain, kMmConv, kMmGate, kMmSwiglu, kMmResSkip, kMmQkv };
struct CfmMm {
  const uint4 *a, *a2;  // planes; a2 (optional) holds K steps nk1 ..
  long sa;
  int zr;               // rows between batch entries that share a's planes
  int kt_a, kt_a2, nk1;  // K steps a row block of a / a2 holds
  const uint4 *w;
  int nk, taps_kt, M, N;
  int T;                // Plain, ResSkip: rows r = b T + t go to batch b's planes (0: entry z's)
  const float *bias, *yr;
  float *y, *y2;
  int ldy;
  long sy;
  uint4 *o, *o2;
  int kt_o;
  long so;
  int o_row0;
  const float *g;
  int ld_g, first;
  int vec, nM, nN, nz, gm;  // set at the launch: y, yr and bias take 16-byte accesses; the tile grid
};
hipError_t cfm_mm_init();  // once per device, before the first product
hipError_t cfm_mm(CfmMm a, int epi, int batch, int n_cu, hipStream_t s);
// Pieces of the attention's Q and K / V fragments, the fragments from fp32 rows qkv [B][T][3d],
// and the attention over them (to planes out [B T][d], or fp32 rows out_f).
size_t cfm_q_pieces(int B, int T, int H);
size_t cfm_kv_pieces(int B, int T, int H);
hipError_t cfm_qkv_frag(const float *qkv, const float *rope_tab, int B, int T, int H, uint4 *qf, uint4 *kvf,
                        hipStream_t s);
hipError_t cfm_attn_frag(const uint4 *qf, const uint4 *kvf, int B, int T, int H, uint4 *out, float *out_f, int n_cu,
                         hipStream_t s);
// The same product in fp32 FMAs for few rows (any M, any alignment; float4 loads when K,
// lda, ldw, sa, sw are multiples of 4 and A, W are 16-byte aligned); beta 0 never reads y.
// With bias: y = A W^T + bias[n] + beta y.
hipError_t cfm_rows_gemm(int batch, int M, int N, int K, const float *A, int lda, long sa, const float *W, int ldw,
                         long sw, float *y, int ldy, long sy, float beta, hipStream_t s, const float *bias = nullptr);
hipError_t cfm_swiglu(const float *gu, int R, int F, float *out, hipStream_t s);
hipError_t cfm_gate(const float *acts, const float *in_b, const float *g, int ld_g, int R, int T, int d, float *act,
                    hipStream_t s);
hipError_t cfm_res_skip(const float *rs, const float *rs_b, int last, int first, int R, int d, float *h, float *out,
                        hipStream_t s);
hipError_t cfm_euler_prep(float *x, int C, int T, int T_ref, float *xt, float *merged, int MD, hipStream_t s);
hipError_t cfm_euler_update(float *x, const float *v, int C, int T, float dt, float cfg, hipStream_t s);
hipError_t cfm_static_tail(float *merged, int MD, int C, int d, int S, int T, const float *ref_mel, int T_ref,
                           const float *style, hipStream_t s);
hipError_t cfm_transpose_tc(const float *v, int B, int T, int C, float *out, hipStream_t s);
hipError_t cfm_fill(float *p, int n, float v, hipStream_t s);

}  // namespace itts
