"""The multi-row forward on operands in fragment order (prompts, replay, all-row forward):
its tiles' edges against the oracle and, for the product alone, against float64."""
import sys

import numpy as np
import pytest

import ito
import itts_hip as H
from itts_hip import synth
from test_oracle_independent import numpy_forward

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


_models = {}


def _model(bits, pd, over=()):
    key = (bits, pd, over)
    if key not in _models:
        cfg = dict(synth.SMALL_CONFIG, quant_bits=bits, param_dtype=pd, **dict(over))
        W = synth.make_weights(cfg, seed=23, init="rich")
        _models[key] = (W, H.Gpt(W), ito.Model(W))
    return _models[key]


# around tiles of 32 and 64 rows and of 32 and 64 keys
@pytest.mark.parametrize("T", [48, 49, 63, 64, 65, 96, 97, 129, 320, 321])
@pytest.mark.parametrize("bits,pd,kv", [(8, H.ITTS_F16, H.ITTS_F32), (8, H.ITTS_F32, H.ITTS_BF16),
                                        (4, H.ITTS_F16, H.ITTS_BF16), (4, H.ITTS_F32, H.ITTS_F32)])
def test_prefill_edges(T, bits, pd, kv):
    say(f"[gpu] rows prefill T={T} bits={bits} pd={pd} kv={kv}")
    W, g, M = _model(bits, pd)
    pr = synth.make_prompt(W.cfg, 3, 20, seed=T)
    prior = (np.arange(T - 26, dtype=np.int32) * 13) % (W.cfg["mel_vocab"] - 2)
    cache, okv = g.kv_cache(400, kv), M.kv(400, kv_bf16=kv == H.ITTS_BF16)
    # a longer prompt first: what it leaves in the buffers must not reach the next one
    g.prefill_after(pr.text_tokens, pr.conds, pr.lang_id, np.zeros(T + 30, np.int32), cache)
    a = g.prefill_after(pr.text_tokens, pr.conds, pr.lang_id, prior, cache)
    b = M.prefill_after(okv, pr.text_tokens, pr.conds, pr.lang_id, prior)
    # 2e-5 with fp32 rows.  bf16 rows that lie near the middle of two values round the other way,
    # half a step (2^-9 of the value) apart: one logit in four layers of them moves by a few 1e-5
    # (3e-4 at the full depth of 24)
    tol = 2e-5 if kv == H.ITTS_F32 else 2e-4
    say(f"[gpu]   max |diff| {np.abs(a - b).max():.2e} of {np.abs(b).max():.2f}")
    assert np.abs(a - b).max() < tol * max(1.0, np.abs(b).max())
    s1, s2 = g.step(cache, 11, len(prior) + 2), M.step(okv, 11, len(prior) + 2)  # on the rows just written
    assert np.abs(s1 - s2).max() < tol * max(1.0, np.abs(s2).max())


# The products on fragment-order operands at 5 to 64 rows (QKV, c_proj, both MLP products and the
# all-row head), where no other entry point reaches them by themselves.
@pytest.mark.parametrize("bits,pd", [(8, H.ITTS_F16), (8, H.ITTS_F32), (4, H.ITTS_F16), (4, H.ITTS_F32)])
@pytest.mark.parametrize("T", [5, 8, 31, 32, 33, 64, 65])
def test_short_prompts_vs_fp64(T, bits, pd):
    say(f"[gpu] all-row logits of {T} rows, bits={bits} pd={pd}")
    W, g, M = _model(bits, pd)
    pr = synth.make_prompt(W.cfg, 0, min(T - 3, 20), seed=T)
    prior = (np.arange(max(0, T - 23), dtype=np.int32) * 13) % (W.cfg["mel_vocab"] - 2)
    emb = M.sequence_embedding(pr.text_tokens, pr.conds, pr.lang_id, prior)
    exact = numpy_forward(W, emb)
    got = g.forward_logits([H.CodePrompt(pr.text_tokens, pr.conds, pr.lang_id, prior)])
    assert len(got) == len(emb) == T
    rms = lambda a: float(np.sqrt(((a - exact) ** 2).mean()))  # noqa: E731
    # no further from float64 than twice the oracle's fp32 (its sums are fp32 too, one by one)
    assert rms(got) < 2 * rms(M.forward_rows(M.kv(128, kv_bf16=False), emb, 0)), rms(got)


# either side of where fp32 rows' attention and the LayerNorms change their form
@pytest.mark.parametrize("T", [384, 385, 512, 513])
@pytest.mark.parametrize("kv", [H.ITTS_F32, H.ITTS_BF16])
def test_prefill_route_edges(T, kv):
    say(f"[gpu] rows prefill T={T} kv={kv}")
    W, g, M = _model(8, H.ITTS_F32)
    pr = synth.make_prompt(W.cfg, 3, 20, seed=T)
    prior = (np.arange(T - 26, dtype=np.int32) * 13) % (W.cfg["mel_vocab"] - 2)
    cache, okv = g.kv_cache(640, kv), M.kv(640, kv_bf16=kv == H.ITTS_BF16)
    a = g.prefill_after(pr.text_tokens, pr.conds, pr.lang_id, prior, cache)
    b = M.prefill_after(okv, pr.text_tokens, pr.conds, pr.lang_id, prior)
    tol = 2e-5 if kv == H.ITTS_F32 else 2e-4  # (as in test_prefill_edges)
    assert np.abs(a - b).max() < tol * max(1.0, np.abs(b).max())
    s1, s2 = g.step(cache, 11, len(prior) + 2), M.step(okv, 11, len(prior) + 2)
    assert np.abs(s1 - s2).max() < tol * max(1.0, np.abs(s2).max())


def test_wide_model_without_folds():
    """d > 2048: the LayerNorms keep their row kernel."""
    over = (("n_layer", 2), ("d_model", 2112), ("n_head", 33), ("d_ffn", 128), ("text_vocab", 50), ("mel_vocab", 130))
    W, g, M = _model(8, H.ITTS_F16, over)
    pr = synth.make_prompt(W.cfg, 3, 60, seed=3)
    cache, okv = g.kv_cache(128, H.ITTS_F32), M.kv(128, kv_bf16=False)
    a = g.prefill(pr.text_tokens, pr.conds, pr.lang_id, cache)
    b = M.prefill_after(okv, pr.text_tokens, pr.conds, pr.lang_id)
    assert np.abs(a - b).max() < 2e-5 * max(1.0, np.abs(b).max())


def _one_block(**over):
    return dict(synth.TINY_CONFIG, n_layer=1, param_dtype=H.ITTS_F32, mel_pos_len=600, **over)


@pytest.mark.parametrize("kv", [H.ITTS_BF16, H.ITTS_F32])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_nonfinite_conditioning_reaches_the_logits(kv, bad):
    """A row that is not finite makes its K and V NaN, and with them every later row's attention;
    one block of two heads, so that nothing else can carry it there."""
    say(f"[gpu] prefill with a {bad} conditioning row, kv {kv}")
    for seed in range(8):
        W = synth.make_weights(_one_block(), seed=seed, init="rich")
        g = H.Gpt(W)
        for T in (24, 100, 450):
            pr = synth.make_prompt(W.cfg, 3, 15, seed=seed)
            pr.conds[1, 7] = bad
            cache = g.kv_cache(512, kv)
            prior = (np.arange(T - 21, dtype=np.int32) * 13) % (W.cfg["mel_vocab"] - 2)
            assert np.isnan(g.prefill_after(pr.text_tokens, pr.conds, pr.lang_id, prior, cache)).all(), (seed, T)
            assert np.isnan(g.step(cache, 5, T - 19)).all(), (seed, T)
        g.close()


@pytest.mark.parametrize("kv,T", [(H.ITTS_BF16, 40), (H.ITTS_BF16, 300), (H.ITTS_BF16, 500), (H.ITTS_F32, 40), (H.ITTS_F32, 384)])
@pytest.mark.parametrize("e", [14, 20])
def test_attention_of_scaled_q_and_k(kv, T, e):
    """q times 2^-e and K times 2^e are the same attention, to the bit: all of it is fp32 (or bf16
    rows) over its whole range."""
    say(f"[gpu] prefill T={T} kv {kv}, q and K scaled by 2^{e}")
    W = synth.make_weights(_one_block(), seed=3, init="rich")
    d = W.cfg["d_model"]
    got = []
    for scale in (1.0, 2.0**e):
        for L in W.layers:
            for a in (L.c_attn.scales, L.c_attn.biases, L.c_attn.bias):
                a[:d] *= np.float32(1.0 / scale)
                a[d:2 * d] *= np.float32(scale)
        g = H.Gpt(W)
        pr = synth.make_prompt(W.cfg, 3, 15, seed=1)
        prior = (np.arange(T - 21, dtype=np.int32) * 13) % (W.cfg["mel_vocab"] - 2)
        got.append(g.prefill_after(pr.text_tokens, pr.conds, pr.lang_id, prior, g.kv_cache(512, kv)))
        g.close()
    assert np.isfinite(got[0]).all() and np.array_equal(got[0], got[1]), float(np.abs(got[0] - got[1]).max())


def test_forward_logits_prompt_boundaries():
    """Prompts that start and end inside query and key tiles, one shorter than a tile."""
    W, g, M = _model(8, H.ITTS_F16)
    prompts = [H.CodePrompt(p.text_tokens, p.conds, p.lang_id, (np.arange(k, dtype=np.int32) * 7) % 1000)
               for p, k in ((synth.make_prompt(W.cfg, 3, n, seed=n), k) for n, k in ((5, 0), (30, 61), (2, 3), (40, 20)))]
    got = g.forward_logits(prompts)
    r = 0
    for p in prompts:
        emb = M.sequence_embedding(p.text_tokens, p.conds, p.lang_id, p.prior_codes)
        ref = M.forward_rows(M.kv(200, kv_bf16=False), emb, 0)
        assert np.abs(got[r:r + len(ref)] - ref).max() < 2e-5 * max(1.0, np.abs(ref).max())
        r += len(ref)
    assert r == len(got)


def test_long_k_split_over_blocks():
    """mlp c_proj with K >= 4096 and few tiles: K over several blocks, the counters reused."""
    over = (("n_layer", 2), ("d_ffn", 4160))
    W, g, M = _model(8, H.ITTS_F16, over)
    for n in (2, 40, 120):
        pr = synth.make_prompt(W.cfg, 3, n, seed=n)
        cache, okv = g.kv_cache(256, H.ITTS_F32), M.kv(256, kv_bf16=False)
        b = M.prefill_after(okv, pr.text_tokens, pr.conds, pr.lang_id)
        for _ in range(2):
            a = g.prefill(pr.text_tokens, pr.conds, pr.lang_id, cache)
            assert np.abs(a - b).max() < 2e-5 * max(1.0, np.abs(b).max())


# qlinear_forward: up to 8 rows the few-row product on row-major codes, up to 512 the 64 x 64 LDS
# tiles, then 32 x 64 tiles and (K >= 4096, many tiles) 64 x 64 on operands in fragment order
@pytest.mark.parametrize("bits,pd", [(8, H.ITTS_F16), (4, H.ITTS_F32)])
@pytest.mark.parametrize("M,N,K", [(2, 37, 192), (8, 130, 1280), (49, 37, 192), (65, 130, 64), (100, 1026, 1280), (70, 132, 4160),
                                   (512, 130, 64), (513, 130, 64), (545, 37, 192), (530, 132, 4160), (577, 1026, 1280),
                                   (2000, 1090, 4096)])
def test_product_vs_fp64(bits, pd, M, N, K):
    say(f"[gpu] rows product M={M} N={N} K={K} bits={bits}")
    _, g, _ = _model(8, H.ITTS_F16)
    rng = np.random.default_rng(M + N + K)
    w = (rng.standard_normal((N, K)) * 0.02).astype(np.float32)
    codes, s, b = H.quantize(w, bits, pd)
    bias = rng.standard_normal(N).astype(np.float32)
    x = rng.standard_normal((M, K)).astype(np.float32)
    got = g.qlinear_forward(codes, s, b, bias, x, N, K, bits, pd)
    Wd = ito.dequant(synth.QLinear(codes, s, b, bias, N, K), bits, pd).astype(np.float64)
    ref = x.astype(np.float64) @ Wd.T + bias
    # the tiled product's bar: 4e-6 of the sum of magnitudes (22-bit operands, fp32 sums)
    bound = np.abs(x).astype(np.float64) @ np.abs(Wd).T + np.abs(bias)
    assert np.all(np.abs(got - ref) <= 4e-6 * bound + 1e-7)


# b + 128 s (b + 8 s) far below fp16's normal range, and past its largest value; groups on one side of zero
@pytest.mark.parametrize("scale,offset", [(1e-5, 0.0), (1e-5, 90.0), (1e3, 0.0), (1e3, 90.0)])
@pytest.mark.parametrize("bits", [8, 4])
def test_product_range_of_f32_params(bits, scale, offset):
    _, g, _ = _model(8, H.ITTS_F16)
    M, N, K = 70, 130, 320
    rng = np.random.default_rng(5)
    codes, _, _ = H.quantize(rng.standard_normal((N, K)).astype(np.float32), bits, H.ITTS_F32)
    top = 2.0 ** bits
    s = (scale * rng.uniform(0.5, 1.5, (N, K // 64))).astype(np.float32)
    b = (s * (rng.uniform(-0.55, -0.45, s.shape) * top + offset * top / 256)).astype(np.float32)
    bias = np.zeros(N, np.float32)
    x = rng.standard_normal((M, K)).astype(np.float32)
    got = g.qlinear_forward(codes, s, b, bias, x, N, K, bits, H.ITTS_F32)
    Wd = ito.dequant(synth.QLinear(codes, s, b, bias, N, K), bits, H.ITTS_F32).astype(np.float64)
    ref = x.astype(np.float64) @ Wd.T
    bound = np.abs(x).astype(np.float64) @ np.abs(Wd).T
    # 22-bit operands and fp32 sums of the terms' magnitudes (codes and group sums, s times half the
    # code range an element)
    assert np.all(np.abs(got - ref) <= 4e-6 * (bound + scale * top / 2 * np.abs(x).sum(1, keepdims=True) / 8))


# activations of one sign: a group's sum is 64 of them, far past the range of an element
@pytest.mark.parametrize("big", [1.0, 1e4, 6e4])
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("M", [5, 40, 70, 600])
def test_product_of_one_signed_activations(bits, big, M):
    say(f"[gpu] product of activations around {big}, M={M} bits={bits}")
    _, g, _ = _model(8, H.ITTS_F16)
    N, K = 130, 1280
    rng = np.random.default_rng(M)
    codes, s, b = H.quantize((rng.standard_normal((N, K)) * 0.02).astype(np.float32), bits, H.ITTS_F32)
    x = (big * rng.uniform(0.9, 1.1, (M, K))).astype(np.float32)
    got = g.qlinear_forward(codes, s, b, np.zeros(N, np.float32), x, N, K, bits, H.ITTS_F32)
    Wd = ito.dequant(synth.QLinear(codes, s, b, np.zeros(N, np.float32), N, K), bits, H.ITTS_F32).astype(np.float64)
    bound = np.abs(x).astype(np.float64) @ np.abs(Wd).T
    # the products' bar (22-bit operands, fp32 sums), whatever the magnitude: below 65504 both
    # planes of an activation are in range
    assert np.all(np.abs(got - x.astype(np.float64) @ Wd.T) <= 4e-6 * bound)


@pytest.mark.parametrize("mean,outlier", [(0.0, 0.0), (100.0, 0.0), (0.0, 2e5)])
def test_long_prompt_of_uncentred_rows(mean, outlier):
    """Rows of a large mean, and one channel past the operand planes' range, at more than 512 rows:
    no further from float64 than the oracle's own fp32 rounding takes the oracle (twice its root
    mean square; the rounding of the residual rows, which both share, makes most of it)."""
    say(f"[gpu] 600 rows of mean {mean}, outlier channel {outlier}")
    W = synth.make_weights(dict(synth.SMALL_CONFIG, param_dtype=H.ITTS_F32), seed=23, init="rich")
    pr = synth.make_prompt(W.cfg, 3, 25, seed=1)
    for tab in (W.mel_emb, W.text_emb, W.lang_emb, pr.conds):
        tab += np.float32(mean)
        tab[:, 5] += np.float32(outlier)
    g, M = H.Gpt(W), ito.Model(W)
    prior = (np.arange(569, dtype=np.int32) * 13) % (W.cfg["mel_vocab"] - 2)
    emb = M.sequence_embedding(pr.text_tokens, pr.conds, pr.lang_id, prior)
    exact = numpy_forward(W, emb)
    rms = lambda a: float(np.sqrt(((a - exact) ** 2).mean()))  # noqa: E731
    bar = 2 * rms(M.forward_rows(M.kv(600, kv_bf16=False), emb, 0)) + 1e-7 * float(np.abs(exact).max())
    got = g.forward_logits([H.CodePrompt(pr.text_tokens, pr.conds, pr.lang_id, prior)])
    assert len(got) == len(emb) == 600 and rms(got) < bar, (rms(got), bar)
    last = g.prefill_after(pr.text_tokens, pr.conds, pr.lang_id, prior, g.kv_cache(600, H.ITTS_F32))
    err = np.abs(last - exact[-1]).max()
    assert err < 6 * bar, (float(err), bar)  # six standard deviations, of a thousand logits
    g.close()


@pytest.mark.parametrize("n_head", [1, 8, 9, 20, 21, 32, 33])
def test_layernorm_widths(n_head):
    """The row kernel's register widths and its last one, which reads rows again: one row, two, and
    an odd count, one LayerNorm and two (the all-row head)."""
    cfg = dict(synth.TINY_CONFIG, n_layer=1, d_model=64 * n_head, n_head=n_head, d_ffn=128, text_vocab=50, mel_vocab=130)
    W = synth.make_weights(cfg, seed=n_head, init="rich")
    g, M = H.Gpt(W), ito.Model(W)
    for n in (2, 3, 4):
        pr = synth.make_prompt(cfg, 0, n, seed=n)
        emb = M.sequence_embedding(pr.text_tokens, pr.conds, pr.lang_id, [])
        ref = M.forward_rows(M.kv(64, kv_bf16=False), emb, 0)
        got = g.forward_logits([H.CodePrompt(pr.text_tokens, pr.conds, pr.lang_id, None)])
        assert got.shape == ref.shape and np.abs(got - ref).max() < 2e-5 * max(1.0, np.abs(ref).max())
    g.close()
