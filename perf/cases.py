"""The work a speech program has this framework do, as cases that can be timed and checked.

A case is a dict of plain values.  ``prepare(case, seed)`` makes what the program holds
before the call (host arrays, as every entry point takes them; the decoder or estimator
with its weights laid out once; the KV caches), ``run(state)`` makes one pass through the
public entry points, and ``exact(case, seed)`` evaluates the same outputs in float64 with
plain torch.  The shapes are the reference architecture's: a 24-layer, d 1280 decoder with
quantised weights and the 13-layer, dim 512 CFM estimator, seeded random weights.

Kinds:
  prefill   one sentence's prompt (conditioning rows, text, codes already spoken) to the
            first logits: the time to the first token
  steps     a prompt, then decode steps one by one, each step's logits on the host (a
            program that samples by itself)
  batch     several sentences of different lengths prefilled and stepped together
  generate  a whole sentence on the device (greedy), then the text attention of its codes
            (word timings)
  replay    log-probabilities (and the text attention) of given codes, teacher-forced
  cfm       one evaluation of the CFM estimator
  solve     the CFM Euler solve with guidance: codes' conditioning to mel frames
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "index-tts-rs_amd"))

import itts_hip as H  # noqa: E402
from itts_hip import cfm as cfm_mod  # noqa: E402
from itts_hip import synth  # noqa: E402

D, HEADS, FFN, LAYERS, VOCAB = 1280, 20, 5120, 24, 8194
MAX_SEQ = 2048
ALIGN = ((4, 10), (5, 10))  # the default alignment heads


def listed():
    return [
        # a short sentence after the reference's three conditioning rows: latency
        dict(name="prefill_short", kind="prefill", bits=8, params="f32", kv="bf16", cond=3, text=19, prior=0),
        # a long sentence (the time to the first token of the headline workload)
        dict(name="prefill_long", kind="prefill", bits=8, params="f16", kv="bf16", cond=32, text=200, prior=0),
        # a sentence continued after codes already spoken, in the reference's cache type
        dict(name="prefill_after", kind="prefill", bits=8, params="f16", kv="f32", cond=32, text=150, prior=701),
        # the first tokens of a sentence, sampled by the caller; fp32 group parameters as
        # the shipped checkpoint has them
        dict(name="steps_start", kind="steps", bits=8, params="f32", kv="bf16", cond=32, text=64, prior=0, steps=24),
        # the same late in a long utterance
        dict(name="steps_late", kind="steps", bits=8, params="f16", kv="bf16", cond=32, text=200, prior=1001, steps=24),
        # four-bit weights
        dict(name="steps_int4", kind="steps", bits=4, params="f16", kv="bf16", cond=32, text=128, prior=0, steps=24),
        # eight sentences together
        dict(name="batch8", kind="batch", bits=8, params="f16", kv="bf16", cond=32, text=20, text_hi=200, batch=8, steps=24),
        # a whole short sentence on the device, then its word timings
        dict(name="generate", kind="generate", bits=8, params="f16", kv="f32", cond=32, text=40, new=64),
        # scoring a spoken sentence
        dict(name="replay", kind="replay", bits=8, params="f16", kv="f32", cond=32, text=150, codes=640, attention=True),
        # one evaluation for a short utterance, the guidance pair
        dict(name="cfm_short", kind="cfm", batch=2, frames=187),
        # 10 s of audio after a 2 s prompt
        dict(name="solve_10s", kind="solve", ref=172, gen=861, steps=25, rate=0.7),
        # 25 s of audio
        dict(name="solve_25s", kind="solve", ref=172, gen=2153, steps=25, rate=0.7),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(["prefill", "prefill", "steps", "batch", "generate", "replay", "cfm", "solve", "solve"])
    c = dict(kind=kind)
    if kind in ("prefill", "steps", "batch", "generate", "replay"):
        c.update(bits=rng.choice([8, 8, 4]), params=rng.choice(["f16", "f32"]), kv=rng.choice(["bf16", "f32"]),
                 cond=rng.choice([3, 32]))
    if kind == "prefill":
        c.update(text=_log(rng, 2, 600), prior=rng.choice([0, 0, _log(rng, 1, 1200)]))
    elif kind == "steps":
        c.update(text=_log(rng, 2, 300), prior=rng.choice([0, _log(rng, 1, 1400)]), steps=rng.randint(8, 32))
    elif kind == "batch":
        lo = _log(rng, 5, 100)
        c.update(text=lo, text_hi=lo + rng.randint(1, 150), batch=rng.randint(2, 8), steps=rng.randint(8, 32))
    elif kind == "generate":
        # caches of the reference's type: its greedy ids do not hang on roundings to bf16
        c.update(kv="f32", bits=8, text=_log(rng, 5, 200), new=_log(rng, 8, 64))
    elif kind == "replay":
        c.update(kv="f32", text=_log(rng, 5, 300), codes=_log(rng, 12, 1400), attention=rng.random() < 0.5)
    elif kind == "cfm":
        c.update(batch=rng.choice([1, 2]), frames=_log(rng, 40, 1500))
    else:
        c.update(ref=_log(rng, 60, 400), gen=_log(rng, 40, 1800), steps=rng.choice([10, 25]), rate=0.7)
    return c


# ---- what the program keeps: decoders and the estimator, one per weight set -------------
_kept = {}


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _normal(g, shape, std):
    return torch.randn(shape, generator=g, device=g.device, dtype=torch.float32) * std


def _tables():
    """Embedding tables, shared by the weight sets."""
    if "tables" not in _kept:
        g = torch.Generator(device=_device()).manual_seed(1)
        c = synth.FULL_CONFIG
        _kept["tables"] = [_normal(g, (c[k], D), 0.02).cpu().numpy()
                           for k in ("text_vocab", "lang_vocab", "mel_vocab", "mel_pos_len", "text_pos_len")]
    return _kept["tables"]


def _weights(bits, params):
    """Seeded decoder weights of the reference shape: N(0, 0.02) linears quantised per group
    of 64 (affine, min to max), LayerNorms around (1, 0)."""
    key = ("weights", bits, params)
    if key in _kept:
        return _kept[key]
    dev = _device()
    g = torch.Generator(device=dev).manual_seed(100 + bits)
    dt = torch.float16 if params == "f16" else torch.float32
    top = 2**bits - 1

    def ql(N, K):
        w = _normal(g, (N, K // 64, 64), 0.02)
        lo, hi = w.amin(-1), w.amax(-1)
        s, b = ((hi - lo) / top).to(dt), lo.to(dt)
        q = ((w - b.float()[..., None]) / s.float()[..., None]).round_().clamp_(0, top).to(torch.uint8).reshape(N, K)
        if bits == 4:
            q = q[:, 0::2] | (q[:, 1::2] << 4)
        host = lambda t: (t.view(torch.int16).cpu().numpy().view(np.uint16) if dt == torch.float16 else t.cpu().numpy())  # noqa: E731
        return synth.QLinear(np.ascontiguousarray(q.cpu().numpy()), np.ascontiguousarray(host(s)),
                             np.ascontiguousarray(host(b)), _normal(g, (N,), 0.02).cpu().numpy(), N, K)

    def ln():
        return (1.0 + _normal(g, (D,), 0.1)).cpu().numpy(), _normal(g, (D,), 0.1).cpu().numpy()

    layers = []
    for _ in range(LAYERS):
        l1, attn, proj = ln(), ql(3 * D, D), ql(D, D)
        l2, fc, mproj = ln(), ql(FFN, D), ql(D, FFN)
        layers.append(synth.Layer(*l1, attn, proj, *l2, fc, mproj))
    lf, fn = ln(), ln()
    cfg = dict(synth.FULL_CONFIG, quant_bits=bits, param_dtype=H.ITTS_F16 if params == "f16" else H.ITTS_F32)
    _kept[key] = synth.ModelWeights(cfg, *_tables(), layers, *lf, *fn, ql(VOCAB, D))
    return _kept[key]


def _gpt(case):
    key = ("gpt", case["bits"], case["params"])
    if key not in _kept:
        _kept[key] = H.Gpt(_weights(case["bits"], case["params"]))
    return _kept[key]


def _cfm_weights():
    if "cfm_w" not in _kept:
        _kept["cfm_w"] = synth.make_cfm_weights(cfm_mod.FULL_CONFIG, seed=3)
    return _kept["cfm_w"]


def _cfm():
    if "cfm" not in _kept:
        _kept["cfm"] = cfm_mod.CfmDit(_cfm_weights(), cfm_mod.FULL_CONFIG)
    return _kept["cfm"]


# ---- inputs -----------------------------------------------------------------------------
def _texts(case):
    """Text length of each sentence of a batch, spread over text..text_hi."""
    if case["kind"] != "batch":
        return [case["text"]]
    span = case["text_hi"] - case["text"] + 1
    return [case["text"] + (i * 83) % span for i in range(case["batch"])]


def _sentence(case, n_text, seed, i):
    g = np.random.default_rng([seed, i])
    return dict(text=g.integers(2, synth.FULL_CONFIG["text_vocab"], n_text).astype(np.int32),
                conds=g.standard_normal((case["cond"], D), dtype=np.float32),
                lang=int(g.integers(0, 4)),
                prior=g.integers(0, VOCAB - 2, case.get("prior", 0)).astype(np.int32),
                codes=g.integers(0, VOCAB - 2, case.get("codes", case.get("steps", 0))).astype(np.int32))


def _cfm_inputs(case, seed):
    c = cfm_mod.FULL_CONFIG
    if case["kind"] == "solve":
        return synth.make_cfm_inputs(c, case["ref"] + case["gen"], case["ref"], seed)
    g = np.random.default_rng([seed, 104729])
    B, T = case["batch"], case["frames"]
    x_t = g.standard_normal((B, T, c["in_ch"]), dtype=np.float32)
    merged = g.standard_normal((B, T, cfm_mod.merged_dim(c)), dtype=np.float32)
    merged[..., : c["in_ch"]] = x_t
    return dict(x_t=x_t, x_merged=merged, t=np.full(B, g.integers(0, 25) / 25.0, np.float32))


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("cfm", "solve"):
        return dict(kind=kind, case=case, model=_cfm(), inputs=_cfm_inputs(case, seed))
    gpt = _gpt(case)
    dtype = H.ITTS_BF16 if case["kv"] == "bf16" else H.ITTS_F32
    texts = _texts(case)
    return dict(kind=kind, case=case, model=gpt, sentences=[_sentence(case, n, seed, i) for i, n in enumerate(texts)],
                caches=[gpt.kv_cache(MAX_SEQ, dtype) for _ in texts])


def run(state):
    kind, case, m = state["kind"], state["case"], state["model"]
    if kind == "cfm":
        return m.forward_merged(**state["inputs"])
    if kind == "solve":
        return m.solve_euler(**state["inputs"], n_timesteps=case["steps"], cfg_rate=case["rate"])
    s, kv = state["sentences"][0], state["caches"][0]
    if kind == "prefill":
        return m.prefill_after(s["text"], s["conds"], s["lang"], s["prior"], kv)
    if kind == "steps":
        out = [m.prefill_after(s["text"], s["conds"], s["lang"], s["prior"], kv)]
        for i, tok in enumerate(s["codes"]):
            out.append(m.step(kv, int(tok), len(s["prior"]) + i + 2))
        return np.stack(out)
    if kind == "batch":
        out = [np.stack([m.prefill_after(q["text"], q["conds"], q["lang"], [], c)
                         for q, c in zip(state["sentences"], state["caches"])])]
        codes = np.stack([q["codes"] for q in state["sentences"]])
        for i in range(case["steps"]):
            out.append(H.step_batch(m, state["caches"], codes[:, i], np.full(len(codes), i + 2, np.int32)))
        return np.stack(out)
    if kind == "generate":
        p = H.SamplingParams(greedy=True, max_mel_tokens=case["new"])
        prompt = H.CodePrompt(s["text"], s["conds"], s["lang"], None, case["new"])
        codes = H.generate_codes_after(m, prompt, kv, p, H.SamplerRng(0))
        att = m.alignment_attention(s["text"], s["conds"], s["lang"], None, codes, kv)
        return dict(codes=codes, attention=att)
    lp, att = m.teacher_forced(s["text"], s["conds"], s["lang"], s["codes"], kv, attention=case["attention"])
    return dict(log_probs=lp, attention=att) if att is not None else dict(log_probs=lp)


# ---- what a pass cannot do without ------------------------------------------------------
def _decoder_bytes(case):
    n = LAYERS * (4 * D * D + 2 * D * FFN) + VOCAB * D
    group = 2 * (2 if case["params"] == "f16" else 4)
    return n * case["bits"] / 8 + n / 64 * group


def _rows_flops(T, head_rows, layers=LAYERS):
    """T causal rows through the blocks, head_rows of them through the head."""
    lin = 2.0 * T * layers * (4 * D * D + 2 * D * FFN)
    att = 2.0 * 2.0 * layers * D * (T * (T + 1) / 2)
    return lin + att + 2.0 * head_rows * D * VOCAB


def work(case):
    kind = case["kind"]
    if kind in ("cfm", "solve"):
        c = cfm_mod.FULL_CONFIG
        d, F, C, L, NL, K = c["dim"], c["inter"], c["in_ch"], c["n_layers"], c["wn_layers"], c["wn_kernel"]
        T = case["ref"] + case["gen"] if kind == "solve" else case["frames"]
        B, n = (2, case["steps"]) if kind == "solve" else (case["batch"], 1)
        blocks = L * (4 * d * d + 3 * d * F) + (L - L // 2 - 1) * 2 * d * d
        rest = d * cfm_mod.merged_dim(c) + d * (d + C) + 3 * d * d + d * C
        wave = NL * (2 * d * K * d + 2 * d * d) - d * d
        params = blocks + rest + wave + (2 * L + 1) * 2 * d * d + 2 * d * d * NL + 2 * d * d
        per = 2.0 * B * T * (blocks + rest + wave) + 4.0 * B * T * T * d * L
        io = 4.0 * B * T * (2 * C + cfm_mod.merged_dim(c))
        return dict(bytes=n * (4.0 * params + io), flops=n * per)
    W, row = _decoder_bytes(case), LAYERS * 2 * D * (2 if case["kv"] == "bf16" else 4)
    Ts = [case["cond"] + t + 3 + case.get("prior", 0) for t in _texts(case)]
    if kind == "replay":
        T = Ts[0] + case["codes"] - 1
        out = 4.0 * case["codes"] * (1 + (case["text"] + 2 if case["attention"] else 0))
        return dict(bytes=W + 4.0 * T * D + out, flops=_rows_flops(T, case["codes"]))
    n = case.get("steps", case.get("new", 1) - 1)
    nbytes = sum(W + T * row + 4.0 * T * D + 4.0 * VOCAB for T in Ts)
    flops = sum(_rows_flops(T, 1) for T in Ts)
    if kind != "prefill":
        for i in range(n):
            nbytes += W + sum((T + i + 2) * row + 4.0 * VOCAB for T in Ts)
            flops += sum(_rows_flops(1, 1) + 4.0 * LAYERS * D * (T + i) for T in Ts)
    if kind == "generate":
        T, last = Ts[0] + case["new"] - 1, 1 + max(l for l, _ in ALIGN)
        nbytes += W * last / LAYERS + 4.0 * case["new"] * (case["text"] + 2)
        flops += _rows_flops(T, 0, last)
    return dict(bytes=nbytes, flops=flops)


def tolerance(case):
    """About four times the largest distance from exact() measured over listed and drawn
    cases: 7.5e-6 for the estimator; 1e-6 for the decoder over fp32 rows, and up to 4e-4 over
    bf16 rows, where a key or value that lies near the middle of two bf16 values goes either
    way."""
    if case["kind"] in ("cfm", "solve"):
        return dict(rel=3e-5, max=1e-3)
    if case["kv"] == "bf16" and case["kind"] != "replay":
        return dict(rel=1.6e-3, max=2e-2)
    return dict(rel=5e-6, max=2e-4, differ=0.01)


# ---- the same in 64 bits, plain torch ---------------------------------------------------
def _t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(_device()).double()


def _dequant(q, bits):
    par = lambda a: _t(a.view(np.float16) if a.dtype == np.uint16 else a).repeat_interleave(64, 1)  # noqa: E731
    c = torch.from_numpy(q.codes).to(_device())
    if bits == 4:
        c = torch.stack([c & 15, c >> 4], -1).reshape(q.N, q.K)
    return par(q.scales) * c.double() + par(q.biases)


def _lnorm(x, w, b):
    m = x.mean(-1, keepdim=True)
    v = ((x - m) ** 2).mean(-1, keepdim=True)
    return (x - m) / torch.sqrt(v + 1e-5) * _t(w) + _t(b)


class _Exact:
    """Float64 decoder rows: a causal prompt, or further rows after kept K/V."""

    def __init__(self, case):
        self.W = _weights(case["bits"], case["params"])
        self.bits = case["bits"]
        self.round = case["kv"] == "bf16" and case["kind"] != "replay"
        self.mats = {}

    def lin(self, q, x):
        if id(q) not in self.mats:
            self.mats[id(q)] = (_dequant(q, self.bits).t().contiguous(), _t(q.bias))
        w, b = self.mats[id(q)]
        return x @ w + b

    def embed(self, s, prior):
        W, n = self.W, len(s["text"]) + 2
        u = np.concatenate([[0], s["text"], [1]])
        rows = [_t(s["conds"]), _t(W.text_emb[u]) + _t(W.lang_emb[s["lang"]]) + _t(W.text_pos[:n]),
                _t(W.mel_emb[VOCAB - 2][None]) + _t(W.mel_pos[:1])]
        if len(prior):
            rows.append(_t(W.mel_emb[prior]) + _t(W.mel_pos[2:2 + len(prior)]))
        return torch.cat(rows)

    def rows(self, x, kept=None, layers=LAYERS, probes=(), cols=None):
        """Blocks over rows x; kept: per-layer (k, v) to attend to and extend."""
        T, att = x.shape[0], []
        for i, L in enumerate(self.W.layers[:layers]):
            qkv = self.lin(L.c_attn, _lnorm(x, L.ln1_w, L.ln1_b)).reshape(T, 3, HEADS, 64).permute(1, 2, 0, 3).contiguous()
            q, k, v = qkv[0], qkv[1], qkv[2]
            if self.round:
                k, v = (z.float().bfloat16().double() for z in (k, v))
            if kept is not None:
                if i < len(kept):
                    k, v = torch.cat([kept[i][0], k], 1), torch.cat([kept[i][1], v], 1)
                    kept[i] = (k, v)
                else:
                    kept.append((k, v))
            n = k.shape[1]
            sc = torch.matmul(q, k.transpose(1, 2).contiguous()) * 0.125
            mask = torch.arange(n, device=x.device)[None] > torch.arange(n - T, n, device=x.device)[:, None]
            p = torch.softmax(sc.masked_fill_(mask, -math.inf), -1)
            att += [p[h][:, cols[0]:cols[1]] for l, h in probes if l == i]
            a = torch.matmul(p, v).permute(1, 0, 2).reshape(T, D)
            del sc, p
            x = x + self.lin(L.c_proj, a)
            f = self.lin(L.c_fc, _lnorm(x, L.ln2_w, L.ln2_b))
            f = 0.5 * f * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (f + 0.044715 * f**3)))
            x = x + self.lin(L.mlp_c_proj, f)
        return x, att

    def head(self, x):
        W = self.W
        return self.lin(W.head, _lnorm(_lnorm(x, W.ln_f_w, W.ln_f_b), W.fn_w, W.fn_b))

    def attention(self, s, codes):
        n0 = len(s["conds"])
        emb = self.embed(s, codes[:-1])
        _, att = self.rows(emb, layers=1 + max(l for l, _ in ALIGN), probes=ALIGN, cols=(n0, n0 + len(s["text"]) + 2))
        return (sum(att) / len(att))[-len(codes):]


def _np(t):
    return t.cpu().numpy()


def _exact_cfm(x_t, merged, t, W):
    """The estimator in float64; W: name -> float64 tensor."""
    c = cfm_mod.FULL_CONFIG
    d, heads, L = c["dim"], c["n_heads"], c["n_layers"]
    B, T = x_t.shape[:2]
    silu = torch.nn.functional.silu
    lin = lambda x, n, b=True: x @ W[n + ".weight"].reshape(W[n + ".weight"].shape[0], -1).t() + (W[n + ".bias"] if b else 0.0)  # noqa: E731

    def temb(p):
        k = torch.arange(128, device=t.device, dtype=torch.float64)
        a = t[:, None] * (1000.0 * torch.exp(-math.log(10000.0) * k / 128))
        return lin(silu(lin(torch.cat([a.cos(), a.sin()], -1), p + ".mlp.layers.0")), p + ".mlp.layers.2")

    t1, t2 = temb("t_embedder"), temb("t_embedder2")

    def adaln(x, p):
        w, b = lin(t1, p + ".project_layer")[:, None].chunk(2, -1)
        return w * (x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * W[p + ".norm.weight"]) + b

    ang = torch.arange(T, device=t.device, dtype=torch.float64)[:, None] / 10000.0 ** (
        torch.arange(32, device=t.device, dtype=torch.float64) * 2 / 64)
    cos, sin = ang.cos(), ang.sin()

    def rope(x):  # [B, heads, T, 64]
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).reshape(x.shape)

    h, skips = lin(merged, "cond_x_merge_linear"), []
    for i in range(L):
        p = "transformer.layers.%d" % i
        if i > L // 2:
            h = lin(torch.cat([h, skips.pop()], -1), p + ".skip_in_linear")
        qkv = lin(adaln(h, p + ".attention_norm"), p + ".attention.wqkv", False)
        q, k, v = (z.reshape(B, T, heads, 64).transpose(1, 2).contiguous() for z in qkv.chunk(3, -1))
        a = torch.softmax(torch.matmul(rope(q), rope(k).transpose(2, 3).contiguous()) * 0.125, -1)
        h = h + lin(torch.matmul(a, v).transpose(1, 2).reshape(B, T, d), p + ".attention.wo", False)
        n = adaln(h, p + ".ffn_norm")
        f = p + ".feed_forward."
        h = h + lin(silu(lin(n, f + "w1", False)) * lin(n, f + "w3", False), f + "w2", False)
        if i < L // 2:
            skips.append(h)
    x_res = lin(torch.cat([adaln(h, "transformer.norm"), x_t], -1), "skip_linear")
    hw, out = lin(x_res, "conv1"), 0.0
    g = lin(t2, "wavenet.cond_layer")
    for l in range(c["wn_layers"]):
        n, K = "wavenet.in_layers.%d" % l, c["wn_kernel"]
        pad = torch.nn.functional.pad(hw, (0, 0, K // 2, K // 2))
        acts = W[n + ".bias"] + g[:, None, l * 2 * d:(l + 1) * 2 * d]
        for j in range(K):
            acts = acts + pad[:, j:j + T] @ W[n + ".weight"][:, j].t()
        rs = lin(torch.tanh(acts[..., :d]) * torch.sigmoid(acts[..., d:]), "wavenet.res_skip_layers.%d" % l)
        if l + 1 == c["wn_layers"]:
            out = out + rs
        else:
            hw, out = hw + rs[..., :d], out + rs[..., d:]
    h = out + lin(x_res, "res_projection")
    shift, scale = lin(silu(t1), "final_layer.adaLN_modulation.layers.1")[:, None].chunk(2, -1)
    h = torch.nn.functional.layer_norm(h, (d,), eps=1e-6) * (1.0 + scale) + shift
    return lin(lin(h, "final_layer.linear"), "conv2").transpose(1, 2)


def exact(case, seed):
    kind = case["kind"]
    with torch.no_grad():
        if kind in ("cfm", "solve"):
            W = {n: _t(a) for n, a in _cfm_weights().items()}
            inp = {k: _t(v) for k, v in _cfm_inputs(case, seed).items()}
            if kind == "cfm":
                return _np(_exact_cfm(inp["x_t"], inp["x_merged"], inp["t"], W))
            c, T, R, n = cfm_mod.FULL_CONFIG, case["ref"] + case["gen"], case["ref"], case["steps"]
            x = inp["noise_z"][0].t().contiguous()  # [T, in_ch]
            tail = x.new_zeros(2, T, c["in_ch"] + c["dim"] + c["style_dim"])
            tail[0, :R, : c["in_ch"]] = inp["ref_mel"][0].t()
            tail[:, :, c["in_ch"]:c["in_ch"] + c["dim"]] = W["cond_projection.bias"]
            tail[0, :, c["in_ch"]:c["in_ch"] + c["dim"]] += inp["cat_condition"][0] @ W["cond_projection.weight"].t()
            tail[0, :, c["in_ch"] + c["dim"]:] = inp["style"][0]
            for i in range(n):
                x[:R] = 0.0
                x_t = torch.stack([x, x])
                v = _exact_cfm(x_t, torch.cat([x_t, tail], -1), x.new_full((2,), i / n), W).transpose(1, 2)
                x = x + (v[0] * (1.0 + case["rate"]) - v[1] * case["rate"]) / n
            return _np(x[R:].t().contiguous()[None])
        E = _Exact(case)
        sent = [_sentence(case, n, seed, i) for i, n in enumerate(_texts(case))]
        s = sent[0]
        if kind == "prefill":
            x, _ = E.rows(E.embed(s, s["prior"]))
            return _np(E.head(x[-1:])[0])
        if kind in ("steps", "batch"):
            per = []
            for q in sent:
                codes = np.concatenate([q["prior"], q["codes"]])
                x, _ = E.rows(E.embed(q, codes))
                per.append(_np(E.head(x[-(case["steps"] + 1):])))
            return per[0] if kind == "steps" else np.stack(per, 1)
        if kind == "generate":
            kept, codes, seen = [], [], [1, VOCAB - 2]
            x, _ = E.rows(E.embed(s, []), kept)
            for i in range(case["new"]):
                lg = E.head(x[-1:])[0]
                lg[VOCAB - 1] = -math.inf
                idx = torch.tensor(seen, device=lg.device)
                lg[idx] = torch.where(lg[idx] < 0, lg[idx] * 10.0, lg[idx] / 10.0)
                codes.append(int(lg.argmax()))
                seen.append(codes[-1])
                if i + 1 < case["new"]:
                    x, _ = E.rows(_t(E.W.mel_emb[codes[-1]] + E.W.mel_pos[i + 2])[None], kept)
            codes = np.array(codes, np.int32)
            return dict(codes=codes, attention=_np(E.attention(s, codes)))
        x, _ = E.rows(E.embed(s, s["codes"][:-1]))
        lp = torch.log_softmax(E.head(x[-case["codes"]:]), -1)
        lp = _np(lp[torch.arange(case["codes"]), torch.from_numpy(s["codes"]).long()])
        return dict(log_probs=lp, attention=_np(E.attention(s, s["codes"]))) if case["attention"] else dict(log_probs=lp)
