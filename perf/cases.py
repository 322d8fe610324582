"""Performance cases of the framework: what users run, through its public entry points.

A case is a dict of plain values; ``kind`` names the path:

  qmv        one quantised projection of a decode step, called by itself
  head       end of a decode step: final norm + LM head, then one sampled token
  attention  single-query GQA attention over a given KV cache
  layers     a run of decoder layers at one position (operator API, captured graph)
  gemm       one prefill projection (dequant-GEMM) over a prompt
  prefill    a prompt through a decoder model
  generate   a whole chat turn: prefill, then greedy decoding
  stacked    one launch over many independent matrices of one shape

Shapes are the Bonsai 1.7B / 4B / 8B layers of the presets and the workloads of
configs.py and bench.py, plus odd sizes around them.  Weights and inputs are
drawn from the seed; scales are of the size trained group-quantised checkpoints
have, 4-bit biases sit near -7.5 scale so that weights have mean zero.
"""
import ctypes as C
import math

import numpy as np
import torch

from nnzap_amd import _lib as L
from nnzap_amd import configs as cf
from nnzap_amd import formats as fm
from nnzap_amd import model as md
from nnzap_amd import ops

# hidden, MLP, query heads, KV heads, head_dim
SHAPES = {"1.7b": (2048, 6144, 16, 8, 128), "4b": (2560, 9728, 32, 8, 128), "8b": (4096, 12288, 32, 8, 128)}
GROUP = {1: 128, 4: 64}
THETA, EPS = 1.0e6, 1e-6
BLOCK_VOCAB = 512          # vocabulary of the cases that measure layers and not the head
_dev = None


def device():
    """The context that every case runs on (a program keeps one per GPU)."""
    global _dev
    if _dev is None:
        _dev = ops.Device(0)
    return _dev


def listed():
    return [
        # the smallest call: one 1-bit attention output projection (8B shape) on its own, as
        # an operator-API program issues it (bound by the call and the launch)
        dict(name="qmv_q1_small", kind="qmv", bits=1, M=4096, K=4096, form="f16io"),
        # the end of every decode step of the 1-bit 1.7B model (vocabulary 151669 of the
        # Bonsai presets) with the sampling settings of a chat program
        dict(name="head_q1_sampled", kind="head", bits=1, V=151669, K=2048, temperature=0.6, top_k=20, top_p=0.95),
        # decode attention over a full 32k context, bf16 cache (the longest)
        dict(name="attention_bf16_32k", kind="attention", L=32768, hq=16, hkv=8, kv="bf16", transposed=False),
        # decode in the middle of a long chat on the 8B layer shape, 1-bit
        dict(name="layers_q1_8b_3001", kind="layers", bits=1, shape="8b", layers=4, seq=3001),
        # decode of a short chat on the 4-bit 1.7B layer shape
        dict(name="layers_q4_1p7b_200", kind="layers", bits=4, shape="1.7b", layers=8, seq=200),
        # down projection of the 8B shape over a one-line prompt (45 tokens, less than one token tile)
        dict(name="gemm_q1_down_45", kind="gemm", bits=1, P=45, M=4096, K=12288, mode="f32"),
        # 4-bit gate/up projections of the 1.7B shape over the 512-token prompt of the benchmark
        dict(name="gemm_q4_gate_up_512", kind="gemm", bits=4, P=512, M=6144, K=2048, mode="silu"),
        # a long document through 4B-shaped layers: ragged length, attention weighs in
        dict(name="prefill_q1_4b_3001", kind="prefill", bits=1, shape="4b", layers=2, P=3001, vocab=BLOCK_VOCAB),
        # whole call: the benchmark's 512-token prompt through the full 1.7B model
        dict(name="prefill_q1_1p7b_512", kind="prefill", bits=1, shape="1.7b", layers=28, P=512, vocab=151669),
        # whole call: a chat turn with the full 1.7B model, 40 prompt tokens, 48 new ones
        dict(name="generate_q1_1p7b", kind="generate", bits=1, shape="1.7b", layers=28, P=40, new=48, vocab=151669),
        # 256 independent 1-bit down projections in one launch (the benchmark's stacked config 2)
        dict(name="stacked_q1_down", kind="stacked", form="q1", M=2048, K=6144, count=256),
        # 256 independent 4-bit gate projections in one launch (the benchmark's stacked config 1)
        dict(name="stacked_q4_gate", kind="stacked", form="q4", M=6144, K=2048, count=256),
    ]


def draw(rng):
    def logint(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["qmv", "head", "attention", "layers", "gemm", "gemm", "prefill", "prefill", "generate", "stacked"])
    bits = rng.choice([1, 1, 4])
    shape = rng.choice(sorted(SHAPES))
    H, I, hq, hkv, D = SHAPES[shape]
    if kind == "qmv":
        return dict(kind=kind, bits=bits, M=logint(256, 12288), K=128 * rng.randint(4, 64), form=rng.choice(["f16io", "f32"]))
    if kind == "head":
        k, p = rng.choice([(0, 1.0), (20, 0.95), (40, 0.95), (50, 1.0), (0, 0.9)])
        return dict(kind=kind, bits=bits, V=rng.randint(32000, 151936), K=rng.choice([2048, 2560, 4096]),
                    temperature=rng.choice([0.6, 0.7, 1.0]), top_k=k, top_p=p)
    if kind == "attention":
        g = rng.choice([2, 4])
        kv, transposed = rng.choice([("bf16", False), ("f16", True)])
        return dict(kind=kind, L=logint(64, 32768), hq=8 * g, hkv=8, kv=kv, transposed=transposed)
    if kind == "layers":
        # 4-bit projections of a decode step take rows of up to 8192 columns: the 1.7B shape
        return dict(kind=kind, bits=bits, shape=shape if bits == 1 else "1.7b", layers=4, seq=logint(16, 8192))
    if kind == "gemm":
        M, K = rng.choice([(hq * D, H), (hkv * D, H), (H, hq * D), (I, H), (H, I)])
        mode = "silu" if M == I else rng.choice(["f16", "f32"])
        return dict(kind=kind, bits=bits, P=logint(8, 2048), M=M, K=K, mode=mode)
    if kind == "prefill":
        return dict(kind=kind, bits=bits, shape=shape, layers=2, P=logint(8, 3001), vocab=BLOCK_VOCAB)
    if kind == "generate":
        return dict(kind=kind, bits=1, shape="1.7b", layers=rng.randint(4, 28), P=logint(8, 128), new=rng.randint(8, 48), vocab=rng.randint(32000, 151936))
    M, K = 8 * rng.randint(64, 1024), rng.choice([2048, 4096, 6144])
    form = rng.choice(["q1", "q4", "silu"])
    per = M * K * {"q1": 1, "q4": 4, "silu": 2}[form] // 8
    return dict(kind=kind, form=form, M=M, K=K, count=rng.randint(8, max(8, min(256, 400_000_000 // per))))


# ------------------------------------------------------------------- weights
def _bf16_bits(x):
    return torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32)).to(torch.bfloat16).view(torch.int16).numpy().view(np.uint16)


def _matrix(rng, bits, M, K, lo=None, hi=None):
    """A group-quantised matrix: uniform codes, scales U(lo, hi)."""
    gs = GROUP[bits]
    codes = rng.integers(0, 1 << 32, (M, K * bits // 32), dtype=np.uint32)
    lo, hi = (lo, hi) if lo else ((0.005, 0.025) if bits == 1 else (0.001, 0.005))
    s = rng.uniform(lo, hi, (M, K // gs)).astype(np.float32)
    if bits == 1:
        return fm.QWeight(1, M, K, gs, codes, fm.f16_bits(s), None, fm.DT_F16)
    b = -7.5 * s * rng.uniform(0.9, 1.1, s.shape).astype(np.float32)
    return fm.QWeight(4, M, K, gs, codes, _bf16_bits(s), _bf16_bits(b), fm.DT_BF16)


def _norm(rng, n):
    return (1.0 + 0.1 * rng.standard_normal(n)).astype(np.float32)


def _layer(rng, bits, shape):
    H, I, hq, hkv, D = SHAPES[shape]
    dims = {"q": (hq * D, H), "k": (hkv * D, H), "v": (hkv * D, H), "o": (H, hq * D), "gate": (I, H), "up": (I, H), "down": (H, I)}
    w = {n: _matrix(rng, bits, *dims[n]) for n in cf.PROJS}
    w.update(attn_norm=_norm(rng, H), ffn_norm=_norm(rng, H), q_norm=_norm(rng, D), k_norm=_norm(rng, D))
    return w


def _weights(case, seed):
    """(config, weights) of a decoder model.  Row t + 1 of the LM head has the codes of
    token t's embedding, so the model is as sure of its next token as a trained one is of
    plain text: with unrelated rows the best two logits nearly tie at every step, and a
    greedy text would hang on single roundings."""
    rng = np.random.default_rng([seed, 5])
    bits, V = case["bits"], case["vocab"]
    H, I, hq, hkv, D = SHAPES[case["shape"]]
    ctx = -(-(case["P"] + case.get("new", 0)) // 8) * 8
    cfg = cf.DecoderConfig(vocab_size=V, hidden_size=H, intermediate_size=I, num_layers=case["layers"], num_query_heads=hq,
                           num_kv_heads=hkv, head_dim=D, max_context_length=ctx, max_prefill_length=case["P"],
                           group_size=GROUP[bits], rope_theta=THETA, rms_eps=EPS, embed_kind=L.EMBED_Q1 if bits == 1 else L.EMBED_Q4,
                           lm_head_kind=L.LMHEAD_Q1 if bits == 1 else L.LMHEAD_Q4, quant_format=0 if bits == 1 else 1)
    w = cf.DecoderWeights(cfg)
    w.embed_q1 = _matrix(rng, bits, V, H, 0.5, 1.5) if bits == 1 else _matrix(rng, bits, V, H, 0.1, 0.3)
    w.lm_head = _matrix(rng, bits, V, H)
    w.lm_head.codes = np.roll(w.embed_q1.codes, 1, axis=0)
    w.final_norm = _norm(rng, H)
    w.layers = [_layer(rng, bits, case["shape"]) for _ in range(case["layers"])]
    return cfg, w


def _prompt(case, seed):
    return np.random.default_rng([seed, 6]).integers(0, case["vocab"] - case.get("new", 0) - 1, case["P"]).astype(np.uint32)


def _gpu(x):
    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


class _Graph:
    """A captured run of operator calls."""

    def __init__(self, dev, body):
        self.dev, self.g = dev, C.c_void_p()
        body()          # once uncaptured, as a program warms up
        dev.sync()
        dev.call("nnz_graph_begin")
        try:
            body()
        finally:
            dev.call("nnz_graph_end", C.byref(self.g))

    def replay(self):
        self.dev.call("nnz_graph_replay", self.g)

    def __del__(self):
        if self.g:
            L.lib().nnz_graph_destroy(self.g)


# ------------------------------------------------------------------- prepare
def prepare(case, seed):
    dev = device()
    with torch.cuda.stream(dev.stream):
        return globals()["_prepare_" + case["kind"]](dev, case, seed)


def _prepare_qmv(dev, case, seed):
    rng = np.random.default_rng([seed, 1])
    w = _matrix(rng, case["bits"], case["M"], case["K"])
    dt = np.float16 if case["form"] == "f16io" else np.float32
    x = rng.standard_normal(case["K"]).astype(dt)
    y = torch.empty(case["M"], dtype=torch.float16 if dt == np.float16 else torch.float32, device="cuda")
    fn = {(1, "f16io"): ops.dispatch_qmv_f16io, (1, "f32"): ops.dispatch_qmv,
          (4, "f16io"): ops.dispatch_q4mv_f16io, (4, "f32"): ops.dispatch_q4mv}[case["bits"], case["form"]]
    return dict(case=case, host=w, w=ops.DeviceQWeight(dev, w), x=_gpu(x), y=y, fn=fn)


def _prepare_head(dev, case, seed):
    rng = np.random.default_rng([seed, 2])
    V, K = case["V"], case["K"]
    w = _matrix(rng, case["bits"], V, K)
    xn = torch.empty(K, dtype=torch.float16, device="cuda")
    state = torch.zeros(4, dtype=torch.int64, device="cuda")
    ops.rng_seed(dev, seed, state)
    return dict(case=case, host=w, w=ops.DeviceQWeight(dev, w), res=_gpu(2.0 * rng.standard_normal(K).astype(np.float32)),
                norm=_gpu(3.0 * _norm(rng, K)), xn=xn, logits=torch.empty(V, dtype=torch.float32, device="cuda"), rng=state,
                ws=torch.empty(ops.sample_workspace_bytes(V), dtype=torch.uint8, device="cuda"),
                token=torch.zeros(1, dtype=torch.int32, device="cuda"), prob=torch.zeros(1, dtype=torch.float32, device="cuda"))


def _prepare_attention(dev, case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    n, hq, hkv, D = case["L"], case["hq"], case["hkv"], 128
    ctx = -(-n // 8) * 8
    dt = torch.bfloat16 if case["kv"] == "bf16" else torch.float16
    randn = lambda *s: torch.randn(*s, generator=g, device="cuda").to(dt)  # noqa: E731
    dims = L.GQADims(hq, hkv, D, n, ctx, hq // hkv)
    return dict(case=case, q=randn(hq, D), k=randn(hkv, ctx, D), v=randn(*((hkv, D, ctx) if case["transposed"] else (hkv, ctx, D))),
                out=torch.empty(hq, D, dtype=torch.float32, device="cuda"), dims=dims,
                scratch=torch.zeros(ops.gqa_scratch_bytes(dims), dtype=torch.uint8, device="cuda"))


def _prepare_layers(dev, case, seed):
    rng = np.random.default_rng([seed, 3])
    bits, seq = case["bits"], case["seq"]
    H, I, hq, hkv, D = SHAPES[case["shape"]]
    ctx = -(-seq // 8) * 8
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    emb = _matrix(rng, bits, BLOCK_VOCAB, H, 0.5 if bits == 1 else 0.1, 1.5 if bits == 1 else 0.3)
    host = [_layer(rng, bits, case["shape"]) for _ in range(case["layers"])]
    lay = []
    for w in host:
        d = {n: ops.DeviceQWeight(dev, w[n]) for n in cf.PROJS}
        d.update({n: _gpu(w[n]) for n in ("attn_norm", "ffn_norm", "q_norm", "k_norm")})
        d["k"], d["wk"] = torch.randn(hkv, ctx, D, generator=g, device="cuda").half(), d["k"]
        d["v"], d["wv"] = torch.randn(hkv, D, ctx, generator=g, device="cuda").half(), d["v"]
        lay.append(d)
    h16 = lambda n: torch.zeros(n, dtype=torch.float16, device="cuda")  # noqa: E731
    s = dict(case=case, host=host, emb_host=emb, emb=ops.DeviceQWeight(dev, emb), layers=lay, id=int(rng.integers(BLOCK_VOCAB)),
             res=torch.zeros(H, device="cuda"), q=h16(hq * D), k=h16(hkv * D), v=h16(hkv * D), att=h16(hq * D), act=h16(I),
             dims=L.GQAFusedDims(hq, hkv, D, seq, ctx, hq // hkv, seq - 1, EPS, THETA))
    s["ids"] = torch.tensor([s["id"]], dtype=torch.int32, device="cuda")
    s["scratch"] = torch.zeros(ops.gqa_scratch_bytes(L.GQADims(hq, hkv, D, seq, ctx, hq // hkv)), dtype=torch.uint8, device="cuda")

    def step():
        ed = L.EmbedDims(BLOCK_VOCAB, H, 1, GROUP[bits])
        e = s["emb"]
        if bits == 1:
            ops.dispatch_embedding_lookup(dev, s["ids"], e.codes, e.scales, s["res"], ed)
        else:
            ops.dispatch_embedding_lookup_q4(dev, s["ids"], e.codes, e.scales, e.biases, s["res"], ed)
        for d in s["layers"]:
            if bits == 1:
                ops.dispatch_fused_norm_qkv_f16io(dev, d["q"], d["wk"], d["wv"], s["res"], s["q"], s["k"], s["v"], d["attn_norm"])
            else:
                ops.dispatch_q4_fused_norm_qmv_f16io(dev, d["q"], s["res"], s["q"], d["attn_norm"])
                ops.dispatch_q4_fused_norm_pair_qmv_f16io(dev, d["wk"], d["wv"], s["res"], s["k"], s["v"], d["attn_norm"])
            ops.dispatch_gqa_attention_fused_1pass(dev, s["q"], d["k"], d["v"], s["att"], s["k"], s["v"], d["q_norm"], d["k_norm"],
                                                   s["scratch"], s["dims"])
            if bits == 1:
                ops.dispatch_qmv_f16io_resadd(dev, d["o"], s["att"], s["res"])
                ops.dispatch_fused_norm_pair_silu_f16io(dev, d["gate"], d["up"], s["res"], s["act"], d["ffn_norm"])
                ops.dispatch_qmv_f16io_resadd(dev, d["down"], s["act"], s["res"])
            else:
                ops.dispatch_q4mv_f16io_resadd(dev, d["o"], s["att"], s["res"])
                ops.dispatch_q4_fused_norm_pair_silu_f16io(dev, d["gate"], d["up"], s["res"], s["act"], d["ffn_norm"])
                ops.dispatch_q4mv_f16io_resadd(dev, d["down"], s["act"], s["res"])

    torch.cuda.synchronize()
    s["graph"] = _Graph(dev, step)
    return s


_MODES = {"f16": L.GEMM_STORE_F16, "f32": L.GEMM_STORE_F32, "silu": L.GEMM_SILU_PAIR}


def _prepare_gemm(dev, case, seed):
    rng = np.random.default_rng([seed, 4])
    P, M, K = case["P"], case["M"], case["K"]
    host = [_matrix(rng, case["bits"], M, K) for _ in range(2 if case["mode"] == "silu" else 1)]
    a = _gpu(rng.standard_normal((P, K), dtype=np.float32).astype(np.float16))
    out = torch.empty(P, M, dtype=torch.float32 if case["mode"] == "f32" else torch.float16, device="cuda")
    return dict(case=case, host=host, w=[ops.DeviceQWeight(dev, h) for h in host], a=a, out=out)


def _prepare_prefill(dev, case, seed):
    cfg, w = _weights(case, seed)
    m = md.DecoderModel(dev, cfg)
    m.load(w)
    return dict(case=case, host=w, model=m, prompt=_prompt(case, seed))


_prepare_generate = _prepare_prefill


def _prepare_stacked(dev, case, seed):
    M, K, n, form = case["M"], case["K"], case["count"], case["form"]
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    x = torch.randn(n, K, generator=g, device="cuda")
    y = torch.empty(n, M, device="cuda")
    if form == "q4":
        w = [ops.StackedQWeights(dev, M, K, 64, 4, n, seed, scale_range=(0.001, 0.005), bias_range=(-0.04, 0.004))]
    else:
        w = [ops.StackedQWeights(dev, M, K, 128, 1, n, seed + 7919 * i, scale_range=(0.005, 0.025)) for i in range(2 if form == "silu" else 1)]
    return dict(case=case, w=w, x=x, y=y)


# ----------------------------------------------------------------------- run
def run(s):
    return globals()["_run_" + s["case"]["kind"]](device(), s)


def _run_qmv(dev, s):
    s["fn"](dev, s["w"], s["x"], s["y"])
    return s["y"]


def _run_head(dev, s):
    c = s["case"]
    if c["bits"] == 1:
        ops.dispatch_fused_norm_qmv_f16in(dev, s["w"], s["res"], s["logits"], s["norm"])
    else:
        ops.dispatch_rms_norm(dev, s["res"], s["norm"], s["xn"], c["K"], 1, EPS, bf16_trunc=True)
        ops.dispatch_q4mv_f16in(dev, s["w"], s["xn"], s["logits"])
    ops.dispatch_sample(dev, s["logits"], s["token"], s["rng"], s["ws"], c["temperature"], c["top_k"], c["top_p"], s["prob"])
    return {"logits": s["logits"], "token": s["token"], "prob": s["prob"]}


def _run_attention(dev, s):
    c = s["case"]
    ops.dispatch_gqa_attention(dev, s["q"], s["k"], s["v"], s["out"], s["scratch"], s["dims"], v_transposed=c["transposed"],
                               rope_position=c["L"] - 1, rope_theta=THETA)
    return s["out"]


def _run_layers(dev, s):
    s["graph"].replay()
    return {"residual": s["res"], "k": [d["k"] for d in s["layers"]], "v": [d["v"] for d in s["layers"]]}


def _run_gemm(dev, s):
    w = s["w"]
    ops.dispatch_dequant_gemm(dev, w[0], s["a"], s["out"], _MODES[s["case"]["mode"]], w[1] if len(w) > 1 else None)
    return s["out"]


def _run_prefill(dev, s):
    return s["model"].prefill(s["prompt"])


def _run_generate(dev, s):
    tokens, margins, _ = s["model"].generate(s["prompt"], s["case"]["new"])
    return {"tokens": tokens.astype(np.int64), "margins": margins, "logits": s["model"].download(md.T_LOGITS)}


def _run_stacked(dev, s):
    f = s["case"]["form"]
    if f == "q1":
        ops.dispatch_qmv_stacked(dev, s["w"][0], s["x"], s["y"])
    elif f == "q4":
        ops.dispatch_q4mv_stacked(dev, s["w"][0], s["x"], s["y"])
    else:
        ops.dispatch_qmv_fused_pair_silu_stacked(dev, s["w"][0], s["w"][1], s["x"], s["y"])
    return s["y"]


# ---------------------------------------------------------------------- work
def _matrix_bytes(bits, M, K):
    return M * K * bits // 8 + (2 if bits == 1 else 4) * M * K // GROUP[bits]


def _layer_params(case):
    """[(M, K)] of a layer's projections."""
    H, I, hq, hkv, D = SHAPES[case["shape"]]
    return [(hq * D, H), (hkv * D, H), (hkv * D, H), (H, hq * D), (I, H), (I, H), (H, I)]


def _model_work(case, tokens, start):
    """Bytes and flops of one pass of `tokens` tokens from position `start`: every weight once,
    the caches read and written, the head for the last token."""
    H, I, hq, hkv, D = SHAPES[case["shape"]]
    b = sum(_matrix_bytes(case["bits"], M, K) for M, K in _layer_params(case)) * case["layers"]
    f = 2 * tokens * sum(M * K for M, K in _layer_params(case)) * case["layers"]
    keys = sum(range(start + 1, start + tokens + 1))
    b += 2 * 2 * (start + tokens) * hkv * D * case["layers"]
    f += 4 * keys * hq * D * case["layers"]
    if "vocab" in case:
        V = case["vocab"]
        b += _matrix_bytes(case["bits"], V, H) + 4 * V + tokens * _matrix_bytes(case["bits"], 1, H)
        f += 2 * V * H
    return b, f


def work(case):
    kind = case["kind"]
    if kind == "qmv":
        M, K, e = case["M"], case["K"], 2 if case["form"] == "f16io" else 4
        b, f = _matrix_bytes(case["bits"], M, K) + e * (M + K), 2 * M * K
    elif kind == "head":
        V, K = case["V"], case["K"]
        b, f = _matrix_bytes(case["bits"], V, K) + 8 * K + 4 * V, 2 * V * K
    elif kind == "attention":
        b = 2 * 2 * case["L"] * case["hkv"] * 128 + (2 + 4) * case["hq"] * 128
        f = 4 * case["L"] * case["hq"] * 128
    elif kind == "layers":
        b, f = _model_work(case, 1, case["seq"] - 1)
    elif kind == "gemm":
        n = 2 if case["mode"] == "silu" else 1
        P, M, K = case["P"], case["M"], case["K"]
        b = n * _matrix_bytes(case["bits"], M, K) + 2 * P * K + (4 if case["mode"] == "f32" else 2) * P * M
        f = 2 * n * P * M * K
    elif kind == "prefill":
        b, f = _model_work(case, case["P"], 0)
    elif kind == "generate":
        b, f = _model_work(case, case["P"], 0)
        for i in range(case["new"]):
            db, df = _model_work(case, 1, case["P"] + i)
            b, f = b + db, f + df
    else:
        n = {"q1": 1, "q4": 1, "silu": 2}[case["form"]]
        M, K = case["M"], case["K"]
        b = case["count"] * (n * _matrix_bytes(4 if case["form"] == "q4" else 1, M, K) + 4 * (M + K))
        f = case["count"] * 2 * n * M * K
    return {"bytes": b, "flops": f}


def tolerance(case):
    """Relative errors: about four times what two correct orders of the sums show.  float32
    results carry float32 sums (measured 2e-7); f16 results may round the other way (f16: 2e-4
    off float64); 4-bit results are truncated to bf16 (single calls 3e-3, eight layers 1e-2).
    Whole models pass such roundings on from layer to layer (1-bit 7e-4 after 28 layers)."""
    kind, q4 = case["kind"], case.get("bits") == 4
    if kind in ("attention", "stacked") or (kind == "qmv" and case["form"] == "f32") or (kind == "gemm" and case["mode"] == "f32" and not q4):
        return {"rel": 1e-5}
    if kind in ("qmv", "head", "gemm"):
        return {"rel": 1e-2 if q4 else 1e-3}
    return {"rel": 3e-2 if q4 else 3e-3}


# --------------------------------------------------------------------- exact
def _dense(w):
    """float64 values of a host QWeight, on the GPU."""
    c = _gpu(w.codes.view(np.int32))
    n = 32 // w.bits
    sh = torch.arange(n, device="cuda", dtype=torch.int32) * w.bits
    v = ((c[:, :, None] >> sh) & ((1 << w.bits) - 1)).reshape(w.M, w.K // w.group_size, w.group_size)

    def param(raw):
        t = _gpu(raw.view(np.int16))
        return t.view(torch.float16 if w.scale_dtype == fm.DT_F16 else torch.bfloat16).double()[:, :, None]

    s = param(w.scales)
    out = (2 * v - 1) * s if w.bits == 1 else v * s + param(w.biases)
    return out.reshape(w.M, w.K)


def _rms(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w


def _rope(x, pos):
    """x [P, heads, D], consecutive pairs; the angles as float32 products of the position
    and the float32 frequency, as the entry points define them."""
    D = x.shape[-1]
    inv = (THETA ** (-torch.arange(0, D, 2, device="cuda", dtype=torch.float64) / D)).float()
    a = (pos.float()[:, None] * inv[None]).double()[:, None, :]
    x0, x1 = x[..., 0::2], x[..., 1::2]
    return torch.stack((x0 * a.cos() - x1 * a.sin(), x0 * a.sin() + x1 * a.cos()), -1).flatten(-2)


def _block(w, shape, res, start, kc, vc):
    """One decoder layer in float64 over tokens at start..; kc, vc [hkv, start, D] of the
    earlier positions.  Returns the residual and the caches with the new positions."""
    H, I, hq, hkv, D = SHAPES[shape]
    P, g = res.shape[0], hq // hkv
    pos = torch.arange(start, start + P, device="cuda")
    x = _rms(res, _gpu(w["attn_norm"]).double())
    q, k, v = ((x @ _dense(w[n]).T).reshape(P, -1, D) for n in "qkv")
    q = _rope(_rms(q, _gpu(w["q_norm"]).double()), pos)
    k = _rope(_rms(k, _gpu(w["k_norm"]).double()), pos)
    kc, vc = torch.cat((kc, k.transpose(0, 1)), 1), torch.cat((vc, v.transpose(0, 1)), 1)
    att = torch.empty(P, hq, D, dtype=torch.float64, device="cuda")
    late = torch.arange(start + P, device="cuda")[None, :] > pos[:, None]
    for h in range(hq):
        s = (q[:, h] @ kc[h // g].T / math.sqrt(D)).masked_fill(late, -math.inf)
        att[:, h] = s.softmax(-1) @ vc[h // g]
    res = res + att.reshape(P, -1) @ _dense(w["o"]).T
    x = _rms(res, _gpu(w["ffn_norm"]).double())
    gate = x @ _dense(w["gate"]).T
    return res + (gate * gate.sigmoid() * (x @ _dense(w["up"]).T)) @ _dense(w["down"]).T, kc, vc


def _forward(cfg, w, shape, ids):
    """float64 final-norm output of every token."""
    rows = fm.QWeight(w.embed_q1.bits, len(ids), w.embed_q1.K, w.embed_q1.group_size, w.embed_q1.codes[ids], w.embed_q1.scales[ids],
                      None if w.embed_q1.biases is None else w.embed_q1.biases[ids], w.embed_q1.scale_dtype)
    res = _dense(rows)
    empty = torch.empty(cfg.num_kv_heads, 0, cfg.head_dim, dtype=torch.float64, device="cuda")
    for lay in w.layers:
        res = _block(lay, shape, res, 0, empty, empty)[0]
    return _rms(res, _gpu(w.final_norm).double())


def exact(case, seed):
    kind = case["kind"]
    if kind in ("prefill", "generate"):
        cfg, w = _weights(case, seed)
        ids = _prompt(case, seed)
        if kind == "prefill":
            return (_forward(cfg, w, case["shape"], ids)[-1:] @ _dense(w.lm_head).T)[0]
        new = ((int(ids[-1]) + 1 + np.arange(case["new"])) % case["vocab"]).astype(np.int64)
        x = _forward(cfg, w, case["shape"], np.concatenate((ids, new.astype(np.uint32))))[case["P"] - 1:]
        logits = x @ _dense(w.lm_head).T
        top = logits[:-1].topk(2).values
        return {"tokens": new, "margins": top[:, 0] - top[:, 1], "logits": logits[-1]}
    s = prepare(case, seed)
    if kind == "qmv":
        return _dense(s["host"]) @ s["x"].double()
    if kind == "head":
        x = _rms(s["res"].double(), s["norm"].double())
        return {"logits": _dense(s["host"]) @ x, "token": None, "prob": None}
    if kind == "attention":
        n, g = case["L"], case["hq"] // case["hkv"]
        q = _rope(s["q"].double()[None], torch.tensor([n - 1], device="cuda"))[0]
        k = s["k"][:, :n].double().repeat_interleave(g, 0)
        v = (s["v"].transpose(1, 2) if case["transposed"] else s["v"])[:, :n].double().repeat_interleave(g, 0)
        p = ((k @ q[:, :, None])[:, :, 0] / math.sqrt(q.shape[1])).softmax(-1)
        return (p[:, None] @ v)[:, 0]
    if kind == "layers":
        n = case["seq"] - 1
        e = s["emb_host"]
        res = _dense(fm.QWeight(e.bits, 1, e.K, e.group_size, e.codes[[s["id"]]], e.scales[[s["id"]]],
                                None if e.biases is None else e.biases[[s["id"]]], e.scale_dtype))
        ks, vs = [], []
        for w, d in zip(s["host"], s["layers"]):
            k0, v0 = d["k"].double(), d["v"].double().transpose(1, 2)
            res, kc, vc = _block(w, case["shape"], res, n, k0[:, :n], v0[:, :n])
            ks.append(torch.cat((kc, k0[:, n + 1:]), 1))
            vs.append(torch.cat((vc, v0[:, n + 1:]), 1).transpose(1, 2))
        return {"residual": res[0], "k": ks, "v": vs}
    if kind == "gemm":
        a = s["a"].double()
        y = a @ _dense(s["host"][0]).T
        return y if case["mode"] != "silu" else y * y.sigmoid() * (a @ _dense(s["host"][1]).T)
    y = []
    for i in range(case["count"]):
        t = [_dense(w.host(i)) @ s["x"][i].double() for w in s["w"]]
        y.append(t[0] if len(t) == 1 else t[0] * t[0].sigmoid() * t[1])
    return torch.stack(y)
