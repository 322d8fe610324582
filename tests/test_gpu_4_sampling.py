"""GPU parity of device-side sampling (sampleToken on device) and of the
decode loop's stop tokens.

* The device random stream equals the oracle's restatement of Zig's
  DefaultPrng word for word after every draw.
* Tokens drawn on the device equal the oracle's for the same logits and the
  same stream wherever the oracle's draw (and top-p cut) lies farther from a
  decision boundary than float32 summation rounding (1e-5 + 2.5e-7 sqrt(V));
  nearer than that, the order of the sum decides and the device's token must
  be the inverse-CDF pick of r within that tolerance.
* Device draws follow the filtered softmax (chi-square).
* The model's generate with sampling equals the oracle's generate up to the
  first step whose decision margin is below 1e-4 (the model's logits differ
  from the oracle's by float32 rounding), and stop tokens end it unemitted.
"""
import numpy as np
import pytest
import torch

from nnzap_amd import _lib as L
from nnzap_amd import configs as cf
from nnzap_amd import ops
from nnzap_amd.model import DecoderModel
from nnzap_amd.ops import Device, NnzError
from oracle import sampling as SM
from oracle.decoder import OracleDecoder

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sdev():
    d = Device(0, own_stream=True)
    yield d
    d.close()


def _buffers(n, draws):
    ws = torch.empty(ops.sample_workspace_bytes(n), dtype=torch.uint8, device="cuda")
    rng = torch.zeros(4, dtype=torch.int64, device="cuda")
    out = torch.full((draws,), -1, dtype=torch.int32, device="cuda")
    prob = torch.zeros(draws, dtype=torch.float32, device="cuda")
    return ws, rng, out, prob


def _state(rng):
    return [int(v) for v in rng.cpu().numpy().view(np.uint64)]


def test_rng_stream_matches_oracle(sdev):
    ws, rng, out, prob = _buffers(1000, 64)
    logits = torch.randn(1000, device="cuda")
    ops.rng_seed(sdev, 12345, rng)
    p = SM.ZigPrng(12345)
    assert _state(rng) == p.s
    for i in range(64):
        ops.dispatch_sample(sdev, logits, out[i:i + 1], rng, ws, 1.0)
        p.float32()
    sdev.sync()
    assert _state(rng) == p.s


def _logits(n, seed, kind):
    g = np.random.default_rng(seed)
    x = g.normal(0.0, 2.5, n).astype(np.float32)
    if kind == "ties":            # coarse grid: many equal logits, ties at every cut
        x = (np.round(x * 2) / 2).astype(np.float32)
    if kind == "peaked":
        x[g.integers(0, n, 3)] += 12.0
    return x


CASES = [
    # (vocab, temperature, top_k, top_p, kind, draws)
    (1000, 1.0, 0, 1.0, "normal", 200),
    (1000, 0.7, 40, 1.0, "normal", 200),
    (1000, 0.8, 50, 0.9, "normal", 200),
    (1000, 1.2, 0, 0.95, "normal", 200),
    (1000, 1.0, 1, 1.0, "normal", 50),
    (1000, 1.0, 0, 1e-6, "normal", 50),     # smallest nucleus: the first candidate
    (1000, 1.0, 20, 0.7, "ties", 200),
    (1000, 1.0, 0, 0.6, "ties", 200),
    (777, 0.9, 2000, 0.5, "peaked", 100),
    (3000, 1.0, 1500, 1.0, "normal", 100),
    (151936, 0.8, 40, 0.95, "normal", 24),
    (151936, 1.0, 0, 0.9, "normal", 12),
    (151936, 0.6, 0, 1.0, "peaked", 12),
    (151936, 0.9, 0, 0.9, "peaked", 12),      # nucleus within the 64 largest
    (151936, 1.0, 100, 0.9, "normal", 12),    # lists cut below k, survivors > 64
    (151936, 1.0, 10000, 1.0, "normal", 6),   # cut lists miss part of the top-k set
    (4096, 1.0, 64, 0.8, "normal", 100),      # 64 survivors: one wave
    (4096, 1.0, 65, 1.0, "normal", 100),      # 65: the block-wide path
]


@pytest.mark.parametrize("V,T,k,p,kind,draws", CASES)
def test_sample_matches_oracle(sdev, V, T, k, p, kind, draws):
    x = _logits(V, V + draws, kind)
    ws, rng, out, prob = _buffers(V, draws)
    logits = torch.from_numpy(x).cuda()
    seed = 1000 + V + draws
    ops.rng_seed(sdev, seed, rng)
    print(f"sample V={V} T={T} k={k} p={p} {kind}", flush=True)
    for i in range(draws):
        ops.dispatch_sample(sdev, logits, out[i:i + 1], rng, ws, T, k, p, out_prob=prob[i:i + 1])
    sdev.sync()
    got = out.cpu().numpy()
    gp = prob.cpu().numpy()
    prng = SM.ZigPrng(seed)
    tol = SM.summation_tolerance(V)
    exact = 0
    for i in range(draws):
        d = SM.sample_token(x, T, k, p, prng)
        if d.margin >= tol:
            exact += 1
            assert got[i] == d.token, (i, got[i], d.token, d.margin)
            assert abs(gp[i] - d.prob) <= 1e-4 * max(d.prob, 1e-3) + 1e-6, (i, gp[i], d.prob)
        else:   # near a boundary: the pick must still be the inverse CDF of r
            assert d.within(int(got[i]), tol + 2 * d.q_cut), (i, got[i], d.token, d.margin)
    if V <= 3000:
        assert exact >= draws * 0.8
    assert _state(rng) == prng.s


FEW = [
    # (vocab, top_k, top_p, kind): the piece maxima take over at 2 k pieces
    (10240, 20, 0.95, "normal"),       # 40 pieces of 256: the smallest for k = 20
    (10239, 20, 0.95, "normal"),       # ragged last piece
    (9984, 20, 0.95, "normal"),        # 39 pieces: the lists
    (32768, 64, 1.0, "normal"),        # 64 kept, the most one wave finishes
    (151669, 1, 1.0, "normal"),
    (151669, 20, 0.95, "clustered"),   # 200 of the largest in one piece
    (151669, 20, 0.95, "ordered"),     # whole pieces over the threshold
    (151669, 20, 0.9, "ties"),
    (151669, 20, 0.95, "equal"),
    (151669, 20, 0.95, "masked"),      # ten finite logits, the rest -inf
    (262144, 40, 0.95, "normal"),      # 1024 pieces of 256
    (262145, 40, 0.95, "clustered"),   # pieces of 512
    (1048576, 40, 0.95, "ordered"),    # 1024 pieces of 1024, the longest
    (1048577, 40, 0.95, "normal"),     # the lists
]


@pytest.mark.parametrize("V,k,p,kind", FEW)
def test_sample_few_kept(sdev, V, k, p, kind):
    """Top-k draws from piece maxima: every route of the finishing block (one
    wave at once, after an exact k-th largest, over the pieces), piece lengths
    and the smallest count that takes it, against the oracle."""
    x = _logits(V, V, kind)
    if kind == "clustered":
        x[5000:5200] += 14.0
    elif kind == "ordered":
        x = -np.sort(-x)
    elif kind == "equal":
        x[:] = 1.5
    elif kind == "masked":
        x[np.random.default_rng(5).permutation(V)[10:]] = -np.inf
    draws = 8
    ws, rng, out, prob = _buffers(V, draws)
    logits = torch.from_numpy(x).cuda()
    ops.rng_seed(sdev, V + k, rng)
    print(f"sample V={V} k={k} p={p} {kind}", flush=True)
    for i in range(draws):
        ops.dispatch_sample(sdev, logits, out[i:i + 1], rng, ws, 0.6, k, p, out_prob=prob[i:i + 1])
    sdev.sync()
    got, gp = out.cpu().numpy(), prob.cpu().numpy()
    prng = SM.ZigPrng(V + k)
    tol = SM.summation_tolerance(V)
    if kind == "equal":   # the oracle's V additions of one value to a sum below 1 may all
        tol = V * 2.0 ** -25   # round the same way, by up to 2^-25 each
    for i in range(draws):
        d = SM.sample_token(x, 0.6, k, p, prng)
        if d.margin >= tol:
            assert got[i] == d.token, (i, got[i], d.token, d.margin)
            assert abs(gp[i] - d.prob) <= 1e-4 * max(d.prob, 1e-3) + 1e-6, (i, gp[i], d.prob)
        else:
            assert d.within(int(got[i]), tol + 2 * d.q_cut), (i, got[i], d.token, d.margin)
    assert _state(rng) == prng.s


CROWDED = [
    # (vocab, top_k, top_p, kind): more logits over the maxima's threshold than LDS holds, or more
    # ties at the k-th largest than a wave finishes
    (33000, 64, 0.9, "hump"),         # the threshold from around the largest logit
    (300000, 50, 1.0, "hump"),        # pieces of 512: one of two windows
    (33005, 20, 0.95, "tail"),        # the largest in the last piece, which is shorter than k
    (33000, 64, 0.95, "coarse"),      # 65..1024 survivors, finished in LDS in index order
    (151669, 50, 0.95, "coarse"),
    (33000, 40, 0.95, "teeth"),       # no window's threshold narrows it to 1024: exact k-th largest
    (151669, 50, 0.95, "plateau"),    # more than 1024 ties at the k-th largest, below a few larger
]


def _crowded(V, kind):
    x = _logits(V, V, "normal")
    i = np.arange(V)
    if kind == "hump":
        x = (8.0 - np.abs(i - V // 3) / 1000.0).astype(np.float32)
    elif kind == "tail":
        x[-3:] += 30.0
        x[1000:4000] += 15.0
    elif kind == "coarse":
        x = np.round(x / 2.5).astype(np.float32)
    elif kind == "teeth":
        x = (8.0 - (i % 256) / 64.0 - i / 1e5).astype(np.float32)
    elif kind == "plateau":
        x[2000:6000] = 14.0
        x[7000:7005] = 14.5
    return x


@pytest.mark.parametrize("V,k,p,kind", CROWDED)
def test_sample_few_kept_crowded(sdev, V, k, p, kind):
    """Top-k draws from piece maxima where the pieces over the threshold are full
    of logits that reach it, against the oracle."""
    x = _crowded(V, kind)
    draws = 8
    ws, rng, out, prob = _buffers(V, draws)
    logits = torch.from_numpy(x).cuda()
    ops.rng_seed(sdev, V + k, rng)
    print(f"sample V={V} k={k} p={p} {kind}", flush=True)
    for i in range(draws):
        ops.dispatch_sample(sdev, logits, out[i:i + 1], rng, ws, 0.6, k, p, out_prob=prob[i:i + 1])
    sdev.sync()
    got, gp = out.cpu().numpy(), prob.cpu().numpy()
    prng = SM.ZigPrng(V + k)
    tol = SM.summation_tolerance(V)
    if kind == "plateau":   # 4000 equal terms added to a sum below 1, each rounding the same way by up to 2^-25
        tol = max(tol, 4000 * 2.0 ** -25)
    for i in range(draws):
        d = SM.sample_token(x, 0.6, k, p, prng)
        if d.margin >= tol:
            assert got[i] == d.token, (i, got[i], d.token, d.margin)
            assert abs(gp[i] - d.prob) <= 1e-4 * max(d.prob, 1e-3) + 1e-6, (i, gp[i], d.prob)
        else:
            assert d.within(int(got[i]), tol + 2 * d.q_cut), (i, got[i], d.token, d.margin)
    assert _state(rng) == prng.s


@pytest.mark.parametrize("kind", ["hump", "coarse"])
def test_sample_few_kept_crowded_time(sdev, kind):
    """Neighbouring or tied large logits cost a draw no multiple of what scattered
    ones do (top-64 of 33000: 20 us scattered, 28 to 34 crowded; 89 to 97 where
    the finishing block went through every logit of the pieces)."""
    V = 33000
    ws, rng, out, _ = _buffers(V, 1)
    ops.rng_seed(sdev, 1, rng)

    def time_us(x):
        logits = torch.from_numpy(x).cuda()
        torch.cuda.synchronize()
        best = []
        for _ in range(5):
            sdev.mark(0)
            for _ in range(40):
                ops.dispatch_sample(sdev, logits, out, rng, ws, 0.6, 64, 1.0)
            sdev.mark(1)
            sdev.sync()
            best.append(sdev.elapsed_ms(0, 1) * 1e3 / 40)
        return min(best)

    assert time_us(_crowded(V, kind)) <= 2.5 * time_us(_logits(V, V, "normal"))


def test_sample_distribution(sdev):
    V, T, k, p, n = 40, 0.9, 12, 0.85, 6000
    x = _logits(V, 3, "normal")
    want = SM.filtered_distribution(x, T, k, p)
    ws, rng, out, prob = _buffers(V, n)
    logits = torch.from_numpy(x).cuda()
    ops.rng_seed(sdev, 99, rng)
    for i in range(n):
        ops.dispatch_sample(sdev, logits, out[i:i + 1], rng, ws, T, k, p)
    sdev.sync()
    counts = np.bincount(out.cpu().numpy(), minlength=V).astype(np.float64)
    assert np.all(counts[want == 0] == 0)
    m = want > 0
    chi2 = np.sum((counts[m] - n * want[m]) ** 2 / (n * want[m]))
    dof = m.sum() - 1
    assert chi2 < dof + 6 * np.sqrt(2 * dof) + 10, (chi2, dof)


def test_temperature_zero_is_argmax(sdev):
    x = _logits(5000, 8, "normal")
    ws, rng, out, prob = _buffers(5000, 1)
    ops.dispatch_sample(sdev, torch.from_numpy(x).cuda(), out, rng, ws, 0.0)
    sdev.sync()
    assert int(out.cpu()[0]) == int(np.argmax(x))


# -- the decode loop ---------------------------------------------------------------

@pytest.fixture(scope="module")
def tiny():
    cfg = cf.TINY
    return cfg, cf.decoder_weights(cfg, norm_mode="unit")


@pytest.mark.parametrize("params", [(1.2, 5, 1.0, 5), (0.8, 40, 0.9, 7)])
def test_generate_sampled_matches_oracle(sdev, tiny, params):
    cfg, w = tiny
    prompt = cf.prompt_ids(cfg, 32)
    ref_toks, ref_probs, margins = OracleDecoder(w).generate_sampled(prompt, 24, *params)
    m = DecoderModel(sdev, cfg)
    try:
        m.load(w)
        m.set_sampling(*params)
        toks, probs, _ = m.generate(prompt, 24, use_graph=True)
        toks2, _, _ = m.generate(prompt, 24, use_graph=False)
    finally:
        m.close()
    assert np.array_equal(toks, toks2)          # graph replay == eager steps
    # steps before the first near-boundary decision must agree exactly
    bad = np.nonzero(margins < 1e-4)[0]
    n_cmp = int(bad[0]) if len(bad) else len(ref_toks)
    assert n_cmp >= 8
    assert np.array_equal(toks[:n_cmp], ref_toks[:n_cmp]), (toks, ref_toks, margins)
    np.testing.assert_allclose(probs[:n_cmp], ref_probs[:n_cmp], rtol=2e-3)


@pytest.mark.parametrize("use_graph", [True, False])
def test_generate_stops_at_eos(sdev, tiny, use_graph):
    cfg, w = tiny
    prompt = cf.prompt_ids(cfg, 32)
    ref, _ = OracleDecoder(w).generate(prompt, 16)
    # a stop token first produced at step j > 0
    j = next(i for i in range(1, 16) if ref[i] not in ref[:i])
    eos = int(ref[j])
    ref_eos, _ = OracleDecoder(w).generate(prompt, 16, eos=(eos, 7777))
    assert len(ref_eos) == j
    m = DecoderModel(sdev, cfg)
    try:
        m.load(w)
        m.set_eos([7777, eos])
        toks, margins, _ = m.generate(prompt, 16, use_graph=use_graph)
        assert np.array_equal(toks, ref[:j]) and len(margins) == j
        assert m.decode_status() == (j, True)
        m.set_eos([int(ref[0])])                  # stop token picked first: nothing emitted
        toks, _, _ = m.generate(prompt, 16, use_graph=use_graph)
        assert len(toks) == 0
        m.set_eos([])
        toks, _, _ = m.generate(prompt, 16, use_graph=use_graph)
        assert np.array_equal(toks, ref)
    finally:
        m.close()


@pytest.mark.parametrize("top_p", [float("nan"), 0.0, -0.5])
def test_bad_top_p_is_rejected(sdev, tiny, top_p):
    """applyTopP asserts 0 < p <= 1 (transformer.zig:3781-3790): NaN and
    p <= 0 are refused by both the model and the sampling dispatch (p >= 1
    stays "off", :3878)."""
    cfg, w = tiny
    m = DecoderModel(sdev, cfg)
    try:
        with pytest.raises(NnzError) as e:
            m.set_sampling(0.8, 0, top_p, 1)
        assert e.value.code == L.EINVAL
        m.set_sampling(0.8, 0, 1.5, 1)      # >= 1: top-p off, accepted
    finally:
        m.close()
    x = _logits(1000, 3, "normal")
    ws, rng, out, prob = _buffers(1000, 1)
    with pytest.raises(NnzError) as e:
        ops.dispatch_sample(sdev, torch.from_numpy(x).cuda(), out, rng, ws, 1.0, 0, top_p)
    assert e.value.code == L.EINVAL
