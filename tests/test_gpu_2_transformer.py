"""GPU parity of attention, norms, RoPE, KV append, embeddings, argmax and the
prefill dequant-GEMM against the CPU oracle."""
import numpy as np
import pytest
import torch

from nnzap_amd import _lib as L
from nnzap_amd import configs as cf
from nnzap_amd import ops
from nnzap_amd import synth as S
from oracle import oracle as O

from gpu_util import (assert_bf16_faithful, assert_close, assert_close_normwise, from_bits16, host,
                      tdev)

pytestmark = pytest.mark.gpu


def _scratch(dims):
    n = ops.gqa_scratch_bytes(dims)
    return torch.empty((n + 3) // 4, dtype=torch.float32, device="cuda")


# --------------------------------------------------------------- attention --
@pytest.mark.parametrize("L_", [512, 4096, 32768])
def test_config4_gqa_decode(dev, L_):
    """q bf16 [16,128] roped at position L, KV bf16 [8,L,128],
    scale 1/sqrt(128), fp32 accumulate; V given as [8, L, 128]."""
    print(f"config4 L={L_}", flush=True)
    q, k, v = cf.config4(L_)
    qd, kd, vd = from_bits16(q, "bf16"), from_bits16(k, "bf16"), from_bits16(v, "bf16")
    out = torch.empty(16, 128, dtype=torch.float32, device="cuda")
    dims = L.GQADims(16, 8, 128, L_, L_, 2)
    ops.dispatch_gqa_attention(dev, qd, kd, vd, out, _scratch(dims), dims, v_transposed=False,
                               rope_position=L_, rope_theta=1e6)
    dev.sync()
    qf = O.rope(S.bf16_bits_to_f32(q).astype(np.float64), L_, 1e6)
    ref = O.attention_decode(qf, S.bf16_bits_to_f32(k), S.bf16_bits_to_f32(v), L_, False)
    assert_close(host(out), ref, what=f"config4 L={L_}")


@pytest.mark.parametrize("L_,max_ctx,hq,hkv,d", [(1, 8, 4, 2, 64), (77, 128, 16, 8, 128),
                                                 (700, 1024, 8, 8, 128), (3000, 4096, 16, 2, 64),
                                                 (2000, 2048, 16, 4, 128), (104, 104, 16, 8, 128),
                                                 (99, 104, 8, 8, 128), (20000, 20000, 2, 1, 128),
                                                 (9000, 9216, 4, 2, 128)])
def test_gqa_transposed_v_f16(dev, L_, max_ctx, hq, hkv, d):
    """Reference layout: f16 caches, V transposed [h][d][max_ctx], f16 q/out."""
    rng_q = (0.3 * S.normal(400, hq * d)).astype(np.float16).reshape(hq, d)
    kf = np.zeros((hkv, max_ctx, d), np.float16)
    vf = np.zeros((hkv, d, max_ctx), np.float16)
    kf[:, :L_] = S.normal(401, hkv * L_ * d).astype(np.float16).reshape(hkv, L_, d)
    vf[:, :, :L_] = S.normal(402, hkv * L_ * d).astype(np.float16).reshape(hkv, d, L_)
    out = torch.empty(hq, d, dtype=torch.float16, device="cuda")
    dims = L.GQADims(hq, hkv, d, L_, max_ctx, hq // hkv)
    ops.dispatch_gqa_attention(dev, tdev(rng_q), tdev(kf), tdev(vf), out, _scratch(dims), dims)
    dev.sync()
    ref = O.attention_decode(rng_q.astype(np.float64), kf.astype(np.float64), vf.astype(np.float64),
                             L_, True)
    assert_close(host(out), O.f16(ref), what=f"gqa L={L_}")


@pytest.mark.parametrize("vt", [False, True])
def test_gqa_long_ragged_bf16(dev, vt):
    """16397 tokens (16384 + 13): the launcher walks chunks of two 64-token
    sub-chunks with an online softmax, the last chunk holding one ragged
    sub-chunk; bf16 caches in both V layouts, f32 q roped at 16397, f32 out."""
    L_, max_ctx, hq, hkv, d = 16397, 16400, 16, 8, 128
    print(f"gqa long ragged vt={vt}", flush=True)
    q = S.normal(410, hq * d).astype(np.float32).reshape(hq, d)
    kb = S.f32_to_bf16_bits(S.normal(411, hkv * max_ctx * d).astype(np.float32)).reshape(hkv, max_ctx, d)
    vb = S.f32_to_bf16_bits(S.normal(412, hkv * max_ctx * d).astype(np.float32))
    vb = vb.reshape(hkv, d, max_ctx) if vt else vb.reshape(hkv, max_ctx, d)
    out = torch.empty(hq, d, dtype=torch.float32, device="cuda")
    dims = L.GQADims(hq, hkv, d, L_, max_ctx, hq // hkv)
    ops.dispatch_gqa_attention(dev, tdev(q), from_bits16(kb, "bf16"), from_bits16(vb, "bf16"), out,
                               _scratch(dims), dims, v_transposed=vt, rope_position=L_,
                               rope_theta=1e6)
    dev.sync()
    qf = O.rope(q.astype(np.float64), L_, 1e6)
    ref = O.attention_decode(qf, S.bf16_bits_to_f32(kb), S.bf16_bits_to_f32(vb), L_, vt)
    assert_close(host(out), ref, what=f"gqa long vt={vt}")


@pytest.mark.parametrize("pos", [0, 5, 600, 1500])
def test_gqa_fused_norm_rope_kv(dev, pos):
    """transformer.metal:1467-1695 semantics: q/k per-head RMSNorm + RoPE, K/V
    append at `pos`, attention over pos+1 tokens; cache contents checked too."""
    hq, hkv, d, max_ctx, theta = 16, 8, 128, 2048, 1e6
    q = S.normal(410, hq * d).astype(np.float16).reshape(hq, d)
    kr = S.normal(411, hkv * d).astype(np.float16).reshape(hkv, d)
    vr = S.normal(412, hkv * d).astype(np.float16).reshape(hkv, d)
    qn = (1 + 0.1 * S.normal(413, d)).astype(np.float32)
    kn = (1 + 0.1 * S.normal(414, d)).astype(np.float32)
    kc = np.zeros((hkv, max_ctx, d), np.float16)
    vc = np.zeros((hkv, d, max_ctx), np.float16)
    if pos:
        kc[:, :pos] = (0.5 * S.normal(415, hkv * pos * d)).astype(np.float16).reshape(hkv, pos, d)
        vc[:, :, :pos] = S.normal(416, hkv * pos * d).astype(np.float16).reshape(hkv, d, pos)
    kcd, vcd = tdev(kc), tdev(vc)
    out = torch.empty(hq, d, dtype=torch.float16, device="cuda")
    fd = L.GQAFusedDims(hq, hkv, d, pos + 1, max_ctx, hq // hkv, pos, 1e-6, theta)
    dims = L.GQADims(hq, hkv, d, pos + 1, max_ctx, hq // hkv)
    ops.dispatch_gqa_attention_fused(dev, tdev(q), kcd, vcd, out, tdev(kr), tdev(vr), tdev(qn),
                                     tdev(kn), _scratch(dims), fd)
    dev.sync()
    kc_ref, vc_ref = kc.astype(np.float64), vc.astype(np.float64)
    ref = O.gqa_fused_step(q.astype(np.float64), kr.astype(np.float64), vr.astype(np.float64),
                           kc_ref, vc_ref, qn, kn, pos, theta, v_transposed=True)
    kg = host(kcd)
    assert_close(kg[:, pos], kc_ref[:, pos], what="k cache row")
    assert np.array_equal(host(vcd)[:, :, pos], vc_ref[:, :, pos])
    assert np.array_equal(kg[:, :pos], kc_ref[:, :pos])  # earlier rows untouched
    assert_close(host(out), O.f16(ref), what=f"fused pos={pos}")


@pytest.mark.parametrize("hq,hkv,d", [(16, 8, 128), (4, 2, 64), (8, 8, 128)])
def test_gqa_fused_1pass_successive_positions(dev, hq, hkv, d):
    """Fused attention (one kernel, plus a merge kernel past one chunk) at
    consecutive positions sharing one scratch, with the sequence length read
    from device memory as in graph replay."""
    max_ctx, theta = 2048, 1e6
    qn = (1 + 0.1 * S.normal(417, d)).astype(np.float32)
    kn = (1 + 0.1 * S.normal(418, d)).astype(np.float32)
    kc = np.zeros((hkv, max_ctx, d), np.float16)
    vc = np.zeros((hkv, d, max_ctx), np.float16)
    start = 1400
    kc[:, :start] = (0.5 * S.normal(419, hkv * start * d)).astype(np.float16).reshape(hkv, start, d)
    vc[:, :, :start] = S.normal(420, hkv * start * d).astype(np.float16).reshape(hkv, d, start)
    kcd, vcd = tdev(kc), tdev(vc)
    kc_ref, vc_ref = kc.astype(np.float64), vc.astype(np.float64)
    max_seq = start + 8
    dims = L.GQAFusedDims(hq, hkv, d, max_seq, max_ctx, hq // hkv, 0, 1e-6, theta)
    gd = L.GQADims(hq, hkv, d, max_seq, max_ctx, hq // hkv)
    scr = torch.zeros(ops.gqa_scratch_bytes(gd) // 4 + 64, dtype=torch.float32, device="cuda")
    dseq = torch.zeros(1, dtype=torch.int32, device="cuda")
    out = torch.empty(hq, d, dtype=torch.float16, device="cuda")
    for i, pos in enumerate(range(start, start + 8)):
        q = S.normal(430 + i, hq * d).astype(np.float16).reshape(hq, d)
        kr = S.normal(440 + i, hkv * d).astype(np.float16).reshape(hkv, d)
        vr = S.normal(450 + i, hkv * d).astype(np.float16).reshape(hkv, d)
        dseq.fill_(pos + 1)
        ops.dispatch_gqa_attention_fused_1pass(dev, tdev(q), kcd, vcd, out, tdev(kr), tdev(vr),
                                               tdev(qn), tdev(kn), scr, dims, d_seq_len=dseq)
        dev.sync()
        ref = O.gqa_fused_step(q.astype(np.float64), kr.astype(np.float64), vr.astype(np.float64),
                               kc_ref, vc_ref, qn, kn, pos, theta, v_transposed=True)
        assert_close(host(out), O.f16(ref), what=f"1pass pos={pos}")
    assert_close(host(kcd)[:, start:start + 8], kc_ref[:, start:start + 8], what="k rows")
    assert np.array_equal(host(vcd)[:, :, start:start + 8], vc_ref[:, :, start:start + 8])


@pytest.mark.parametrize("hq,hkv,seq,ctx", [(32, 8, 1, 64), (32, 8, 512, 512), (32, 8, 513, 520),
                                            (32, 8, 576, 576), (32, 8, 1024, 1024), (32, 8, 1025, 1032),
                                            (16, 8, 1153, 1280), (8, 8, 2113, 2120), (16, 2, 2200, 2304),
                                            (32, 2, 610, 616), (24, 8, 715, 720), (40, 8, 900, 904)])
def test_gqa_fused_1pass_kernels(dev, hq, hkv, seq, ctx):
    """The fused attention where its kernels and chunk lengths change (wave
    kernel up to 256 (chunk, head) blocks, the MFMA one with 64- and 128-token
    chunks), at the edges of chunks and of a wave's tokens, with groups of 1,
    2, 3, 4, 5, 8 and 16 heads (two blocks of eight).  Everything past the
    live length holds NaN and must not be read into a result."""
    d, theta, pos = 128, 1e6, seq - 1
    rng = np.random.default_rng([hq, hkv, seq])
    qn, kn = ((1 + 0.1 * rng.standard_normal(d)).astype(np.float32) for _ in range(2))
    kc = np.full((hkv, ctx, d), np.nan, np.float16)
    vc = np.full((hkv, d, ctx), np.nan, np.float16)
    kc[:, :pos] = rng.standard_normal((hkv, pos, d))
    vc[:, :, :pos] = rng.standard_normal((hkv, d, pos))
    q = rng.standard_normal((hq, d)).astype(np.float16)
    kr = rng.standard_normal((hkv, d)).astype(np.float16)
    vr = rng.standard_normal((hkv, d)).astype(np.float16)
    kcd, vcd, qd, krd, vrd = tdev(kc), tdev(vc), tdev(q), tdev(kr), tdev(vr)
    dims = L.GQAFusedDims(hq, hkv, d, seq, ctx, hq // hkv, pos, 1e-6, theta)
    gd = L.GQADims(hq, hkv, d, seq, ctx, hq // hkv)
    scr = torch.zeros(ops.gqa_scratch_bytes(gd) // 4 + 64, dtype=torch.float32, device="cuda")
    out = torch.empty(hq, d, dtype=torch.float16, device="cuda")
    ops.dispatch_gqa_attention_fused_1pass(dev, qd, kcd, vcd, out, krd, vrd, tdev(qn), tdev(kn), scr, dims)
    dev.sync()
    kr_, vr_ = kc[:, :seq].astype(np.float64), vc[:, :, :seq].astype(np.float64)
    ref = O.gqa_fused_step(q.astype(np.float64), kr.astype(np.float64), vr.astype(np.float64),
                           kr_, vr_, qn, kn, pos, theta, v_transposed=True)
    assert_close(host(out), O.f16(ref), what=f"1pass {hq}/{hkv} seq={seq}")
    assert_close(host(kcd)[:, pos], kr_[:, pos], what="k row")
    assert np.array_equal(host(vcd)[:, :, pos], vr_[:, :, pos])
    assert np.array_equal(host(kcd)[:, :pos], kr_[:, :pos])
    assert np.isnan(host(kcd)[:, seq:]).all() and np.isnan(host(vcd)[:, :, seq:]).all()


def test_gqa_fused_1pass_infinite_cache(dev):
    """An infinity in the caches of a long context does what it does to a
    float32 product: a key whose score is -inf has no weight (the output is
    finite and the other tokens'), a value of +inf makes its dim +inf."""
    hq, hkv, d, seq, ctx, theta = 16, 8, 128, 1100, 1104, 1e6
    pos = seq - 1
    rng = np.random.default_rng(2202)
    qn, kn = ((1 + 0.1 * rng.standard_normal(d)).astype(np.float32) for _ in range(2))
    kc = np.zeros((hkv, ctx, d), np.float16)
    vc = np.zeros((hkv, d, ctx), np.float16)
    kc[:, :pos] = rng.standard_normal((hkv, pos, d))
    vc[:, :, :pos] = rng.standard_normal((hkv, d, pos))
    q = rng.standard_normal((hkv, 1, d)).repeat(hq // hkv, 1).reshape(hq, d).astype(np.float16)
    kr, vr = (rng.standard_normal((hkv, d)).astype(np.float16) for _ in range(2))
    rot = O.head_norm_rope(q.astype(np.float64), qn, pos, theta)
    kc[0, 500, 3] = -np.inf * np.sign(rot[0, 3])
    kc[2, 1098, 70] = -np.inf * np.sign(rot[4, 70])
    vc[1, 7, 20] = np.inf
    dims = L.GQAFusedDims(hq, hkv, d, seq, ctx, hq // hkv, pos, 1e-6, theta)
    scr = torch.zeros(ops.gqa_scratch_bytes(L.GQADims(hq, hkv, d, seq, ctx, hq // hkv)), dtype=torch.uint8, device="cuda")
    out = torch.empty(hq, d, dtype=torch.float16, device="cuda")
    ops.dispatch_gqa_attention_fused_1pass(dev, tdev(q), tdev(kc), tdev(vc), out, tdev(kr), tdev(vr), tdev(qn),
                                           tdev(kn), scr, dims)
    dev.sync()
    got = host(out)
    ref = O.gqa_fused_step(q.astype(np.float64), kr.astype(np.float64), vr.astype(np.float64),
                           kc[:, :seq].astype(np.float64), vc[:, :, :seq].astype(np.float64), qn, kn, pos, theta)
    assert (got[2:4, 7] == np.inf).all() and (ref[2:4, 7] == np.inf).all()
    got[2:4, 7] = ref[2:4, 7] = 0.0
    assert_close(got, O.f16(ref), what="infinite cache")


@pytest.mark.parametrize("form,qscale,kscale", [("plain", 1.0, 1.0), ("small norms", 2.0 ** -10, 2.0 ** 10),
                                                ("large norms", 2.0 ** 20, 2.0 ** -17), ("sink", 1.0, 1.0)])
def test_attention_partials_precision(dev, form, qscale, kscale):
    """The matrix-core decode attention holds float32 queries and weights: its
    float32 partials (288 blocks: 16 heads x 18 chunks), merged here in float64,
    against the oracle.  Norm weights far from 1 against keys that bring the
    scores back to size (16-bit parts of q would lose their last bits, or
    overflow), and a sink: one token without a value takes the weight, the rest
    (2^-20 of it each) is what is left to see.

    Tolerance, relative in the 2-norm: 1e-5.  The scores (up to 14) are float32
    sums, a few 14 2^-24 = 8e-7 off, which is their weights' relative error;
    the weights are kept to 2^-40 of the largest, 2^-20 of the sink's others."""
    hq, hkv, d, seq, theta, ctx = 16, 8, 128, 1100, 1e6, 1104
    pos = seq - 1
    rng = np.random.default_rng(2201)
    qn = (qscale * (1 + 0.1 * rng.standard_normal(d))).astype(np.float32)
    kn = (kscale * (1 + 0.1 * rng.standard_normal(d))).astype(np.float32)
    kc = np.zeros((hkv, ctx, d), np.float16)
    vc = np.zeros((hkv, d, ctx), np.float16)
    kc[:, :pos] = kscale * rng.standard_normal((hkv, pos, d))
    vc[:, :, :pos] = rng.standard_normal((hkv, d, pos))
    q = rng.standard_normal((hkv, 1, d)).repeat(hq // hkv, 1).reshape(hq, d).astype(np.float16)
    kr, vr = (rng.standard_normal((hkv, d)).astype(np.float16) for _ in range(2))
    if form == "sink":
        kc[:, 0] = 1.25 * O.head_norm_rope(q.astype(np.float64), qn, pos, theta)[::hq // hkv]
        vc[:, :, 0] = 0.0
    n = ops.gqa_partial_chunks(seq)
    part_o = torch.empty(n, hq * d, dtype=torch.float32, device="cuda")
    part_ml = torch.empty(n, hq, 2, dtype=torch.float32, device="cuda")
    dims = L.GQAFusedDims(hq, hkv, d, seq, ctx, hq // hkv, pos, 1e-6, theta)
    ops.dispatch_gqa_attention_partials(dev, tdev(q), tdev(kc), tdev(vc), tdev(kr), tdev(vr), tdev(qn), tdev(kn),
                                        part_o, part_ml, dims, rope_inv_freq=tdev(O.rope_inv_freq(d, theta)))
    dev.sync()
    k = np.arange(hq * d)
    at = ((k >> 2) & 7) * (hq * d // 8) + (k >> 5) * 4 + (k & 3)   # unit-major columns
    o, ml = host(part_o)[:, at].reshape(n, hq, d), host(part_ml)
    w = np.exp(ml[..., 0] - ml[..., 0].max(0))
    got = (w[..., None] * o).sum(0) / (w * ml[..., 1]).sum(0)[..., None]
    ref = O.gqa_fused_step(q.astype(np.float64), kr.astype(np.float64), vr.astype(np.float64),
                           kc[:, :seq].astype(np.float64), vc[:, :, :seq].astype(np.float64), qn, kn, pos, theta)
    e = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert e <= 1e-5, f"{form}: relative error {e:.2e}"


@pytest.mark.parametrize("pos", [30, 700, 1023])
@pytest.mark.parametrize("freq_table", [False, True])
@pytest.mark.parametrize("hq,hkv", [(16, 8), (24, 12)])
def test_attention_partials_merged_o_projection(dev, pos, freq_table, hq, hkv):
    """The decode step's two halves: attention to per-chunk partials, then the
    1-bit O projection (residual +=) merging them in its prologue.  Checked
    against the one-call fused attention + plain O projection on the GPU
    (same f16 attention output, different QMV order: 1e-4), and against the
    oracle (normwise, after the f16 rounding of the attention output).
    24 heads: K = 3072, rows of one and a half wave-widths (the second unit
    block is half past the row end)."""
    d, max_ctx, theta = 128, 1024, 1e6
    H = 2048
    qn = (1 + 0.1 * S.normal(461, d)).astype(np.float32)
    kn = (1 + 0.1 * S.normal(462, d)).astype(np.float32)
    kc = np.zeros((hkv, max_ctx, d), np.float16)
    vc = np.zeros((hkv, d, max_ctx), np.float16)
    kc[:, :pos] = (0.5 * S.normal(463, hkv * pos * d)).astype(np.float16).reshape(hkv, pos, d)
    vc[:, :, :pos] = S.normal(464, hkv * pos * d).astype(np.float16).reshape(hkv, d, pos)
    q = S.normal(465, hq * d).astype(np.float16).reshape(hq, d)
    kr = S.normal(466, hkv * d).astype(np.float16).reshape(hkv, d)
    vr = S.normal(467, hkv * d).astype(np.float16).reshape(hkv, d)
    wo = cf.q1_matrix(H, hq * d, 128, 468, 469)
    res0 = S.normal(470, H).astype(np.float32)
    dwo = ops.DeviceQWeight(dev, wo)
    seq = pos + 1
    dims = L.GQAFusedDims(hq, hkv, d, seq, max_ctx, hq // hkv, pos, 1e-6, theta)
    dseq = torch.full((1,), seq, dtype=torch.int32, device="cuda")
    n = ops.gqa_partial_chunks(seq)
    assert 1 <= n <= 16
    part_o = torch.empty(hq * n * d, dtype=torch.float32, device="cuda")
    part_ml = torch.empty(hq * n * 2, dtype=torch.float32, device="cuda")
    freqs = tdev(O.rope_inv_freq(d, theta)) if freq_table else None
    # path 1: partials + merged O projection
    kc1, vc1, res1 = tdev(kc), tdev(vc), tdev(res0)
    ops.dispatch_gqa_attention_partials(dev, tdev(q), kc1, vc1, tdev(kr), tdev(vr), tdev(qn),
                                        tdev(kn), part_o, part_ml, dims, d_seq_len=dseq,
                                        rope_inv_freq=freqs)
    ops.dispatch_qmv_merge_f16io_resadd(dev, dwo, part_o, part_ml, seq, d, res1, d_seq_len=dseq)
    # path 2: fused attention output + plain O projection
    kc2, vc2, res2 = tdev(kc), tdev(vc), tdev(res0)
    gd = L.GQADims(hq, hkv, d, seq, max_ctx, hq // hkv)
    scr = torch.zeros(ops.gqa_scratch_bytes(gd) // 4 + 64, dtype=torch.float32, device="cuda")
    att = torch.empty(hq * d, dtype=torch.float16, device="cuda")
    ops.dispatch_gqa_attention_fused_1pass(dev, tdev(q), kc2, vc2, att, tdev(kr), tdev(vr),
                                           tdev(qn), tdev(kn), scr, dims, d_seq_len=dseq)
    ops.dispatch_qmv_f16io_resadd(dev, dwo, att, res2)
    dev.sync()
    assert np.array_equal(host(kc1), host(kc2)) and np.array_equal(host(vc1), host(vc2))
    # The two O projections sum the same f32 products in different orders,
    # and the merge divides by the softmax sum as a reciprocal product, so an
    # f16 input where num * (1 / den) and num / den straddle a rounding edge
    # moves by one ulp.  Per row |res1 - res2| stays within 64 float32 ulps of
    # the sum of |terms| plus one ulp of the residual: two summation orders
    # emulated in float32 reach 0.04 of that, one flipped input ~0.06.
    r1, r2 = host(res1), host(res2)
    terms = np.abs(O.dequant(wo)) @ np.abs(host(att))
    bound = 64 * 2.0 ** -24 * terms + 2.0 ** -23 * np.abs(r2)
    worst = float(np.max(np.abs(r1 - r2) / bound))
    assert worst <= 1.0, f"merged vs unmerged pos={pos}: {worst:.2f} x the rounding bound"
    ref_att = O.f16(O.gqa_fused_step(q.astype(np.float64), kr.astype(np.float64),
                                     vr.astype(np.float64), kc.astype(np.float64),
                                     vc.astype(np.float64), qn, kn, pos, theta, v_transposed=True))
    ref = res0.astype(np.float64) + O.qmv(wo, ref_att.reshape(-1))
    assert_close_normwise(host(res1), ref, rtol=1e-3, what=f"oracle pos={pos}")


# ------------------------------------------------------------------ norms ---
@pytest.mark.parametrize("variant", ["f32", "f16", "bf16_f16"])
@pytest.mark.parametrize("H,T", [(2048, 3), (2560, 5), (4096, 9), (200, 2), (512, 513)])
def test_rms_norm_variants(dev, variant, H, T):
    """Wave-per-row path (hidden a multiple of 256 up to 4096, any row count)
    and the block-per-row path (hidden 200)."""
    x = S.normal(420, H * T).astype(np.float32)
    w = (1 + 0.1 * S.normal(421, H)).astype(np.float32)
    odt = torch.float32 if variant == "f32" else torch.float16
    out = torch.empty(T * H, dtype=odt, device="cuda")
    ops.dispatch_rms_norm(dev, tdev(x), tdev(w), out, H, T, bf16_trunc=(variant == "bf16_f16"))
    dev.sync()
    ref = O.rmsnorm(x.reshape(T, H), w).reshape(-1)
    if variant == "f16":
        ref = O.f16(ref)
    elif variant == "bf16_f16":
        ref = O.f16(O.bf16_trunc(ref))
        assert_close(host(out), ref, rtol=1e-2, what=variant)  # 1 bf16 ulp band
        return
    assert_close(host(out), ref, what=variant)


def test_rope_and_kv_update(dev):
    """rope (transformer_test.zig:1185-1240 case) and kv_cache_update (:1242-1336)."""
    vals = ((np.arange(16) + 1) * 0.1).astype(np.float32)
    t = tdev(vals)
    ops.dispatch_rope(dev, t, 2, 8, 3, 10000.0)
    dev.sync()
    assert_close(host(t), O.rope(vals.reshape(2, 8), 3, 10000.0).reshape(-1), rtol=1e-5, what="rope")
    # large position, f16 in place
    x = S.normal(430, 16 * 128).astype(np.float16)
    t16 = tdev(x)
    ops.dispatch_rope(dev, t16, 16, 128, 30000, 1e6)
    dev.sync()
    assert_close(host(t16), O.f16(O.rope(x.astype(np.float64).reshape(16, 128), 30000, 1e6).reshape(-1)),
                 what="rope f16")
    # kv update: K[h][pos][d], V[h][d][pos]
    hkv, d, max_ctx, pos = 2, 4, 8, 2
    k = (np.arange(hkv * d) * 0.5).astype(np.float32)
    v = (np.arange(hkv * d) * -0.25).astype(np.float32)
    kc = torch.zeros(hkv * max_ctx * d, dtype=torch.float16, device="cuda")
    vc = torch.zeros(hkv * max_ctx * d, dtype=torch.float16, device="cuda")
    ops.dispatch_kv_cache_update(dev, tdev(k), tdev(v), kc, vc, hkv, d, pos, max_ctx)
    dev.sync()
    K = host(kc).reshape(hkv, max_ctx, d)
    V = host(vc).reshape(hkv, d, max_ctx)
    assert np.array_equal(K[:, pos], k.reshape(hkv, d))
    assert np.array_equal(V[:, :, pos], v.reshape(hkv, d))
    K[:, pos] = 0
    V[:, :, pos] = 0
    assert not K.any() and not V.any()


def test_fused_rope_kernels(dev):
    hkv, hq, d, max_ctx, pos, theta = 8, 16, 128, 64, 17, 1e6
    k = S.normal(440, hkv * d).astype(np.float16)
    v = S.normal(441, hkv * d).astype(np.float16)
    ks = (1 + 0.1 * S.normal(442, d)).astype(np.float32)
    kc = torch.zeros(hkv, max_ctx, d, dtype=torch.float16, device="cuda")
    vc = torch.zeros(hkv, d, max_ctx, dtype=torch.float16, device="cuda")
    ops.dispatch_fused_rope_kv_cache(dev, tdev(k), tdev(v), kc, vc,
                                     L.FusedRoPEKVDims(hkv, d, pos, max_ctx, theta))
    dev.sync()
    kr = O.f16(O.rope(k.astype(np.float64).reshape(hkv, d), pos, theta))
    assert_close(host(kc)[:, pos], kr, what="fused rope kv")
    assert np.array_equal(host(vc)[:, :, pos], v.reshape(hkv, d).astype(np.float64))
    ops.dispatch_fused_k_norm_rope_kv_cache(dev, tdev(k), tdev(v), kc, vc, tdev(ks),
                                            L.FusedKNormRoPEKVDims(hkv, d, pos + 1, max_ctx, 1e-6, theta))
    dev.sync()
    kr2 = O.f16(O.head_norm_rope(k.astype(np.float64).reshape(hkv, d), ks, pos + 1, theta))
    assert_close(host(kc)[:, pos + 1], kr2, what="fused k norm rope kv")
    q = S.normal(443, hq * d).astype(np.float16)
    qd = tdev(q)
    ops.dispatch_fused_norm_rope(dev, qd, tdev(ks), L.FusedNormRoPEDims(hq, d, pos, 1e-6, theta))
    dev.sync()
    assert_close(host(qd).reshape(hq, d),
                 O.f16(O.head_norm_rope(q.astype(np.float64).reshape(hq, d), ks, pos, theta)),
                 what="fused norm rope")


# ------------------------------------------------------- embedding / misc ---
def test_embedding_known_answer(dev):
    """transformer_test.zig:1450-1541 (bits 0xAA, scale 0.5, tokens [1, 3])."""
    ids = tdev(np.array([1, 3], np.int32))
    bits = tdev(np.full(8, 0xAA, np.uint8))
    sc = tdev(np.array([0.5], np.float16))
    out = torch.empty(32, dtype=torch.float32, device="cuda")
    ops.dispatch_embedding_lookup(dev, ids, bits, sc, out, L.EmbedDims(4, 16, 2, 128))
    dev.sync()
    assert np.array_equal(host(out), np.tile([-0.5, 0.5], 16))


def test_embedding_q1_q4_bf16_random(dev):
    V, H = 64, 256
    w1 = cf.q1_matrix(V, H, 128, 450, 451)
    ids = np.array([0, 63, 17, 17, 5], np.int32)
    out = torch.empty(len(ids) * H, dtype=torch.float32, device="cuda")
    ops.dispatch_embedding_lookup(dev, tdev(ids), tdev(w1.codes.view(np.uint8)),
                                  tdev(w1.scales.view(np.float16)), out,
                                  L.EmbedDims(V, H, len(ids), 128))
    dev.sync()
    ref = O.embed_q1(ids, w1.codes.view(np.uint8).reshape(-1), w1.scales.view(np.float16).reshape(-1), H, 128)
    assert np.array_equal(host(out), ref.reshape(-1))
    w4 = cf.q4_matrix(V, H, 64, 452, 453, 454, scale_dtype=1 + 1)
    ops.dispatch_embedding_lookup_q4(dev, tdev(ids), tdev(w4.codes), tdev(w4.scales.view(np.int16)),
                                     tdev(w4.biases.view(np.int16)), out, L.EmbedDims(V, H, len(ids), 64))
    dev.sync()
    ref4 = O.embed_q4(ids, w4.codes, w4.scales, w4.biases, H, 64, 2)
    assert np.array_equal(host(out), ref4.reshape(-1))
    tab = S.f64_to_bf16_bits(S.normal(455, V * H)).reshape(V, H)
    ops.dispatch_embedding_lookup_bf16(dev, tdev(ids), tdev(tab.view(np.int16)), out,
                                       L.EmbedDims(V, H, len(ids), 0))
    dev.sync()
    assert np.array_equal(host(out), S.bf16_bits_to_f32(tab[ids]).reshape(-1).astype(np.float64))


def test_residual_silu_argmax(dev):
    r = tdev(np.arange(1, 9, dtype=np.float32))
    a = tdev((np.arange(1, 9) * 0.1).astype(np.float32))
    ops.dispatch_residual_add(dev, r, a)
    x = S.normal(460, 1000).astype(np.float32)
    s = torch.empty(1000, dtype=torch.float32, device="cuda")
    ops.dispatch_silu(dev, tdev(x), s)
    g, u = S.normal(461, 1000).astype(np.float16), S.normal(462, 1000).astype(np.float16)
    sm = torch.empty(1000, dtype=torch.float16, device="cuda")
    ops.dispatch_silu_elementwise_mul(dev, tdev(g), tdev(u), sm)
    logits = S.normal(463, 151936).astype(np.float32)
    logits[[100, 90000]] = 9.0  # tie: the first maximum wins
    idx = torch.zeros(1, dtype=torch.int32, device="cuda")
    val = torch.zeros(2, dtype=torch.float32, device="cuda")
    ops.dispatch_argmax(dev, tdev(logits), idx, val)
    dev.sync()
    assert np.allclose(host(r), np.arange(1, 9) * 1.1, rtol=1e-6)
    assert_close(host(s), O.silu(x), rtol=1e-5, what="silu")
    assert_close(host(sm), O.f16(O.silu(g.astype(np.float64)) * u), what="silu mul f16")
    assert int(idx.item()) == 100
    assert host(val)[0] == 9.0 and host(val)[1] == 9.0


# ------------------------------------------------------------ prefill GEMM --
@pytest.mark.parametrize("P", [1, 37, 512])
def test_dequant_gemm_modes(dev, P):
    M, K = 1024, 2048
    wa, wb = cf.q1_matrix(M, K, 128, 470, 471), cf.q1_matrix(M, K, 128, 472, 473)
    a16 = (0.5 * S.normal(474, P * K)).astype(np.float16).reshape(P, K)
    A = a16.astype(np.float64)
    da, db = ops.DeviceQWeight(dev, wa), ops.DeviceQWeight(dev, wb)
    ad = tdev(a16)
    ra, rb = A @ O.dequant(wa).T, A @ O.dequant(wb).T
    out16 = torch.empty(P, M, dtype=torch.float16, device="cuda")
    ops.dispatch_dequant_gemm(dev, da, ad, out16, L.GEMM_STORE_F16)
    out32 = torch.empty(P, M, dtype=torch.float32, device="cuda")
    ops.dispatch_dequant_gemm(dev, da, ad, out32, L.GEMM_STORE_F32)
    res0 = S.normal(475, P * M).astype(np.float32).reshape(P, M)
    res = tdev(res0)
    ops.dispatch_dequant_gemm(dev, da, ad, res, L.GEMM_RESADD)
    ops.dispatch_dequant_gemm(dev, da, ad, out16, L.GEMM_SILU_PAIR, wb=db)
    dev.sync()
    assert_close(host(out32), ra, what="gemm f32")
    assert_close(host(res), res0 + ra, what="gemm resadd")
    assert_close(host(out16), O.f16(O.silu(ra) * rb), what="gemm silu pair")


@pytest.mark.parametrize("P,M,K,gs", [(100, 192, 2112, 64), (512, 128, 6144, 128),
                                       (64, 64, 192, 64), (1024, 64, 320, 64),
                                       (512, 4096, 576, 64)])
def test_dequant_gemm_shapes(dev, P, M, K, gs):
    """K not a multiple of the stage (last stage partial), group size 64,
    token tiles that do and do not divide by 8, grids of up to one block per
    CU (eight k-phases) and beyond (four), and the silu pair."""
    wa, wb = cf.q1_matrix(M, K, gs, 490, 491), cf.q1_matrix(M, K, gs, 492, 493)
    a16 = (0.5 * S.normal(494, P * K)).astype(np.float16).reshape(P, K)
    A = a16.astype(np.float64)
    da, db = ops.DeviceQWeight(dev, wa), ops.DeviceQWeight(dev, wb)
    ra, rb = A @ O.dequant(wa).T, A @ O.dequant(wb).T
    ad = tdev(a16)   # held until the sync: the kernels run on the library's stream
    out32 = torch.empty(P, M, dtype=torch.float32, device="cuda")
    ops.dispatch_dequant_gemm(dev, da, ad, out32, L.GEMM_STORE_F32)
    out16 = torch.empty(P, M, dtype=torch.float16, device="cuda")
    ops.dispatch_dequant_gemm(dev, da, ad, out16, L.GEMM_SILU_PAIR, wb=db)
    dev.sync()
    assert_close(host(out32), ra, what="gemm f32")
    assert_close(host(out16), O.f16(O.silu(ra) * rb), what="gemm silu pair")


@pytest.mark.parametrize("P,M,K,gs,sdt", [(37, 256, 2048, 64, 2), (512, 512, 2048, 64, 2),
                                           (100, 128, 6144, 128, 1), (64, 64, 192, 64, 2),
                                           (512, 2560, 2048, 64, 2)])
def test_dequant_gemm_q4_modes(dev, P, M, K, gs, sdt):
    """4-bit (q4_mlx) weights: s * (A . n) + b * sum(A) per group on the MFMA,
    every mode BF16-faithful like the Q4 decode kernels (one bf16 ulp bar).
    The last case has 320 blocks (more than one per CU), so the single-matrix
    modes run the main kernel's two k-phases, as real 4-bit prefill does at
    hidden 2560 (the general kernel's: test_dequant_gemm_q4_general_grids)."""
    from nnzap_amd import formats as fm
    sd = fm.DT_BF16 if sdt == 2 else fm.DT_F16
    wa = cf.q4_matrix(M, K, gs, 520, 521, 522, scale_dtype=sd)
    wb = cf.q4_matrix(M, K, gs, 523, 524, 525, scale_dtype=sd)
    a16 = (0.5 * S.normal(526, P * K)).astype(np.float16).reshape(P, K)
    A = a16.astype(np.float64)
    da, db = ops.DeviceQWeight(dev, wa), ops.DeviceQWeight(dev, wb)
    ra, rb = A @ O.dequant(wa).T, A @ O.dequant(wb).T
    ad = tdev(a16)   # held until the sync: the kernels run on the library's stream
    out16 = torch.empty(P, M, dtype=torch.float16, device="cuda")
    ops.dispatch_dequant_gemm(dev, da, ad, out16, L.GEMM_STORE_F16)
    out32 = torch.empty(P, M, dtype=torch.float32, device="cuda")
    ops.dispatch_dequant_gemm(dev, da, ad, out32, L.GEMM_STORE_F32)
    res0 = S.normal(527, P * M).astype(np.float32).reshape(P, M)
    res = tdev(res0)
    ops.dispatch_dequant_gemm(dev, da, ad, res, L.GEMM_RESADD)
    pair = torch.empty(P, M, dtype=torch.float16, device="cuda")
    ops.dispatch_dequant_gemm(dev, da, ad, pair, L.GEMM_SILU_PAIR, wb=db)
    dev.sync()
    # fp32 summation error of a K-term sum (random-walk bound, 4 sigma)
    se = 4 * 2.0 ** -24 * np.sqrt(K) * (np.abs(A) @ np.abs(O.dequant(wa)).T)
    assert_bf16_faithful(host(out32), ra, "q4 gemm f32", sum_err=se)
    assert_bf16_faithful(host(out16), ra, "q4 gemm f16", sum_err=se)
    # residual += bf16(sum): one bf16 ulp of the added term (the GPU's fp32 sum
    # and the fp64 oracle may straddle a truncation boundary) plus the f32 add
    ref = res0 + O.bf16_trunc(ra)
    err = np.abs(host(res).astype(np.float64) - ref)
    assert (err <= 2.0 ** -7 * np.abs(ra) + 2.0 ** -23 * np.abs(ref) + se + 2.0 ** -30).all(), \
        f"q4 gemm resadd: {int((err > 2.0 ** -7 * np.abs(ra)).sum())} elements beyond one bf16 ulp"
    # silu(a) * b: the fp32 summation errors of a and b propagate through
    # d(silu(a) b) = silu'(a) b da + silu(a) db, |silu'| <= 1.1
    se_b = 4 * 2.0 ** -24 * np.sqrt(K) * (np.abs(A) @ np.abs(O.dequant(wb)).T)
    se_pair = 1.1 * np.abs(rb) * se + np.abs(O.silu(ra)) * se_b
    assert_bf16_faithful(host(pair), O.silu(ra) * rb, "q4 gemm silu pair", sum_err=se_pair)


@pytest.mark.parametrize("P,M,K,gs,sdt", [(512, 2560, 2112, 64, 2), (512, 2560, 2048, 128, 1), (512, 2560, 2048, 64, 1)])
def test_dequant_gemm_q4_general_grids(dev, P, M, K, gs, sdt):
    """4-bit weights that the main kernel does not take (K not a multiple of
    512, group size 128, f16 scales) on 320 blocks: the general kernel's
    two-k-phase single-matrix forms, every mode."""
    test_dequant_gemm_q4_modes(dev, P, M, K, gs, sdt)


def test_dequant_gemm_split_under_capture(dev):
    """A launch that would split K over the context's workspace does not while
    its stream is captured: the graph replays right between eager calls that
    use the workspace, several times over."""
    import ctypes as C
    P, M, K = 45, 192, 4608
    w = cf.q1_matrix(M, K, 128, 484, 485)
    a16 = S.normal(486, P * K).astype(np.float16).reshape(P, K)
    ref = a16.astype(np.float64) @ O.dequant(w).T
    dw, ad, other = ops.DeviceQWeight(dev, w), tdev(a16), tdev(-a16)
    eager, graphed = (torch.empty(P, M, dtype=torch.float32, device="cuda") for _ in range(2))
    dev.call("nnz_graph_begin")
    ops.dispatch_dequant_gemm(dev, dw, ad, graphed, L.GEMM_STORE_F32)
    g = C.c_void_p()
    dev.call("nnz_graph_end", C.byref(g))
    try:
        for _ in range(3):
            graphed.zero_()
            ops.dispatch_dequant_gemm(dev, dw, other, eager, L.GEMM_STORE_F32)
            dev.call("nnz_graph_replay", g)
            dev.sync()
            assert_close(host(graphed), ref, rtol=1e-4, what="graph replay")
            assert_close(host(eager), -ref, rtol=1e-4, what="eager beside the graph")
    finally:
        L.lib().nnz_graph_destroy(g)


def test_gemm_row_equals_decode_qmv(dev):
    """Per-token equivalence: GEMM row p equals the decode QMV of token p."""
    M, K, P = 512, 2048, 8
    w = cf.q1_matrix(M, K, 128, 480, 481)
    a16 = S.normal(482, P * K).astype(np.float16).reshape(P, K)
    dw = ops.DeviceQWeight(dev, w)
    out = torch.empty(P, M, dtype=torch.float32, device="cuda")
    ops.dispatch_dequant_gemm(dev, dw, tdev(a16), out, L.GEMM_STORE_F32)
    y = torch.empty(M, dtype=torch.float32, device="cuda")
    ops.dispatch_qmv_f16in(dev, dw, tdev(a16[5]), y)
    dev.sync()
    assert_close(host(out)[5], host(y), rtol=1e-4, what="gemm row vs qmv")


@pytest.mark.parametrize("bits,P,M,K", [(1, 1, 64, 512), (1, 65, 192, 1536), (1, 64, 128, 4096),
                                        (1, 1030, 3136, 512), (1, 833, 3840, 512),
                                        (1, 45, 192, 4608), (1, 7, 128, 9728), (1, 130, 2112, 6656),
                                        (4, 45, 192, 2560), (4, 70, 4096, 4608),
                                        (4, 1, 64, 512), (4, 65, 192, 1536), (4, 64, 128, 4096),
                                        (4, 1030, 3136, 512), (4, 833, 3840, 512)])
def test_dequant_gemm_main_shapes(dev, bits, P, M, K):
    """The prefill GEMM at the edges of its launch shapes (short 1-bit ones,
    here of up to 128 blocks and K <= 1536, are the general kernel's): one
    token, one past a token tile, one 64-row block, eight and four k-phases, two
    k-phases on 64-row blocks (rows not a multiple of 128, and up to 768 blocks)
    and on 128-row ones, one W chunk and several, K split four and two ways with
    parts of unequal length.  The 4-bit rows hold scales over
    eleven octaves, negative and zero ones among them, each row at a size of
    its own."""
    from nnzap_amd import formats as fm
    from nnzap_amd.formats import QWeight
    rng = np.random.default_rng([bits, P, M, K])

    def weight():
        if bits == 1:
            return cf.q1_matrix(M, K, 128, int(rng.integers(1 << 30)), int(rng.integers(1 << 30)))
        s = np.exp2(rng.uniform(-11, 0, (M, K // 64)) + rng.integers(-20, 20, (M, 1)))
        s *= rng.choice([-1.0, 0.0, 1.0, 1.0], s.shape)
        b = 8 * s * rng.uniform(-1.2, 0.2, s.shape)
        return QWeight(4, M, K, 64, rng.integers(0, 1 << 32, (M, K // 8), dtype=np.uint32),
                       S.f64_to_bf16_bits(s), S.f64_to_bf16_bits(b), fm.DT_BF16)

    wa, wb = weight(), weight()
    a16 = (0.5 * rng.standard_normal((P, K))).astype(np.float16)
    A, da, db = a16.astype(np.float64), ops.DeviceQWeight(dev, wa), ops.DeviceQWeight(dev, wb)
    Wa, Wb = O.dequant(wa), O.dequant(wb)
    ra, rb, ad = A @ Wa.T, A @ Wb.T, tdev(a16)
    out16 = torch.empty(P, M, dtype=torch.float16, device="cuda")
    out32 = torch.empty(P, M, dtype=torch.float32, device="cuda")
    ops.dispatch_dequant_gemm(dev, da, ad, out32, L.GEMM_STORE_F32)
    # residual += on zeros and the f16 store are the same sums, to the bit
    res = torch.zeros(P, M, dtype=torch.float32, device="cuda")
    ops.dispatch_dequant_gemm(dev, da, ad, res, L.GEMM_RESADD)
    ops.dispatch_dequant_gemm(dev, da, ad, out16, L.GEMM_STORE_F16)
    dev.sync()
    assert torch.equal(res, out32) and torch.equal(out16, out32.half())
    if bits == 1:
        ops.dispatch_dequant_gemm(dev, da, ad, out16, L.GEMM_SILU_PAIR, wb=db)
        dev.sync()
        # fp32 summation (random walk, 4 sigma) of terms |a| s
        se = 4 * 2.0 ** -24 * np.sqrt(K) * (np.abs(A) @ np.abs(Wa).T)
        assert (np.abs(host(out32) - ra) <= se).all()
        assert_close(host(out16), O.f16(O.silu(ra) * rb), what="silu pair")
        return
    dev.sync()
    # the sums run over centred weights (n - 8) s and (b + 8 s): their terms
    # bound the summation error
    def terms(w):
        s = S.bf16_bits_to_f32(w.scales).astype(np.float64)[:, :, None]
        b = S.bf16_bits_to_f32(w.biases).astype(np.float64)[:, :, None]
        n = fm.unpack_q4(w.codes, K).reshape(M, K // 64, 64).astype(np.float64)
        return (np.abs((n - 8) * s) + np.abs(b + 8 * s)).reshape(M, K)
    se = 4 * 2.0 ** -24 * np.sqrt(K) * (np.abs(A) @ terms(wa).T)
    assert_bf16_faithful(host(out32), ra, "q4 gemm main", sum_err=se)


@pytest.mark.parametrize("P,M,K", [(256, 4096, 2048), (320, 3072, 2048), (321, 2880, 2048), (1, 64, 1536),
                                   (512, 4096, 512), (513, 3648, 512), (130, 192, 2560)])
def test_dequant_gemm_short_launches(dev, P, M, K):
    """Single 1-bit launches on both sides of the line between the short ones
    (K <= 2048 on up to 256 blocks, K = 512 on up to 512) and the main kernel:
    every store, the fp32 sums within the random-walk bound."""
    w = cf.q1_matrix(M, K, 128, 500, 501)
    a16 = (0.5 * S.normal(502, P * K)).astype(np.float16).reshape(P, K)
    A, W = a16.astype(np.float64), O.dequant(w)
    dw, ad = ops.DeviceQWeight(dev, w), tdev(a16)
    out32 = torch.empty(P, M, dtype=torch.float32, device="cuda")
    res = torch.zeros(P, M, dtype=torch.float32, device="cuda")
    out16 = torch.empty(P, M, dtype=torch.float16, device="cuda")
    ops.dispatch_dequant_gemm(dev, dw, ad, out32, L.GEMM_STORE_F32)
    ops.dispatch_dequant_gemm(dev, dw, ad, res, L.GEMM_RESADD)
    ops.dispatch_dequant_gemm(dev, dw, ad, out16, L.GEMM_STORE_F16)
    dev.sync()
    se = 4 * 2.0 ** -24 * np.sqrt(K) * (np.abs(A) @ np.abs(W).T)
    assert (np.abs(host(out32) - A @ W.T) <= se).all()
    assert torch.equal(res, out32) and torch.equal(out16, out32.half())


def test_dequant_gemm_precision_over_shapes(dev):
    """The launch shape does not cost precision: the fp32 sums of the same 640
    tokens on two k-phases (64-row blocks at 672 and 1280 blocks, 128-row ones
    at 1024) are no further from float64 than on four (320 blocks).  A chain of
    half the roundings is 1 / sqrt(2) of the error, so a launch whose chains are
    twice as long shows as 1.4; 1.1 leaves room for the sample (1.3M sums, the
    ratio of two such norms good to 0.1 %)."""
    M, K, n = 2048, 2560, 640
    w = cf.q1_matrix(M, K, 128, 510, 511)
    dw, W = ops.DeviceQWeight(dev, w), tdev(O.dequant(w))
    a = tdev((0.5 * S.normal(512, 2500 * K)).astype(np.float16).reshape(2500, K))
    ref = a[:n].double() @ W.T

    def error(P):
        out = torch.empty(P, M, dtype=torch.float32, device="cuda")
        ops.dispatch_dequant_gemm(dev, dw, a[:P], out, L.GEMM_STORE_F32)
        dev.sync()
        return float((out[:n].double() - ref).norm() / ref.norm())

    base = error(n)
    for P in (1300, 2048, 2500):
        assert error(P) <= 1.1 * base, (P, error(P), base)


@pytest.mark.parametrize("P,M,K", [(3, 64, 512), (65, 192, 1536), (45, 192, 2560), (70, 4096, 4608),
                                   (1024, 1088, 512), (1030, 3136, 512), (833, 3840, 512)])
def test_dequant_gemm_q4_wide_rows(dev, P, M, K):
    """4-bit rows that the main kernel's scaled f16 weights cannot hold: scales
    2^24 apart (every second token is zero where the large ones are, so only
    the small ones show), scales far below the biases (denormal ones, and none
    at all), and an infinite scale.  Blocks of 32 rows (a wave's) are of one
    kind, the first of ordinary rows.  Every launch shape: four and two
    k-phases, K split four and two ways, 64- and 128-row blocks, pairs."""
    from nnzap_amd import formats as fm
    from nnzap_amd.formats import QWeight
    rng = np.random.default_rng([P, M, K])
    G = K // 64
    kind = (np.arange(M) // 32) % 4   # 0 ordinary, 1 spread, 2 tiny scales, 3 large scales

    def weight():
        s = rng.uniform(0.5, 1.0, (M, G)) / 64 * rng.choice([-1.0, 1.0], (M, G))
        b = 8 * s * rng.uniform(-1.2, 0.2, s.shape)
        s[kind == 1, 1::2] *= 2.0 ** -24
        b[kind == 1, 1::2] *= 2.0 ** -24
        s[kind == 2] *= np.where(rng.random((int((kind == 2).sum()), 1)) < 0.5, 2.0 ** -130, 0.0)
        s[kind == 3] *= 2.0 ** 60
        codes = rng.integers(0, 1 << 32, (M, K // 8), dtype=np.uint32)
        return QWeight(4, M, K, 64, codes, S.f64_to_bf16_bits(s), S.f64_to_bf16_bits(b), fm.DT_BF16)

    wa, wb = weight(), weight()
    if M > 64:   # one more row: infinite in its first group, nibbles >= 1
        wa.scales[40, 0] = 0x7F80
        wa.codes[40] |= np.uint32(0x11111111)
    a16 = (0.5 * rng.standard_normal((P, K))).astype(np.float16)
    a16[0] = np.abs(a16[0]) + np.float16(0.125)
    a16.reshape(P, G, 64)[1::2, 0::2] = 0.0
    A, da, db, ad = a16.astype(np.float64), ops.DeviceQWeight(dev, wa), ops.DeviceQWeight(dev, wb), tdev(a16)

    def ref_and_bound(w):
        sc = S.bf16_bits_to_f32(w.scales).astype(np.float64)[:, :, None]
        bi = S.bf16_bits_to_f32(w.biases).astype(np.float64)[:, :, None]
        n = fm.unpack_q4(w.codes, K).reshape(M, G, 64).astype(np.float64)
        terms = (n * np.abs(sc) + np.abs(bi) + 16 * np.abs(sc)).reshape(M, K)
        # fp32 sums of s n and b, centred or not (random walk, 4 sigma)
        return A @ (sc * n + bi).reshape(M, K).T, 4 * 2.0 ** -24 * np.sqrt(K) * (np.abs(A) @ terms.T)

    out32 = torch.empty(P, M, dtype=torch.float32, device="cuda")
    pair = torch.empty(P, M, dtype=torch.float16, device="cuda")
    ops.dispatch_dequant_gemm(dev, da, ad, out32, L.GEMM_STORE_F32)
    ops.dispatch_dequant_gemm(dev, da, ad, pair, L.GEMM_SILU_PAIR, wb=db)
    dev.sync()
    got, gp = host(out32), host(pair)
    with np.errstate(invalid="ignore"):
        ra, sa = ref_and_bound(wa)
    rb, sb = ref_and_bound(wb)
    rows = np.arange(M) != 40 if M > 64 else np.ones(M, bool)
    if M > 64:
        assert got[0, 40] == np.inf
    assert_bf16_faithful(got[:, rows], ra[:, rows], "wide rows", sum_err=sa[:, rows])
    rows &= kind < 2   # the others leave f16's range
    ra, rb, sa, sb = (v[:, rows] for v in (ra, rb, sa, sb))
    se = 1.1 * np.abs(rb) * sa + np.abs(O.silu(ra)) * sb + 1.1 * sa * sb
    assert_bf16_faithful(gp[:, rows], O.silu(ra) * rb, "wide rows, pair", sum_err=se + 2.0 ** -24)
