"""GPU tests of the varlen causal GQA attention kernels against the CPU oracle
(oracle.ops.attention_varlen_fwd / _bwd, float64 on the same fp16 inputs).

Tolerances follow the kernels' two roundings: P (forward) and dS (backward) are rounded to fp16
for their MFMA products, relative error at most 2^-11 each, and the stored O that the backward's
D = rowsum(dO o O) reads is fp16. Each element's bound is that error carried through the
absolute values of the other operand (computed here in float64 from the same inputs), doubled,
plus one fp16 ulp of the output. lse is fp32: 1e-5 absolute.
"""

from __future__ import annotations

import math

import numpy as np
import pytest
import torch

from oracle import ops as ref
from rus_amd import kernels as K

pytestmark = pytest.mark.gpu
DEV = "cuda"
EPS16 = 2.0**-11


def _inputs(lens, hq, hkv, seed, qk_scale=1.0):
    g = torch.Generator().manual_seed(seed)
    n = sum(lens)
    q = (torch.randn(n, hq, 128, generator=g) * qk_scale).half()
    k = (torch.randn(n, hkv, 128, generator=g) * qk_scale).half()
    v = torch.randn(n, hkv, 128, generator=g).half()
    dout = torch.randn(n, hq, 128, generator=g).half()
    cu = [0]
    for L in lens:
        cu.append(cu[-1] + L)
    return q, k, v, dout, cu


def _dev(*ts):
    return [t.to(DEV) for t in ts]


def _bounds(q, k, v, dout, cu):
    """float64 per-element error bounds (before doubling) for out, dq, dk, dv."""
    n, hq, d = q.shape
    hkv = k.shape[1]
    grp = hq // hkv
    sc = 1.0 / math.sqrt(d)
    q, k, v, dout = q.double(), k.double(), v.double(), dout.double()
    bo = torch.zeros(n, hq, d, dtype=torch.float64)
    bq = torch.zeros_like(bo)
    bk = torch.zeros(n, hkv, d, dtype=torch.float64)
    bv = torch.zeros_like(bk)
    for a, e in zip(cu[:-1], cu[1:]):
        L = e - a
        if L == 0:
            continue
        qh = q[a:e].transpose(0, 1)
        ks = k[a:e].repeat_interleave(grp, dim=1).transpose(0, 1)
        vs = v[a:e].repeat_interleave(grp, dim=1).transpose(0, 1)
        do = dout[a:e].transpose(0, 1)
        s = sc * (qh @ ks.transpose(1, 2))
        s = s.masked_fill(~torch.ones(L, L, dtype=torch.bool).tril(), float("-inf"))
        p = torch.softmax(s, -1)
        o = p @ vs
        ds = p * (do @ vs.transpose(1, 2) - (do * o).sum(-1, keepdim=True))
        # |dS| rounding + P * sum|dO||O| (fp16 O in D)
        eds = EPS16 * ds.abs() + p * EPS16 * (do.abs() * o.abs()).sum(-1, keepdim=True)
        bo[a:e] = (EPS16 * (p @ vs.abs())).transpose(0, 1)
        bq[a:e] = (sc * (eds @ ks.abs())).transpose(0, 1)
        bk[a:e] = (sc * (eds.transpose(1, 2) @ qh.abs())).reshape(hkv, grp, L, d).sum(1).transpose(0, 1)
        bv[a:e] = (EPS16 * (p.transpose(1, 2) @ do.abs())).reshape(hkv, grp, L, d).sum(1).transpose(0, 1)
    return bo, bq, bk, bv


def _check(name, got, want, bound):
    g = got.double().cpu()
    tol = 2.0 * bound + ref.fp16_ulp(want.float()).double() + 1e-6
    err = (g - want).abs()
    bad = err > tol
    assert not bool(bad.any()), (
        f"{name}: {int(bad.sum())} elements out of tolerance, worst excess "
        f"{float((err - tol).max()):.3e} (max err {float(err.max()):.3e})")


def _run(lens, hq, hkv, seed, qk_scale=1.0, check_bwd=True):
    q, k, v, dout, cu = _inputs(lens, hq, hkv, seed, qk_scale)
    out_ref, lse_ref = ref.attention_varlen_fwd(q, k, v, cu)
    bo, bq, bk, bv = _bounds(q, k, v, dout, cu)
    qd, kd, vd, dd = _dev(q, k, v, dout)
    cud = torch.tensor(cu, dtype=torch.int32, device=DEV)
    out, lse = K.attn_varlen_fwd(qd, kd, vd, cud, lens=lens)
    torch.cuda.synchronize()
    _check("out", out, out_ref, bo)
    torch.testing.assert_close(lse.double().cpu(), lse_ref, rtol=1e-6, atol=1e-5)
    if not check_bwd:
        return
    dq_ref, dk_ref, dv_ref = ref.attention_varlen_bwd(dout, q, k, v, cu)
    dq, dk, dv = K.attn_varlen_bwd(dd, qd, kd, vd, out, lse, cud, lens=lens)
    torch.cuda.synchronize()
    _check("dq", dq, dq_ref, bq)
    _check("dk", dk, dk_ref, bk)
    _check("dv", dv, dv_ref, bv)


@pytest.mark.parametrize("lens,hq,hkv", [
    ([1, 17, 32, 33, 64, 100], 12, 2),  # edges of the 32-token blocks, rows at ragged offsets
    ([40, 7], 4, 4),                     # no GQA
    ([70, 1, 1, 5], 8, 1),               # MQA, single-token rows
])
def test_attention_matches_oracle(lens, hq, hkv):
    _run(lens, hq, hkv, seed=sum(lens) + hq)


def test_attention_longest_row():
    _run([512], 12, 2, seed=7)


def test_attention_bench_shaped_batch():
    # 4 rows with lognormal lengths (median 140, mean 220, clipped to [16, 512]) + a padding row
    # of the kind a captured-graph bucket appends.
    rng = np.random.default_rng(11)
    lens = [int(x) for x in np.clip(rng.lognormal(math.log(140), 0.92, 4), 16, 512)]
    lens.append(256 - sum(lens) % 256)
    _run(lens, 12, 2, seed=3)


def test_attention_peaked_scores():
    # Large logits: the running max moves across key blocks (online-softmax rescaling).
    _run([96, 45], 12, 2, seed=5, qk_scale=3.0)


def test_attention_rising_scores():
    # Scores that grow along the row by more than 2^8 per key block: the running maximum
    # (and its lazily updated reference point) moves on every block.
    lens = [200, 70]
    q, k, v, dout, cu = _inputs(lens, 12, 2, seed=8)
    ramp = torch.cat([torch.linspace(0.0, 1.0, L) for L in lens])
    k = (k.float() * 0.1 + 4.0 * ramp[:, None, None]).half()
    q = (q.float() * 0.1 + 1.0).half()
    out_ref, lse_ref = ref.attention_varlen_fwd(q, k, v, cu)
    bo, bq, bk, bv = _bounds(q, k, v, dout, cu)
    qd, kd, vd, dd = _dev(q, k, v, dout)
    cud = torch.tensor(cu, dtype=torch.int32, device=DEV)
    out, lse = K.attn_varlen_fwd(qd, kd, vd, cud)
    dq, dk, dv = K.attn_varlen_bwd(dd, qd, kd, vd, out, lse, cud)
    torch.cuda.synchronize()
    _check("out", out, out_ref, bo)
    torch.testing.assert_close(lse.double().cpu(), lse_ref, rtol=1e-6, atol=1e-4)
    dq_ref, dk_ref, dv_ref = ref.attention_varlen_bwd(dout, q, k, v, cu)
    _check("dq", dq, dq_ref, bq)
    _check("dk", dk, dk_ref, bk)
    _check("dv", dv, dv_ref, bv)


def test_attention_deterministic_and_extra_blocks():
    lens = [33, 90]
    q, k, v, dout, cu = _inputs(lens, 12, 2, seed=1)
    qd, kd, vd, dd = _dev(q, k, v, dout)
    cud = torch.tensor(cu, dtype=torch.int32, device=DEV)
    o1, l1 = K.attn_varlen_fwd(qd, kd, vd, cud)
    o2, l2 = K.attn_varlen_fwd(qd, kd, vd, cud, max_blocks=K.attn_max_blocks(123, 2) + 40)
    g1 = K.attn_varlen_bwd(dd, qd, kd, vd, o1, l1, cud)
    g2 = K.attn_varlen_bwd(dd, qd, kd, vd, o2, l2, cud, max_blocks=64)
    torch.cuda.synchronize()
    assert torch.equal(o1, o2) and torch.equal(l1, l2)
    for a, b in zip(g1, g2):
        assert torch.equal(a, b)


def test_attention_matches_torch_flash_on_device():
    # Same call as the engine's previous path (aten flash attention, varlen, causal).
    lens = [50, 130, 16]
    q, k, v, dout, cu = _inputs(lens, 12, 2, seed=9)
    qd, kd, vd, dd = _dev(q, k, v, dout)
    cud = torch.tensor(cu, dtype=torch.int32, device=DEV)
    out, _ = K.attn_varlen_fwd(qd, kd, vd, cud)
    o_t = torch.ops.aten._flash_attention_forward(qd, kd, vd, cud, cud, max(lens), max(lens), 0.0,
                                                  True, False)[0]
    torch.cuda.synchronize()
    assert (out.float() - o_t.float()).abs().max().item() < 4e-3


@pytest.mark.parametrize("lens,hq,hkv", [([33, 90, 1, 200], 12, 2), ([40, 7], 4, 4), ([70, 5], 8, 1)])
def test_attention_partials_equal_group_sum(lens, hq, hkv):
    # The partial-output backward: dq is the group-summing backward's bit for bit, and each KV
    # head's per-query-head partials summed in head order and rounded once are its dk / dv.
    q, k, v, dout, cu = _inputs(lens, hq, hkv, seed=sum(lens))
    qd, kd, vd, dd = _dev(q, k, v, dout)
    cud = torch.tensor(cu, dtype=torch.int32, device=DEV)
    out, lse = K.attn_varlen_fwd(qd, kd, vd, cud)
    dq, dk, dv = K.attn_varlen_bwd(dd, qd, kd, vd, out, lse, cud)
    dq_p, dk_p, dv_p = K.attn_varlen_bwd_parts(dd, qd, kd, vd, out, lse, cud)
    torch.cuda.synchronize()
    assert torch.equal(dq_p, dq)
    grp = hq // hkv
    for part, full in ((dk_p, dk), (dv_p, dv)):
        acc = part.view(hkv, grp, -1, 128)[:, 0].clone()
        for j in range(1, grp):
            acc += part.view(hkv, grp, -1, 128)[:, j]
        assert torch.equal(acc.half().permute(1, 0, 2).contiguous(), full)


@pytest.mark.parametrize("hq,hkv", [(2, 1), (6, 2), (5, 1), (14, 2)])
def test_attention_group_sum_of_every_group_size(hq, hkv):
    """dk and dv of the group sizes the other tests leave out (2, 3, 5, 7): the partials in head order,
    rounded once, with a last block of the sum that is part empty."""
    q, k, v, dout, cu = _inputs([33, 4], hq, hkv, seed=hq)
    qd, kd, vd, dd = _dev(q, k, v, dout)
    cud = torch.tensor(cu, dtype=torch.int32, device=DEV)
    out, lse = K.attn_varlen_fwd(qd, kd, vd, cud)
    full = K.attn_varlen_bwd(dd, qd, kd, vd, out, lse, cud)
    parts = K.attn_varlen_bwd_parts(dd, qd, kd, vd, out, lse, cud)
    torch.cuda.synchronize()
    assert torch.equal(parts[0], full[0])
    for part, got in zip(parts[1:], full[1:]):
        part = part.view(hkv, hq // hkv, -1, 128)
        acc = part[:, 0].clone()
        for j in range(1, hq // hkv):
            acc += part[:, j]
        assert torch.equal(acc.half().permute(1, 0, 2).contiguous(), got)


def test_rope_mid_over_attention_partials_equals_group_sum_path():
    # Attention partials -> RoPE backward that sums them equals attention group sum -> RoPE
    # backward, for all five outputs, bit for bit (bench-shaped heads, rank 16).
    lens = [100, 37, 250]
    hq, hkv, hd, r = 12, 2, 128, 16
    q, k, v, dout, cu = _inputs(lens, hq, hkv, seed=21)
    qd, kd, vd, dd = _dev(q, k, v, dout)
    cud = torch.tensor(cu, dtype=torch.int32, device=DEV)
    n = sum(lens)
    g = torch.Generator().manual_seed(5)
    ang = torch.rand(600, hd, generator=g) * 6.3
    cos, sin = ang.cos().half().to(DEV), ang.sin().half().to(DEV)
    pos = torch.randint(0, 600, (n,), generator=g).to(DEV)
    bqt = (torch.randn(r, hq * hd, generator=g) * 0.05).half().to(DEV)
    bvt = (torch.randn(r, hkv * hd, generator=g) * 0.05).half().to(DEV)
    out, lse = K.attn_varlen_fwd(qd, kd, vd, cud)
    dq, dk, dv = K.attn_varlen_bwd(dd, qd, kd, vd, out, lse, cud)
    want = K.qkv_rope_bwd_lora_mid(dq, dk, dv, cos, sin, pos, 2.0, 0.5, bqt, bvt,
                                   h_q=hq, h_kv=hkv, head_dim=hd)
    dq_p, dk_p, dv_p = K.attn_varlen_bwd_parts(dd, qd, kd, vd, out, lse, cud)
    got = K.qkv_rope_bwd_lora_mid_parts(dq_p, dk_p, dv_p, cos, sin, pos, 2.0, 0.5, bqt, bvt,
                                        h_q=hq, h_kv=hkv, head_dim=hd)
    torch.cuda.synchronize()
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("lens,hq,hkv", [
    ([1100, 385, 129, 128, 127, 33, 1, 950], 12, 2),  # edges of the 128-token blocks
    ([1537, 2048, 600], 8, 8),                         # no GQA
    ([2047, 2050], 8, 1),                              # MQA
])
def test_attention_wide_blocks_match_oracle(lens, hq, hkv):
    """Batches large enough for the 128-token blocks (edges of blocks and tiles, rows shorter than a
    block, ragged offsets), with large scores in one of them so that the running maximum moves."""
    _run(lens, hq, hkv, seed=sum(lens) + hq, qk_scale=3.0 if hkv == 1 else 1.0)


def _exact(q, k, v, dout, lens):
    """float64 (out, dq, dk, dv) on the device, one head at a time."""
    leaves = [t.double().requires_grad_(True) for t in (q, k, v)]
    qd, kd, vd = leaves
    grp, outs, a = q.shape[1] // k.shape[1], [], 0
    for n in lens:
        causal = torch.ones(n, n, dtype=torch.bool, device=q.device).tril()
        heads = []
        for h in range(q.shape[1]):
            s = qd[a:a + n, h] @ kd[a:a + n, h // grp].t().contiguous() / math.sqrt(128)
            p = torch.softmax(s.masked_fill(~causal, -math.inf), -1)
            heads.append(p @ vd[a:a + n, h // grp])
        outs.append(torch.stack(heads, 1))
        a += n
    out = torch.cat(outs)
    return [out.detach(), *torch.autograd.grad(out, leaves, dout.double())]


@pytest.mark.parametrize("qk_scale", [1.0, 3.0])
def test_wide_attention_is_as_accurate_as_the_narrow_blocks(qk_scale):
    """16 rows of 512 in one call (128-token blocks) and one call each (32-token blocks): the errors
    of both against float64 are those of P's fp16 rounding and of the outputs', and the first must not
    exceed the second's by more than 1% (their own scatter over inputs is 0.3%)."""
    lens, (hq, hkv) = [512] * 16, (12, 2)
    q, k, v, dout, cu = _inputs(lens, hq, hkv, seed=2, qk_scale=qk_scale)
    q, k, v, dout = _dev(q, k, v, dout)

    def run(a, b, rows):
        c = torch.tensor(rows, dtype=torch.int32, device=DEV)
        x = [t[a:b].contiguous() for t in (q, k, v, dout)]
        out, lse = K.attn_varlen_fwd(*x[:3], c)
        return [out, *K.attn_varlen_bwd(x[3], *x[:3], out, lse, c)]

    wide = run(0, cu[-1], cu)
    narrow = [torch.cat(t) for t in zip(*(run(a, a + 512, [0, 512]) for a in cu[:-1]))]
    for name, w, s, x in zip(("out", "dq", "dk", "dv"), wide, narrow, _exact(q, k, v, dout, lens)):
        e_w, e_s = (float((t.double() - x).norm() / x.norm()) for t in (w, s))
        assert e_w <= 1.01 * e_s, (name, e_w, e_s)


def test_mixed_rows_below_the_wide_lines_take_the_narrow_blocks():
    """One long row among short ones, too few blocks for the 128-token kernels: the 32-token blocks,
    whose results do not depend on the rest of the batch, so each row alone gives the same bits."""
    lens = [1024] + [35] * 11
    q, k, v, dout, cu = _inputs(lens, 12, 2, seed=4)
    q, k, v, dout = _dev(q, k, v, dout)

    def run(a, b, rows):
        c = torch.tensor(rows, dtype=torch.int32, device=DEV)
        x = [t[a:b].contiguous() for t in (q, k, v, dout)]
        out, lse = K.attn_varlen_fwd(*x[:3], c)
        return [out, *K.attn_varlen_bwd(x[3], *x[:3], out, lse, c)]

    whole = run(0, cu[-1], cu)
    alone = [torch.cat(t) for t in zip(*(run(a, b, [0, b - a]) for a, b in zip(cu[:-1], cu[1:])))]
    for a, b in zip(whole, alone):
        assert torch.equal(a, b)


# batches for the 128-token blocks of both passes: over 64 rows, empty ones among them, none longer
# than a block; a few long rows
WIDE_SHORT = [(37 * i) % 129 for i in range(100)]
WIDE_LONG = [1500, 0, 300, 129, 1400]


@pytest.mark.parametrize("lens,hq,hkv", [
    (WIDE_SHORT, 12, 2),
    (WIDE_LONG, 12, 2),
    ([512] * 4, 12, 2),  # 192 blocks: 32-token blocks forward, 128-token blocks backward
    ([1700, 1790, 1500], 8, 8),
    ([2400, 2500], 8, 1),
])
def test_attention_wide_row_mixtures_match_oracle(lens, hq, hkv):
    _run(lens, hq, hkv, seed=len(lens), qk_scale=3.0 if hkv == 1 else 1.0)


@pytest.mark.parametrize("lens", [WIDE_SHORT, [1700, 1500]])
def test_attention_wide_rising_scores(lens):
    """As test_attention_rising_scores for the 128-token blocks: the running maximum moves at every
    pair of key tiles, by more than 2^8 where the row is long."""
    q, k, v, dout, cu = _inputs(lens, 12, 2, seed=8)
    ramp = torch.cat([torch.linspace(0.0, 1.0, n) for n in lens])
    k = (k.float() * 0.1 + 24.0 * ramp[:, None, None]).half()
    q = (q.float() * 0.1 + 1.0).half()
    out_ref, lse_ref = ref.attention_varlen_fwd(q, k, v, cu)
    bounds = _bounds(q, k, v, dout, cu)
    qd, kd, vd, dd = _dev(q, k, v, dout)
    cud = torch.tensor(cu, dtype=torch.int32, device=DEV)
    out, lse = K.attn_varlen_fwd(qd, kd, vd, cud)
    grads = K.attn_varlen_bwd(dd, qd, kd, vd, out, lse, cud)
    torch.cuda.synchronize()
    _check("out", out, out_ref, bounds[0])
    torch.testing.assert_close(lse.double().cpu(), lse_ref, rtol=1e-6, atol=1e-4)
    want = ref.attention_varlen_bwd(dout, q, k, v, cu)
    for name, g, w, b in zip(("dq", "dk", "dv"), grads, want, bounds[1:]):
        _check(name, g, w, b)


@pytest.mark.parametrize("lens", [WIDE_SHORT, WIDE_LONG])
def test_attention_wide_deterministic_extra_blocks_and_partials(lens):
    """The 128-token blocks give the same bits again and with more blocks announced than there are;
    their per-query-head partials, summed in head order and rounded once, are dk and dv."""
    hq, hkv = 12, 2
    q, k, v, dout, cu = _inputs(lens, hq, hkv, seed=1)
    qd, kd, vd, dd = _dev(q, k, v, dout)
    cud = torch.tensor(cu, dtype=torch.int32, device=DEV)
    more = K.attn_max_blocks(sum(lens), len(lens)) + 40
    o1, l1 = K.attn_varlen_fwd(qd, kd, vd, cud)
    o2, l2 = K.attn_varlen_fwd(qd, kd, vd, cud, max_blocks=more)
    g1 = K.attn_varlen_bwd(dd, qd, kd, vd, o1, l1, cud)
    g2 = K.attn_varlen_bwd(dd, qd, kd, vd, o2, l2, cud, max_blocks=more)
    parts = K.attn_varlen_bwd_parts(dd, qd, kd, vd, o1, l1, cud)
    torch.cuda.synchronize()
    assert torch.equal(o1, o2) and torch.equal(l1, l2)
    for a, b in zip(g1, g2):
        assert torch.equal(a, b)
    assert torch.equal(parts[0], g1[0])
    for part, full in zip(parts[1:], g1[1:]):
        part = part.view(hkv, hq // hkv, -1, 128)
        acc = part[:, 0].clone()
        for j in range(1, hq // hkv):
            acc += part[:, j]
        assert torch.equal(acc.half().permute(1, 0, 2).contiguous(), full)
