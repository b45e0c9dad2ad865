"""GPU parity of the vocab-tiled lm_head cross-entropy (fp16 MFMA) against the CPU oracle.

Cases follow solution/test_kernels.py:189-226 (B=2, S=32, D=256, V=4099, chunk 1024, masked
prompt labels) plus the BASELINE config 2 shape (N=2048, D=1536, V=151936, 10% labels -100),
whose per-token results, hidden gradient and loss are checked against the oracle for every
token.

Tolerances (written per assertion): loss / entropy / lse within 1e-3 absolute; nll within 1e-3
plus one fp16 ulp of the target logit (the fp32 accumulation order of an MFMA differs from the
CPU GEMM, so the fp16 rounding of a logit can land one ulp apart); argmax equal except where the
oracle's top two fp16 logits are within one ulp; hidden gradient within rtol 1e-2.
"""

from __future__ import annotations

import pytest
import torch

from oracle import ops as ref
from rus_amd import kernels as K

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _check_against_oracle(h, w, labels, out, rows=None, denom=None, check_dh=True):
    nll, lse, ent, amax, dn, dh_pre = out[:6]
    rows = torch.arange(h.shape[0]) if rows is None else rows
    o = ref.lm_head_ce(h[rows], w, labels[rows], num_items_in_batch=denom, v_chunk=16384,
                       need_grad=check_dh)
    lse_g, ent_g, nll_g = lse.cpu()[rows], ent.cpu()[rows], nll.cpu()[rows]
    assert torch.all((lse_g - o["lse"]).abs() <= 1e-3)
    assert torch.all((ent_g - o["entropy"]).abs() <= 1e-3)
    lab = labels[rows]
    tgt_ulp = torch.zeros_like(o["nll"])
    valid = lab != -100
    if valid.any():
        z_t = (h[rows][valid].float() * w[lab[valid]].float()).sum(-1).half().float()
        tgt_ulp[valid] = ref.fp16_ulp(z_t)
    assert torch.all((nll_g - o["nll"]).abs() <= 1e-3 + tgt_ulp)
    # argmax: exact unless the oracle's top-2 fp16 logits are within one ulp of each other.
    z = ref.lm_head_logits(h[rows], w)
    top2 = z.topk(2, dim=-1).values
    near_tie = (top2[:, 0] - top2[:, 1]) <= ref.fp16_ulp(top2[:, 0])
    am = amax.cpu()[rows]
    assert torch.all((am == o["argmax"]) | near_tie)
    assert torch.all(z.gather(1, am[:, None]).squeeze(1) >= top2[:, 0] - ref.fp16_ulp(top2[:, 0]))
    if check_dh:
        dh = K.lm_head_dh_reduce(dh_pre.unsqueeze(0), 1.0 / 65536.0, torch.float16).cpu()[rows]
        want = o["dh"].float()
        scale = want.abs().max().item() + 1e-12
        assert torch.allclose(dh.float(), want, rtol=1e-2, atol=1e-2 * scale)
    return o


@pytest.mark.parametrize("v_chunk", [None, 1024])
def test_lmhead_reference_case(v_chunk):
    # solution/test_kernels.py:192-220: B=2, S=32, D=256, V=4099, chunk 1024, 8 masked labels/row.
    g = torch.Generator().manual_seed(3)
    B, S, D, V = 2, 32, 256, 4099
    hidden = torch.randn(B, S, D, generator=g).half()
    weight = (torch.randn(V, D, generator=g) * 0.02).half()
    labels = torch.randint(0, V, (B, S), generator=g)
    labels[:, :8] = -100
    shift = torch.full((B, S), -100, dtype=torch.long)
    shift[:, :-1] = labels[:, 1:]
    h2, lab = hidden.view(-1, D), shift.view(-1)
    out = K.lm_head_ce(h2.to(DEV), weight.to(DEV), lab.to(DEV), v_chunk=v_chunk)
    torch.cuda.synchronize()
    o = _check_against_oracle(h2, weight, lab, out)
    loss = out[0].sum().cpu() / out[4].cpu()
    assert abs(float(loss) - float(o["loss"])) <= 1e-3
    assert abs(float(out[6].cpu()) - float(loss)) <= 1e-6 * abs(float(loss))  # device loss kernel
    # Full-logit library reference, as the reference test does (test_kernels.py:203-217).
    z = h2.float() @ weight.float().t()
    loss_lib = torch.nn.functional.cross_entropy(z, lab, ignore_index=-100)
    assert abs(float(loss) - float(loss_lib)) <= 2e-3


@pytest.mark.parametrize("v_chunk", [None, 8192])
def test_lmhead_unpadded_vocab_chunked(v_chunk):
    g = torch.Generator().manual_seed(4)
    N, D, V = 777, 1536, 32901  # V not a multiple of 64: padded K in the gradient GEMM
    h = torch.randn(N, D, generator=g).half()
    w = (torch.randn(V, D, generator=g) * 0.02).half()
    lab = torch.randint(0, V, (N,), generator=g)
    lab[torch.rand(N, generator=g) < 0.1] = -100
    lab[-1] = V - 1
    out = K.lm_head_ce(h.to(DEV), w.to(DEV), lab.to(DEV), v_chunk=v_chunk)
    torch.cuda.synchronize()
    rows = torch.cat([torch.arange(0, 64), torch.tensor([N - 1])])
    denom = float(out[4].item())
    _check_against_oracle(h, w, lab, out, rows=rows, denom=denom)


def test_lmhead_baseline_config2_all_tokens():
    # H [2048,1536] ~ N(0,1), W [151936,1536] ~ N(0,0.02), 10% labels -100:
    # every token's statistics and hidden-gradient row against the oracle, and the loss.
    g = torch.Generator().manual_seed(0)
    N, D, V = 2048, 1536, 151936
    h = torch.randn(N, D, generator=g).half()
    w = (torch.randn(V, D, generator=g) * 0.02).half()
    lab = torch.randint(0, V, (N,), generator=g)
    lab[torch.rand(N, generator=g) < 0.1] = -100
    out = K.lm_head_ce(h.to(DEV), w.to(DEV), lab.to(DEV))
    torch.cuda.synchronize()
    denom = float(out[4].item())
    assert denom == float((lab != -100).sum())
    o = _check_against_oracle(h, w, lab, out, denom=denom)
    assert abs(float(out[6].cpu()) - float(o["loss"])) <= 1e-3
    nll = out[0].cpu()
    assert torch.all(nll[lab == -100] == 0)
    # size-independent invariants over every token: 0 <= H <= ln V, lse >= max logit.
    ent = out[2].cpu()
    assert torch.all(ent >= -1e-4) and torch.all(ent <= torch.log(torch.tensor(float(V))) + 1e-4)


def test_lmhead_token_block_size_leaves_the_statistics_unchanged():
    # 1100 tokens in five 256-token blocks and in two (768 + 332, the default for a small
    # vocabulary, which allows any block size but never one block for all tokens):
    # each token's logits, statistics and argmax are formed from its own row alone, so they are
    # bit-identical; the hidden gradient's split-K sum order follows the block's split count, so
    # it agrees within rtol 1e-3 and both match the oracle on a sample of tokens.
    g = torch.Generator().manual_seed(11)
    N, D, V = 1100, 256, 5000
    h = torch.randn(N, D, generator=g).half()
    w = (torch.randn(V, D, generator=g) * 0.05).half()
    lab = torch.randint(0, V, (N,), generator=g)
    lab[torch.rand(N, generator=g) < 0.1] = -100
    assert K.lm_head_token_blocks(N, K.lm_head_block_tokens(V)) == [(0, 768), (768, N)]
    two = K.lm_head_ce(h.to(DEV), w.to(DEV), lab.to(DEV))
    five = K.lm_head_ce(h.to(DEV), w.to(DEV), lab.to(DEV), block_tokens=256)
    torch.cuda.synchronize()
    for i in (0, 1, 2, 3, 4, 6):
        assert torch.equal(two[i].cpu(), five[i].cpu()), i
    assert torch.allclose(two[5].cpu(), five[5].cpu(), rtol=1e-3, atol=1e-3 * two[5].abs().max().item())
    rows = torch.cat([torch.arange(0, 20), torch.arange(760, 780), torch.arange(1080, 1100)])
    _check_against_oracle(h, w, lab, two, rows=rows, denom=float(two[4].item()))
    _check_against_oracle(h, w, lab, five, rows=rows, denom=float(five[4].item()))


def test_lmhead_all_masked_and_ties():
    N, D, V = 8, 64, 700
    h = torch.ones(N, D).half()
    w = torch.zeros(V, D).half()
    w[3] = 0.01
    w[600] = 0.01  # tie between index 3 and 600 (different 256-row partials)
    lab = torch.full((N,), -100, dtype=torch.long)
    nll, lse, ent, amax, denom, dh_pre, loss = K.lm_head_ce(h.to(DEV), w.to(DEV), lab.to(DEV))
    torch.cuda.synchronize()
    assert float(denom.item()) == 1.0 and float(loss.item()) == 0.0
    assert torch.all(nll.cpu() == 0)
    assert torch.all(amax.cpu() == 3)
    assert torch.all(dh_pre.cpu() == 0)


def test_lmhead_num_items_in_batch_scales_gradient():
    g = torch.Generator().manual_seed(5)
    N, D, V = 100, 128, 1000
    h = torch.randn(N, D, generator=g).half().to(DEV)
    w = (torch.randn(V, D, generator=g) * 0.05).half().to(DEV)
    lab = torch.randint(0, V, (N,), generator=g).to(DEV)
    a = K.lm_head_ce(h, w, lab)
    b = K.lm_head_ce(h, w, lab, num_items_in_batch=2 * N)
    torch.cuda.synchronize()
    assert float(a[4].item()) == N and float(b[4].item()) == 2 * N
    assert torch.allclose(a[5].cpu() * 0.5, b[5].cpu(), rtol=1e-2, atol=1e-3)


@pytest.mark.parametrize("n,d,v,start", [(37, 128, 1031, 0), (300, 256, 4099, 0), (64, 64, 700, 256)])
def test_kept_logits_gradient_equals_recomputed_gradient(n, d, v, start):
    # Single-pass head: the statistics pass keeps its fp16 logits in the gradient buffer and the
    # elementwise pass turns them into the gradient; both must give the bits of the recompute
    # GEMM's epilogue. Ragged vocabulary (v % 64 != 0), masked labels, labels outside the range.
    g = torch.Generator().manual_seed(n + v)
    h = torch.randn(n, d, generator=g).half()
    w = (torch.randn(start + v, d, generator=g) * 0.05).half()
    lab = torch.randint(0, start + v, (n,), generator=g)
    lab[torch.rand(n, generator=g) < 0.2] = -100
    hd, wd, ld = h.to(DEV), w[start:].to(DEV), lab.to(DEV)
    kp = (v + 63) // 64 * 64
    parts = K.LMHeadPartials(start // 256 + K.lm_head_num_parts(v), n, DEV)
    parts.m.fill_(-float("inf"))
    parts.s.zero_()
    parts.w.zero_()
    parts.idx.fill_(0)
    tgt_a = torch.zeros(n, dtype=torch.float32, device=DEV)
    tgt_b = torch.zeros(n, dtype=torch.float32, device=DEV)
    z = torch.full((n, kp + 64), 7.0, dtype=torch.float16, device=DEV)  # stride > kp
    K.lm_head_ce_fwd_chunk(hd, wd, ld, start, parts, tgt_a, logits_out=z[:, :kp])
    m_keep = parts.m.clone()
    K.lm_head_ce_fwd_chunk(hd, wd, ld, start, parts, tgt_b)
    torch.cuda.synchronize()
    assert torch.equal(m_keep, parts.m) and torch.equal(tgt_a, tgt_b)
    zc = z.cpu()
    assert torch.all(zc[:, v:kp] == 0) and torch.all(zc[:, kp:] == 7.0)
    # the kept logits are fp16(H.W^T) of an fp32 accumulation: the two fp32 sums differ by at
    # most d * 2^-24 * sum|h_i w_i| (summation order), then each rounds to fp16 (an ulp apart at
    # most, taken at the larger binade)
    want = (h.float() @ w[start:].float().T).half().float()
    acc_err = d * 2.0 ** -24 * (h.abs().float() @ w[start:].abs().float().T)
    assert torch.all((zc[:, :v].float() - want).abs() <= 2 * ref.fp16_ulp(want) + acc_err)
    lse = torch.randn(n, generator=g).abs().to(DEV) + zc[:, :v].float().amax(1).to(DEV)
    denom = torch.tensor([float((lab != -100).sum())], dtype=torch.float32, device=DEV)
    g_ref = torch.empty((n, kp), dtype=torch.float16, device=DEV)
    K.lm_head_ce_grad_logits(hd, wd, ld, lse, denom, start, g_ref)
    K.lm_head_ce_grad_from_logits(z[:, :kp], ld, lse, denom, v, start)
    torch.cuda.synchronize()
    assert torch.equal(z[:, :kp].cpu(), g_ref.cpu())
    assert torch.all(z[:, kp:].cpu() == 7.0)


@pytest.mark.parametrize("n,d,v,chunk", [(300, 256, 5000, 1024), (700, 1536, 20000, 8192)])
def test_single_pass_head_chunking_and_streaming(n, d, v, chunk):
    # The single-pass head over different vocabulary chunkings: statistics bit-identical (the
    # per-256-row partials do not depend on the chunking), hidden gradient within rtol 1e-2 of the
    # oracle. A HostHead streamed from pinned host memory with the same chunk gives the resident
    # head's bits, including the gradient; back-to-back calls without the gradient (which leave a
    # streamed slot's last reader to the next call's prefetch) and with it, on fresh inputs.
    from rus_amd import ops
    from rus_amd.hostload import HostHead

    g = torch.Generator().manual_seed(n + v)
    w = (torch.randn(v, d, generator=g) * 0.03).half()
    lab = torch.randint(0, v, (n,), generator=g)
    lab[torch.rand(n, generator=g) < 0.1] = -100
    lab[0] = v - 1  # a label in the last (partial) chunk
    labd = lab.to(DEV)
    streamed = HostHead(w, DEV, v_chunk=chunk, resident=False)
    resident = HostHead(w, DEV, v_chunk=chunk, resident=True)
    for step, need_grad in enumerate((False, False, True, True, False)):
        h = torch.randn(n, d, generator=g).half()
        outs = []
        for head in (streamed, resident):
            hd = h.to(DEV).requires_grad_(need_grad)
            with torch.set_grad_enabled(need_grad):
                loss, nll, ent, amax = ops.chunked_lm_head(hd, labd, head, v_chunk=chunk)
            if need_grad:
                loss.backward()
            torch.cuda.synchronize()
            outs.append((loss.detach().cpu(), nll.cpu(), ent.cpu(), amax.cpu(),
                         hd.grad.cpu() if need_grad else None))
        for a, b in zip(outs[0][:4], outs[1][:4]):
            assert torch.equal(a, b), step
        if need_grad:
            assert torch.equal(outs[0][4], outs[1][4]), step
    # the last gradient against the oracle; other chunkings agree on the statistics bitwise
    out = K.lm_head_ce(h.to(DEV), w.to(DEV), labd, v_chunk=chunk)
    auto = K.lm_head_ce(h.to(DEV), w.to(DEV), labd)
    torch.cuda.synchronize()
    # the token-blocked default forms the statistics per row (another fp32 summation order):
    # same argmax, lse / nll / entropy / loss within a few fp32 ulps of the chunked pass
    assert torch.equal(out[3].cpu(), auto[3].cpu())
    for i in (0, 1, 2, 6):
        assert torch.allclose(out[i].cpu(), auto[i].cpu(), rtol=1e-6, atol=2e-5), i
    rows = torch.arange(0, min(n, 40))
    _check_against_oracle(h, w, lab, out, rows=rows, denom=float(out[4].item()))
    _check_against_oracle(h, w, lab, auto, rows=rows, denom=float(auto[4].item()))


def test_chunk_choice_bounds_the_logit_buffer():
    # The default chunk keeps the per-chunk fp16 logits within the 128 MiB budget at any token
    # count and, from a few hundred tokens up, below the whole vocabulary (the [N, V] logits are
    # never held); a small vocabulary fits one chunk.
    assert K.LM_CHUNK_BUDGET == 128 << 20
    for n in (1, 707, 2048, 8192, 65536):
        c = K.lm_head_chunk_cols(n, 151936)
        assert c % 256 == 0 and c >= 256
        assert n * c * 2 <= max(K.LM_CHUNK_BUDGET, n * 256 * 2)
        if n >= 512:
            assert c < 151936
    assert K.lm_head_chunk_cols(64, 4099) >= 4099


@pytest.mark.parametrize("n,d,v", [(37, 128, 1031), (256, 1536, 20000), (5, 64, 700)])
def test_row_kernel_statistics_and_gradient(n, d, v):
    # Logits GEMM + per-row kernel: statistics against the oracle (1e-3; argmax exact unless an
    # oracle near-tie); the in-place gradient equals, bit for bit, the recompute GEMM's epilogue
    # given the same lse (same formula on the same fp16 logits), zeros past the vocabulary.
    g = torch.Generator().manual_seed(n * 7 + v)
    h = torch.randn(n, d, generator=g).half()
    w = (torch.randn(v, d, generator=g) * 0.05).half()
    lab = torch.randint(0, v, (n,), generator=g)
    lab[torch.rand(n, generator=g) < 0.2] = -100
    lab[0] = v - 1
    hd, wd, ld = h.to(DEV), w.to(DEV), lab.to(DEV)
    kp = (v + 63) // 64 * 64
    z = torch.full((n, kp + 64), 7.0, dtype=torch.float16, device=DEV)
    K.lm_head_ce_logits(hd, wd, z[:, :kp])
    lse = torch.empty(n, device=DEV)
    nll, ent = torch.empty_like(lse), torch.empty_like(lse)
    amax = torch.empty(n, dtype=torch.int64, device=DEV)
    zc = z.clone()
    K.lm_head_ce_rows(zc[:, :kp], v, ld, None, lse, nll, ent, amax)  # statistics only
    torch.cuda.synchronize()
    assert torch.equal(zc.cpu(), z.cpu())
    assert torch.all(z[:, v:kp].cpu() == 0) and torch.all(z[:, kp:].cpu() == 7.0)
    denom = torch.tensor([float(max((lab != -100).sum(), 1))], device=DEV)
    lse2, nll2, ent2 = torch.empty_like(lse), torch.empty_like(lse), torch.empty_like(lse)
    amax2 = torch.empty_like(amax)
    K.lm_head_ce_rows(z[:, :kp], v, ld, denom, lse2, nll2, ent2, amax2)
    g_ref = torch.empty((n, kp), dtype=torch.float16, device=DEV)
    K.lm_head_ce_grad_logits(hd, wd, ld, lse2, denom, 0, g_ref)
    torch.cuda.synchronize()
    assert torch.equal(lse.cpu(), lse2.cpu()) and torch.equal(amax.cpu(), amax2.cpu())
    assert torch.equal(z[:, :kp].cpu(), g_ref.cpu())
    assert torch.all(z[:, kp:].cpu() == 7.0)
    o = ref.lm_head_ce(h, w, lab, v_chunk=4096, need_grad=False)
    assert torch.all((lse.cpu() - o["lse"]).abs() <= 1e-3)
    assert torch.all((ent.cpu() - o["entropy"]).abs() <= 1e-3)
    zo = ref.lm_head_logits(h, w)
    tgt_ulp = torch.zeros(n)
    valid = lab != -100
    tgt_ulp[valid] = ref.fp16_ulp(zo[valid, lab[valid]])
    assert torch.all((nll.cpu() - o["nll"]).abs() <= 1e-3 + tgt_ulp)
    top2 = zo.topk(2, dim=-1).values
    near_tie = (top2[:, 0] - top2[:, 1]) <= ref.fp16_ulp(top2[:, 0])
    assert torch.all((amax.cpu() == o["argmax"]) | near_tie)


@pytest.mark.parametrize("n,v,chunk", [(37, 1216, 256), (300, 1100, 512), (5, 700, 256)])
@pytest.mark.parametrize("shifts", [(0, 0, 0, 0, 0), (-300, 0, 12, 40, 300), (300, 40, 0, -8, -1000),
                                    (0, 5, -1000, 9, -60)])
def test_single_pass_probabilities_over_logit_ranges(n, v, chunk, shifts):
    """The stored probabilities are relative to references that follow the chunks' maxima: logits
    whose level jumps between 256-row tiles, by less and by more than the window, up and down. The
    reference forms softmax from the device's own fp16 logits in float64; each element of dH may
    differ by P's fp16 rounding (2^-11 of each product, doubled) and fp32 sums of terms that size."""
    g = torch.Generator().manual_seed(n + v)
    d = 128
    h = torch.randn(n, d, generator=g)
    h[:, 0] = 4.0
    w = torch.randn(v, d, generator=g) * 0.1
    for t, s in enumerate(shifts):
        w[256 * t: 256 * (t + 1), 0] = s / 4.0
    h, w = h.half().to(DEV), w.half().to(DEV)
    labels = torch.randint(0, v, (n,), generator=g)
    labels[::3] = -100
    labels = labels.to(DEV)
    z = torch.empty(n, K._round_up(v, 64), dtype=torch.float16, device=DEV)
    K.lm_head_ce_logits(h, w, z)
    nll, lse, ent, amax, denom, dh, loss = K.lm_head_ce(h, w, labels, v_chunk=chunk)
    torch.cuda.synchronize()
    z = z[:, :v].double().cpu()
    p = torch.softmax(z, -1)
    assert torch.allclose(lse.double().cpu(), torch.logsumexp(z, -1), rtol=1e-6, atol=1e-5)
    want_ent = torch.logsumexp(z, -1) - (p * z).sum(-1)
    # w / s is of the logits' size and is subtracted from lse: fp32 resolution of that size
    assert torch.all((ent.double().cpu() - want_ent).abs() <= 1e-5 + 1e-6 * z.abs().amax(-1))
    assert torch.equal(amax.cpu(), z.argmax(-1))
    valid = (labels != -100).cpu()
    scale = 65536.0 / max(1, int(valid.sum()))
    wd, y = w.double().cpu(), labels.clamp(min=0).cpu()
    want = (p @ wd - wd[y]) * scale * valid[:, None]
    tol = scale * (2.0**-10 * (p @ wd.abs()) + 1e-5 * (wd[y].abs() + p @ wd.abs())) + 1e-6
    err = (dh.double().cpu() - want).abs()
    assert bool((err <= tol).all()), float((err / tol).max())


@pytest.mark.parametrize("n", [1, 32, 33, 64, 65, 128, 129, 192, 193, 256, 257, 352])
def test_lmhead_of_token_tiles_partly_filled(n):
    """Column quarters of a tile without a token are left out: token counts on both sides of each
    (and of the 32 tokens of an MFMA tile), with a last vocabulary tile half inside. 64 items: the
    oracle's gradient is 2^16 / items times at most 1 x |w|, |w| < 0.6, in fp16 (with the one item
    of the smallest case it overflows)."""
    g = torch.Generator().manual_seed(n)
    d, v = 128, 1100
    h = torch.randn(n, d, generator=g).half()
    w = (torch.randn(v, d, generator=g) * 0.1).half()
    lab = torch.randint(0, v, (n,), generator=g)
    lab[1::7] = -100
    for chunk in (512, None):
        out = K.lm_head_ce(h.to(DEV), w.to(DEV), lab.to(DEV), num_items_in_batch=64.0,
                           v_chunk=chunk)
        _check_against_oracle(h, w, lab, out, denom=64.0)
    out = K.lm_head_ce(h.to(DEV), w.to(DEV), lab.to(DEV), num_items_in_batch=64.0,
                       need_grad=False)
    _check_against_oracle(h, w, lab, out, denom=64.0, check_dh=False)


@pytest.mark.parametrize("n,v,chunk", [(37, 1216, 256), (300, 1100, 512)])
def test_pass_over_kept_logits_agrees_with_the_stored_probabilities(n, v, chunk):
    """The launchers that keep a chunk's logits and scale them by the running maximum, against the
    single pass: both round P to fp16 once (2^-11 relative), so two gradients differ by at most
    2^-10 of sum P |w| plus the fp32 sums (doubled: p below comes from unrounded logits)."""
    g = torch.Generator().manual_seed(v)
    d = 128
    h = (torch.randn(n, d, generator=g) * 2).half().to(DEV)
    w = (torch.randn(v, d, generator=g) * 0.3).half().to(DEV)
    labels = torch.randint(0, v, (n,), generator=g).to(DEV)
    want = K.lm_head_ce(h, w, labels, num_items_in_batch=64.0, v_chunk=chunk)
    wt = K.lm_head_weight_t(w)
    parts, target = K.LMHeadPartials(K.lm_head_num_parts(v), n, DEV), torch.zeros(n, device=DEV)
    z = torch.empty(n, K._round_up(chunk, 64), dtype=torch.float16, device=DEV)
    m_run, alpha = torch.empty(n, device=DEV), torch.empty(n, device=DEV)
    acc = torch.empty(1, n, d, device=DEV)
    for c in range(0, v, chunk):
        rows = w[c:c + chunk]
        K.lm_head_ce_fwd_chunk(h, rows, labels, c, parts, target, logits_out=z)
        K.lm_head_ce_chunk_scale(z, rows.shape[0], parts, c // 256, m_run, alpha, c == 0)
        K.lm_head_ce_grad_hidden_scaled(z, wt[:, c:], rows.shape[0], acc, c > 0, alpha)
    lse, nll, _, amax = K.lm_head_ce_combine(parts, target, labels)
    denom = torch.tensor([64.0], device=DEV)
    dh = K.lm_head_ce_dh_finish(acc, m_run, lse, labels, w, denom, 1.0, None, torch.float32)
    assert torch.equal(amax, want[3]) and torch.allclose(lse, want[1], rtol=1e-6, atol=1e-5)
    hp = K.LMHeadPass(n, d, v, v, DEV, True)  # chunks shorter than announced
    for c in range(0, v, 256):
        hp.add_chunk(h, w[c:c + 256], wt[:, c:], c, labels)
    short = hp.finish(labels, 64.0, w)
    p = torch.softmax(h.double() @ w.double().t(), -1)
    tol = 1024.0 * (2.0**-9 * (p @ w.double().abs()) + 1e-4)
    for other in (dh, short[5]):
        assert bool(((other.double() - want[5].double()).abs() <= tol).all())


def _peaked(n, d, v, label_up, other_up, seed):
    """Tokens whose label's and one other row's logit are raised above the rest (0: not raised),
    with ignored labels and labels outside the vocabulary among them."""
    g = torch.Generator().manual_seed(seed)
    h = torch.randn(n, d, generator=g)
    w = torch.randn(v, d, generator=g) * 0.05
    rows = torch.randperm(v, generator=g)[: 2 * n]
    dirs = h / h.pow(2).sum(1, keepdim=True)
    w[rows[:n]] += label_up * dirs
    w[rows[n:]] += other_up * dirs
    labels = rows[:n].clone()
    labels[3::11] = -100
    labels[5], labels[6] = v + 300, -7
    return h.half().to(DEV), w.half().to(DEV), labels.to(DEV)


# log(sum of the other logits) is about 9.3: mean nll near 1e-1, 1e-3 and 1e-5 with the label the
# argmax; another row at p 0.999; label and another row at about one half each; nothing raised
@pytest.mark.parametrize("label_up,other_up", [(11.6, 0), (16.2, 0), (20.8, 0), (0, 16.2),
                                               (18.0, 18.0), (0, 0)])
@pytest.mark.parametrize("layout", ["chunks", "one chunk", "256 rows", "streamed", "blocks"])
def test_hidden_gradient_of_peaked_tokens(layout, label_up, other_up):
    """dH of tokens that the model predicts well, or wrongly with confidence, against float64 softmax
    of the device's own fp16 logits. In the single pass only the probabilities beside the label and
    the largest other one are rounded to fp16 (2^-11 relative, 2^-24 of the largest below fp16's
    normal range); the rest is fp32 relative to lse's size. The token blocks round G once and form
    p - 1 from lse, whose fp32 resolution stays in the label's coefficient."""
    from rus_amd import ops
    from rus_amd.hostload import HostHead

    n, d, v = 300, 256, 8192 + 130
    h, w, labels = _peaked(n, d, v, label_up, other_up, seed=int(10 * label_up + other_up))
    if layout == "streamed":
        head = HostHead(w.cpu(), DEV, v_chunk=2048, resident=False)
        out = ops._lm_head_streamed(h, labels, head, None, True)
    else:
        chunk = {"chunks": 2048, "one chunk": 33 * 256, "256 rows": 256, "blocks": None}[layout]
        out = K.lm_head_ce(h, w, labels, v_chunk=chunk)
    nll, lse, dh = out[0], out[1], out[5]
    z = torch.empty(n, K._round_up(v, 64), dtype=torch.float16, device=DEV)
    K.lm_head_ce_logits(h, w, z)
    torch.cuda.synchronize()
    z, wd, y = z[:, :v].double().cpu(), w.double().cpu(), labels.cpu()
    want_lse = torch.logsumexp(z, -1)
    e32 = 2.0**-22 * (4 + want_lse.abs())
    assert bool(((lse.double().cpu() - want_lse).abs() <= e32).all())
    inside = (y >= 0) & (y < v)
    at = torch.arange(n)
    yc = torch.where(inside, y, 0)
    p = torch.exp(z - want_lse[:, None])
    p_y = torch.where(inside, p[at, yc], 0.0)
    others = p.clone()
    others[at[inside], y[inside]] = 0
    rest = torch.where(inside, others.sum(1), 0.0)
    want_nll = torch.where(inside, -torch.log1p(-rest), want_lse) * (y != -100)
    assert bool(((nll.double().cpu() - want_nll).abs() <= e32).all())
    scale = 65536.0 / int((y != -100).sum())
    live = (y != -100)[:, None]
    want = (others @ wd - rest[:, None] * wd[yc]) * scale * live
    top = others.amax(1)
    rounded = others.clone()
    if layout != "blocks":
        rounded[at, others.argmax(1)] *= (top < 0.065).double()
    mag = others @ wd.abs() + rest[:, None] * wd[yc].abs()
    tol = 2.0**-11 * (rounded @ wd.abs()) + 2.0**-24 * top[:, None] * wd.abs().sum(0)
    tol = tol + 2 * e32[:, None] * mag
    if layout == "blocks":
        tol = tol + 2.0**-11 * rest[:, None] * wd[yc].abs() + 2.0**-25 / scale * wd.abs().sum(0) \
            + e32[:, None] * p_y[:, None] * wd[yc].abs()
    got = dh.double().cpu()
    err = (got - want).abs()
    assert bool((err <= tol * scale + 1e-30).all()), float((err / (tol * scale + 1e-30)).max())
    if layout != "blocks":
        assert float((got - want).norm() / want.norm()) <= 1e-3


def test_labels_past_the_vocabulary_within_its_last_tile():
    """A label of the last 256-row tile that is no vocabulary row counts as outside the vocabulary
    (target logit 0, no weight row), whatever lies in the tile's padding."""
    n, d, v = 70, 128, 700  # rows 700 .. 767 pad the third tile
    g = torch.Generator().manual_seed(3)
    h = torch.randn(n, d, generator=g).half().to(DEV)
    w = (torch.randn(v, d, generator=g) * 0.2).half().to(DEV)
    labels = torch.randint(0, v, (n,), generator=g).to(DEV)
    labels[::2] = torch.arange(700, 735, device=DEV)
    far = torch.where(labels >= v, labels + 1000, labels)
    for kw in ({"v_chunk": 256}, {"v_chunk": 1024}, {"need_grad": False}, {"block_tokens": 256}):
        a, b = (K.lm_head_ce(h, w, lab, **kw) for lab in (labels, far))
        for x, y in zip(a, b):
            assert (x is None and y is None) or torch.equal(x, y), kw
        assert torch.equal(a[0][::2], a[1][::2])  # nll = lse - 0


@pytest.mark.parametrize("kw", [{"v_chunk": 256}, {"v_chunk": 512}, {"v_chunk": 1280},
                                {"need_grad": False}, {"block_tokens": 256}])
def test_nan_logit_far_below_the_maximum_stays_in_the_loss(kw):
    """A NaN among logits far below the rest (here e^-400 of the total) is not summed away."""
    n, d, v = 300, 128, 1100
    g = torch.Generator().manual_seed(5)
    h, w = torch.randn(n, d, generator=g), torch.randn(v, d, generator=g) * 0.1
    h[:, 0] = 4.0
    w[:, 0] = 50.0
    w[256:512, 0] = -50.0
    w[300, 5] = float("nan")
    labels = torch.randint(0, 200, (n,), generator=g)
    out = K.lm_head_ce(h.half().to(DEV), w.half().to(DEV), labels.to(DEV), **kw)
    for i in (0, 1, 2, 6):  # nll, lse, entropy, loss
        assert bool(out[i].isnan().all()), i
    if out[5] is not None:
        assert bool(out[5].isnan().all())


@pytest.mark.parametrize("v,chunk", [(513, 512), (513, 256), (385, 256), (2, 256), (1, 256)])
def test_label_alone_in_its_rows_and_equal_to_the_maximum(v, chunk):
    """The label as the only vocabulary row of a chunk, of a half tile and of the vocabulary, and level
    with the maximum from either side of it (the first index is the argmax): float64 over the device's
    own logits, tolerances of fp32 and of one fp16 rounding of the other probabilities."""
    n, d = 40, 64
    g = torch.Generator().manual_seed(v)
    h = torch.randn(n, d, generator=g)
    w = torch.randn(v, d, generator=g) * 0.3
    labels = torch.full((n,), v - 1)
    if v > 300:
        h[:, 0], w[:, 0] = 4.0, 0.0
        w[7, 0] = 8.0
        w[300] = w[7]  # both 32 above the rest, equal in every element
        labels[::3], labels[1::3] = 7, 300
    h, w, labels = h.half().to(DEV), w.half().to(DEV), labels.to(DEV)
    nll, lse, ent, amax, _, dh, _ = K.lm_head_ce(h, w, labels, v_chunk=chunk)
    z = torch.empty(n, K._round_up(v, 64), dtype=torch.float16, device=DEV)
    K.lm_head_ce_logits(h, w, z)
    torch.cuda.synchronize()
    z, wd, y = z[:, :v].double().cpu(), w.double().cpu(), labels.cpu()
    at = torch.arange(n)
    want_lse = torch.logsumexp(z, -1)
    p = torch.exp(z - want_lse[:, None])
    e32 = 2.0**-22 * (4 + z.abs().amax(-1))
    assert bool(((lse.double().cpu() - want_lse).abs() <= e32).all())
    assert bool(((nll.double().cpu() - (want_lse - z[at, y])).abs() <= e32).all())
    assert bool(((ent.double().cpu() - (want_lse - (p * z).sum(-1))).abs() <= 4 * e32).all())
    assert torch.equal(amax.cpu(), (z == z.amax(-1, keepdim=True)).int().argmax(-1))
    p[at, y] = 0
    rest = p.sum(1, keepdim=True)
    scale = 65536.0 / n
    want, mag = (p @ wd - rest * wd[y]) * scale, (p @ wd.abs() + rest * wd[y].abs()) * scale
    err = (dh.double().cpu() - want).abs()
    tol = (2.0**-11 + 2 * e32[:, None]) * mag + 2.0**-24 * scale * wd.abs().sum(0)
    assert bool((err <= tol).all()), float((err / tol.clamp(min=1e-30)).max())
    if v == 1:
        assert float(dh.abs().max()) == 0.0
