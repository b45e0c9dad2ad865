"""Performance cases: the work a QLoRA training run on packed tokens has this framework do.

Each case is one call (or one forward/backward pair) through a public entry point at the widths of
the repository's training configuration (hidden 1536, intermediate 8960, 12 query and 2 KV heads of
128, vocabulary 151936, LoRA rank 16 on q and v), over the token counts such runs meet: from one
short row of 16 tokens, over the default batch (4 rows, median length 140, up to 512), to batches of
rows as long as the rotary table (2048 positions).

Kinds of case:
  norm     residual add + RMSNorm, forward and backward: under autograd (``ops.rms_norm``, the
           patched model's norm) or by the launchers, as the engine calls them
  glu      SwiGLU over a fused [gate | up], forward and backward, in the same two ways
  lora     a layer's LoRA branches around attention: dropout bits, LoRA-down, LoRA delta + RoPE;
           then the adjoint RoPE with d_mid and the weight / input gradients (``kernels``)
  attn     varlen causal GQA attention, forward and backward (``kernels.attn_varlen_*``)
  head     the lm_head cross-entropy, with the hidden gradient (training) or without (evaluation)
  dequant  one layer's four NF4 segments to fp16 (``kernels.dequant_nf4_segments``)
  stack    decoder layers forward and backward, eager, engine defaults (``FusedQwen2StackFn``)
  step     a whole captured training step of a shallow model (``graph.GraphedTrainStep``)
"""

import math

import numpy as np
import torch
import torch.nn.functional as F

from rus_amd import graph, hostload, kernels, model, ops, quant

HIDDEN, INTER, HEADS, KV_HEADS, HEAD_DIM, VOCAB = 1536, 8960, 12, 2, 128, 151936
RANK, ALPHA, DROPOUT, EPS, THETA, MAX_POS = 16, 32.0, 0.05, 1e-6, 1e6, 2048
Q_DIM, KV_DIM = HEADS * HEAD_DIM, KV_HEADS * HEAD_DIM
SCALE = ALPHA / RANK
LOSS_SCALE = 1024.0  # fp16 training scales the loss: the hidden gradient stays in fp16's range
MASK_SEED = 20240607  # dropout seed of the passes: the same masks each time
LAYER_WEIGHTS = (Q_DIM + 2 * KV_DIM) * HIDDEN + HIDDEN * Q_DIM + 3 * HIDDEN * INTER

# Row lengths of the default batch distribution (lognormal, median 140, mean 220, 16 to 512).
DEFAULT_ROWS = "289,94,207,117"  # 707 tokens, the average step
LONG_ROWS = "2048,1237,1811,640,2048,377"  # 8161 tokens, rows up to the rotary table


def listed():
    return [
        # one short row: nothing but launch latency and the host path
        {"name": "norm_16", "kind": "norm", "n": 16, "d": HIDDEN, "dtype": "float16",
         "autograd": True},
        # the norm of a batch of long rows: bandwidth
        {"name": "norm_16381", "kind": "norm", "n": 16381, "d": HIDDEN, "dtype": "float16",
         "autograd": False},
        # the MLP activation of the default batch's largest size (config 4 of the benchmark)
        {"name": "glu_880", "kind": "glu", "n": 880, "inner": INTER, "dtype": "float16",
         "autograd": False},
        # LoRA branches and rotary embedding of one layer, default batch and long rows
        {"name": "lora_707", "kind": "lora", "lens": DEFAULT_ROWS},
        {"name": "lora_8161", "kind": "lora", "lens": LONG_ROWS},
        # attention of one layer, default batch and long rows
        {"name": "attn_707", "kind": "attn", "lens": DEFAULT_ROWS},
        {"name": "attn_8161", "kind": "attn", "lens": LONG_ROWS},
        # loss and hidden gradient at the largest batch of rows up to 512 (config 2)
        {"name": "head_2048", "kind": "head", "n": 2048, "train": True},
        # evaluation loss of a small batch
        {"name": "head_eval_345", "kind": "head", "n": 345, "train": False},
        # the weights of one layer, decoded once per layer and pass
        {"name": "dequant_layer", "kind": "dequant", "rows_qkv": Q_DIM + 2 * KV_DIM,
         "hidden": HIDDEN, "inner": INTER},
        # decoder layers at a long-row batch, eager (the drop-in path), activations recomputed
        {"name": "stack_8161", "kind": "stack", "layers": 2, "lens": LONG_ROWS},
        # the training step as the benchmark runs it, 4 layers deep
        {"name": "step_707", "kind": "step", "layers": 4, "lens": DEFAULT_ROWS},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _row_lengths(rng, total, longest):
    """Rows of uneven length, together about ``total`` tokens."""
    lens = []
    while total > 0:
        n = min(total, _log_int(rng, min(16, total), min(longest, max(16, total))))
        lens.append(max(1, n))
        total -= lens[-1]
    return ",".join(map(str, lens[:64]))


def draw(rng):
    kind = rng.choice(["norm", "glu", "lora", "attn", "head", "dequant", "stack", "step"])
    if kind == "norm":
        return {"kind": kind, "n": _log_int(rng, 16, 16384),
                "d": rng.choice([512, 896, 1024, HIDDEN, HIDDEN, HIDDEN, 2048]),
                "dtype": rng.choice(["float16", "float16", "float16", "float32"]),
                "autograd": rng.random() < 0.3}
    if kind == "glu":
        return {"kind": kind, "n": _log_int(rng, 16, 8192),
                "inner": rng.choice([1111, 2816, 4864, INTER, INTER, INTER]),
                "dtype": rng.choice(["float16", "float16", "float16", "float32"]),
                "autograd": rng.random() < 0.3}
    if kind in ("lora", "attn"):
        return {"kind": kind, "lens": _row_lengths(rng, _log_int(rng, 16, 8192),
                                                   rng.choice([512, MAX_POS]))}
    if kind == "head":
        return {"kind": kind, "n": _log_int(rng, 16, 2048), "train": rng.random() < 0.75}
    if kind == "dequant":
        hidden = 64 * rng.randint(8, 24)
        return {"kind": kind, "rows_qkv": 64 * rng.randint(8, 32), "hidden": hidden,
                "inner": 64 * rng.randint(16, 140)}
    if kind == "stack":
        return {"kind": kind, "layers": rng.randint(1, 2),
                "lens": _row_lengths(rng, _log_int(rng, 16, 8000), rng.choice([512, MAX_POS]))}
    return {"kind": kind, "layers": rng.randint(1, 4),
            "lens": _row_lengths(rng, _log_int(rng, 16, 2000), 512)}


# ---------------------------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------------------------


def _lens(case):
    return [int(x) for x in case["lens"].split(",")]


class _Draws:
    """Seeded normal / integer tensors on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(self, *shape, std=1.0, mean=0.0, dtype=torch.float16):
        return (torch.randn(*shape, generator=self.g, device="cuda") * std + mean).to(dtype)

    def ints(self, lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=self.g, device="cuda")


def _labels(draws, n):
    """Uniform labels, a tenth of them ignored."""
    lab = draws.ints(0, VOCAB, n)
    return torch.where(draws.ints(0, 10, n) == 0, torch.full_like(lab, -100), lab)


def _positions(lens):
    return torch.cat([torch.arange(n, dtype=torch.int64) for n in lens]).cuda()


def _cu(lens):
    return torch.tensor([0] + list(np.cumsum(lens)), dtype=torch.int32, device="cuda")


def _norm_inputs(case, seed):
    d = _Draws(seed)
    dt = getattr(torch, case["dtype"])
    n, w = case["n"], case["d"]
    return {"x": d.normal(n, w, dtype=dt), "res": d.normal(n, w, dtype=dt),
            "weight": d.normal(w, std=0.05, mean=1.0, dtype=torch.float32),
            "dy": d.normal(n, w, std=0.1, dtype=dt), "dh": d.normal(n, w, std=0.1, dtype=dt)}


def _glu_inputs(case, seed):
    d = _Draws(seed)
    dt = getattr(torch, case["dtype"])
    return {"gu": d.normal(case["n"], 2 * case["inner"], dtype=dt),
            "dout": d.normal(case["n"], case["inner"], std=0.1, dtype=dt)}


def _lora_inputs(case, seed):
    d = _Draws(seed)
    lens = _lens(case)
    n = sum(lens)
    s = {"x": d.normal(n, HIDDEN), "qkv": d.normal(n, Q_DIM + 2 * KV_DIM, std=0.8),
         "pos": _positions(lens), "dq": d.normal(n, HEADS, HEAD_DIM, std=0.1),
         "dk": d.normal(HEADS, n, HEAD_DIM, std=0.1, dtype=torch.float32),
         "dv": d.normal(HEADS, n, HEAD_DIM, std=0.1, dtype=torch.float32)}
    for b, out in (("q", Q_DIM), ("v", KV_DIM)):
        s["A" + b] = d.normal(RANK, HIDDEN, std=0.02)
        s["B" + b] = d.normal(out, RANK, std=0.02)
    return s


def _attn_inputs(case, seed):
    d = _Draws(seed)
    n = sum(_lens(case))
    return {"q": d.normal(n, HEADS, HEAD_DIM), "k": d.normal(n, KV_HEADS, HEAD_DIM),
            "v": d.normal(n, KV_HEADS, HEAD_DIM), "dout": d.normal(n, HEADS, HEAD_DIM, std=0.1)}


def _head_inputs(case, seed):
    d = _Draws(seed)
    return {"h": d.normal(case["n"], HIDDEN), "w": d.normal(VOCAB, HIDDEN, std=0.02),
            "labels": _labels(d, case["n"])}


def _segments(case, seed):
    """The layer's NF4 projections by segment: [q | k | v], o, [gate | up], down."""
    d = _Draws(seed)
    hid, inner, rows = case["hidden"], case["inner"], case["rows_qkv"]
    kv = rows // 8 // 64 * 64
    shapes = [[(rows - 2 * kv, hid), (kv, hid), (kv, hid)], [(hid, rows - 2 * kv)],
              [(inner, hid), (inner, hid)], [(hid, inner)]]
    return [[quant.quantize_nf4(d.normal(*sh, std=0.02)) for sh in group]
            for group in shapes]


def _model(case, seed):
    """A random model of ``layers`` layers on the GPU, and the draws its inputs go on from."""
    d = _Draws(seed)
    cfg = model.Qwen2Config(num_hidden_layers=case["layers"], lora_dropout=DROPOUT)

    def w(rows, cols):
        return quant.quantize_nf4(d.normal(rows, cols, std=0.02))

    def factor(rows, cols):
        return torch.nn.Parameter(d.normal(rows, cols, std=0.02, dtype=torch.float32))

    def norm_weight():
        return d.normal(HIDDEN, std=0.05, mean=1.0, dtype=torch.float32)

    layers = [model.LayerWeights(
        q=w(Q_DIM, HIDDEN), k=w(KV_DIM, HIDDEN), v=w(KV_DIM, HIDDEN), o=w(HIDDEN, Q_DIM),
        gate=w(INTER, HIDDEN), up=w(INTER, HIDDEN), down=w(HIDDEN, INTER),
        q_bias=d.normal(Q_DIM, std=0.02), k_bias=d.normal(KV_DIM, std=0.02),
        v_bias=d.normal(KV_DIM, std=0.02), ln1=norm_weight(), ln2=norm_weight(),
        q_A=factor(RANK, HIDDEN), q_B=factor(Q_DIM, RANK), v_A=factor(RANK, HIDDEN),
        v_B=factor(KV_DIM, RANK)) for _ in range(case["layers"])]
    vocab = VOCAB if case["kind"] == "step" else 1024  # the stack alone never reads the head
    embed = d.normal(vocab, HIDDEN, std=0.02)
    return model.QLoRAQwen2(cfg, layers, embed, norm_weight()), d


def _stack_inputs(case, seed):
    m, d = _model(case, seed)
    n = sum(_lens(case))
    # hidden states of embedding size, and a loss-scaled gradient of the final norm's output
    return {"model": m, "h": d.normal(n, HIDDEN, std=0.02), "d_final": d.normal(n, HIDDEN, std=0.01)}


def _step_inputs(case, seed):
    m, _ = _model(case, seed)
    lens = _lens(case)
    g = torch.Generator().manual_seed(int(seed))
    ids = torch.randint(0, VOCAB, (len(lens), max(lens)), generator=g)
    mask = torch.zeros_like(ids)
    for r, n in enumerate(lens):
        mask[r, :n] = 1
    labels = torch.where(mask.bool(), ids, torch.full_like(ids, -100))
    return {"model": m, "ids": ids, "mask": mask, "labels": labels}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "norm":
        s = _norm_inputs(case, seed)
        s["x"].requires_grad_(case["autograd"])
        s["res"].requires_grad_(case["autograd"])
        return dict(s, kind=kind)
    if kind == "glu":
        s = _glu_inputs(case, seed)
        s["gu"].requires_grad_(case["autograd"])
        return dict(s, kind=kind)
    if kind == "lora":
        s = _lora_inputs(case, seed)
        s["cos"], s["sin"] = ops.rope_cache(MAX_POS, HEAD_DIM, THETA, "cuda")
        for f in ("Aq", "Av", "Bq", "Bv"):  # the rank-major copies a step makes once
            s[f + "t"] = s[f].t().contiguous()
        s["seed"] = torch.tensor([MASK_SEED], dtype=torch.int64, device="cuda")
        return dict(s, kind=kind)
    if kind == "attn":
        return dict(_attn_inputs(case, seed), kind=kind, cu=_cu(_lens(case)))
    if kind == "head":
        s = _head_inputs(case, seed)
        s["h"].requires_grad_(case["train"])
        return {"kind": kind, "h": s["h"], "labels": s["labels"], "train": case["train"],
                "head": hostload.HostHead(s["w"], "cuda")}
    if kind == "dequant":
        segs = []
        for group in _segments(case, seed):
            w, split, offs, bases = quant.concat_segments(group)
            segs.append({"packed": w.packed, "absmax": w.absmax, "absmax2": w.absmax2,
                         "offset": offs, "out_shape": w.shape, "split_bytes": split,
                         "absmax2_bases": bases,
                         "out_buf": torch.empty(w.shape, dtype=torch.float16, device="cuda")})
        return {"kind": kind, "segments": segs, "code2": w.code2}
    lens = _lens(case)
    if kind == "stack":
        s = _stack_inputs(case, seed)
        engine = ops.Qwen2FusedEngine(s["model"], "cuda", resident_weights=True,
                                      dropout_seed=MASK_SEED)
        return {"kind": kind, "engine": engine, "h": s["h"], "pos": _positions(lens),
                "lens": lens, "d_final": s["d_final"]}
    s = _step_inputs(case, seed)
    engine = ops.Qwen2FusedEngine(s["model"], "cuda", resident_weights=True, recompute=False,
                                  dequant_once=True, dropout_seed=MASK_SEED)
    step = graph.GraphedTrainStep(engine)
    batch = (s["ids"].pin_memory(), s["mask"].pin_memory(), s["labels"].pin_memory())
    step.prepare(*batch)
    return {"kind": kind, "engine": engine, "step": step, "batch": batch}


# ---------------------------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------------------------


def _run_lora(s):
    n = s["x"].shape[0]
    bits = kernels.dropout_keep_bits(s["seed"], 0, 2, n, HIDDEN, DROPOUT, DROPOUT)
    drop = (bits[0], bits[1], DROPOUT, DROPOUT)
    mid_q, mid_v = kernels.lora_down_rows(s["x"], s["Aq"], s["Av"], *drop)
    q, k, v = kernels.qkv_rope_fwd_mid(s["qkv"], mid_q, mid_v, s["Bq"], s["Bv"], s["cos"],
                                       s["sin"], s["pos"], SCALE, SCALE, HEADS, KV_HEADS, HEAD_DIM)
    dqkv, dql, dvl, dmq, dmv = kernels.qkv_rope_bwd_lora_mid_parts(
        s["dq"], s["dk"], s["dv"], s["cos"], s["sin"], s["pos"], SCALE, SCALE, s["Bqt"], s["Bvt"],
        h_q=HEADS, h_kv=KV_HEADS, head_dim=HEAD_DIM)
    dx = torch.zeros_like(s["x"])
    grads = [torch.empty_like(s[f]) for f in ("Aq", "Bq", "Av", "Bv")]
    kernels.lora_bwd_w(s["x"], dql, dvl, mid_q, mid_v, dmq, dmv, *grads, *drop,
                       expand=(s["Aqt"], s["Avt"], dx))
    return [q, k, v, dqkv, dx, *grads]


def run(state):
    kind, s = state["kind"], state
    if kind == "norm" and not s["x"].requires_grad:
        y, h, rstd = kernels.rms_norm_fwd(s["x"], s["weight"], eps=EPS, residual=s["res"])
        return [y, h, kernels.rms_norm_bwd(s["dy"], h, s["weight"], rstd, dresidual=s["dh"])]
    if kind == "norm":
        y, h = ops.rms_norm(s["x"], s["weight"], EPS, s["res"])
        dx, _ = torch.autograd.grad((y, h), (s["x"], s["res"]), (s["dy"], s["dh"]))
        return [y, h, dx]
    if kind == "glu" and not s["gu"].requires_grad:
        out = kernels.mlp_glu_fwd(s["gu"])
        return [out, kernels.mlp_glu_bwd(s["dout"], s["gu"], dgu_out=torch.empty_like(s["gu"]))]
    if kind == "glu":
        out = ops.mlp_glu(s["gu"])
        (dgu,) = torch.autograd.grad(out, s["gu"], s["dout"])
        return [out, dgu]
    if kind == "lora":
        return _run_lora(s)
    if kind == "attn":
        out, lse = kernels.attn_varlen_fwd(s["q"], s["k"], s["v"], s["cu"])
        dq, dk, dv = kernels.attn_varlen_bwd(s["dout"], s["q"], s["k"], s["v"], out, lse, s["cu"])
        return [out, lse, dq, dk, dv]
    if kind == "head":
        loss, nll, ent, amax = ops.chunked_lm_head(s["h"], s["labels"], s["head"])
        if not s["train"]:
            return [loss, nll, ent, amax]
        (dh,) = torch.autograd.grad(loss * LOSS_SCALE, s["h"])
        return [loss, nll, ent, amax, dh]
    if kind == "dequant":
        return kernels.dequant_nf4_segments(s["segments"], s["code2"])
    eng = s["engine"]
    eng.dropout_seed.fill_(MASK_SEED)  # a pass's masks are those of its seed
    if kind == "stack":
        final = ops.FusedQwen2StackFn.apply(s["h"], s["pos"], s["lens"], eng, True,
                                            *eng.lora_params)
        grads = torch.autograd.grad(final, eng.lora_params, s["d_final"])
        return [final, *grads]
    loss = s["step"].step(*s["batch"])
    nll, ent, amax = s["step"].last_token_outputs()
    return [loss, nll, ent, amax, *(p.grad for p in eng.lora_params)]


# ---------------------------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------------------------


def _attn_flops(lens):
    """(forward, backward): two, then five products over the causal half."""
    fwd = sum(2.0 * n * (n + 1) * HEAD_DIM * HEADS for n in lens)
    return fwd, 2.5 * fwd


def work(case):
    kind = case["kind"]
    if kind == "norm":
        e = 2 if case["dtype"] == "float16" else 4
        # x, residual -> y, h; dy, dh (h kept) -> dx
        return {"bytes": 7.0 * e * case["n"] * case["d"], "flops": 10.0 * case["n"] * case["d"]}
    if kind == "glu":
        e = 2 if case["dtype"] == "float16" else 4
        # gate, up -> out; dout -> d_gate, d_up
        return {"bytes": 6.0 * e * case["n"] * case["inner"],
                "flops": 20.0 * case["n"] * case["inner"]}
    if kind == "dequant":
        n = case["rows_qkv"] * case["hidden"] + 3 * case["hidden"] * case["inner"]
        kv = case["rows_qkv"] // 8 // 64 * 64
        n += (case["rows_qkv"] - 2 * kv) * case["hidden"]
        return {"bytes": n * (0.5 + 1 / 64 + 2), "flops": 2.0 * n}
    if kind == "head":
        n, wide = case["n"], 2.0 * case["n"] * HIDDEN * VOCAB
        return {"bytes": 2.0 * VOCAB * HIDDEN + 2.0 * n * HIDDEN * (2 if case["train"] else 1)
                + 24.0 * n, "flops": wide * (2 if case["train"] else 1)}
    lens = _lens(case)
    n = sum(lens)
    width = Q_DIM + 2 * KV_DIM
    if kind == "attn":
        # q, k, v -> out, lse; dout (q, k, v, out kept) -> dq, dk, dv
        f, b = _attn_flops(lens)
        return {"bytes": n * (2.0 * (4 * Q_DIM + 4 * KV_DIM) + 4 * HEADS), "flops": f + b}
    if kind == "lora":
        # x, qkv, positions -> q, k, v; dq, the partials of dk and dv -> dqkv, dx
        down = 2.0 * n * HIDDEN * 2 * RANK
        up = 2.0 * n * RANK * (Q_DIM + KV_DIM)
        return {"bytes": n * (2.0 * (2 * HIDDEN + 3 * width + Q_DIM) + 8 * Q_DIM + 8)
                + 8.0 * RANK * (2 * HIDDEN + Q_DIM + KV_DIM), "flops": 3 * (down + up)}
    L = case["layers"]
    f, b = _attn_flops(lens)
    # forward and input gradient of the frozen weights; the LoRA products are 3% beside them
    flops = L * (4.0 * n * LAYER_WEIGHTS + f + b + 6.0 * n * RANK * (2 * HIDDEN + Q_DIM + KV_DIM))
    byts = L * LAYER_WEIGHTS * (0.5 + 1 / 64) + 4.0 * n * HIDDEN
    byts += L * 4.0 * RANK * (2 * HIDDEN + Q_DIM + KV_DIM) * 2
    if kind == "step":
        flops += 4.0 * n * HIDDEN * VOCAB
        byts += 2.0 * VOCAB * HIDDEN
    return {"bytes": byts, "flops": flops}


def tolerance(case):
    """About four times the distance measured to the 64-bit results."""
    kind = case["kind"]
    if kind in ("norm", "glu") and case["dtype"] == "float32":
        return {"rel": 1e-5, "max": 1e-4}  # row sums in another order, exponentials
    if kind == "norm":  # two fp16 roundings of y: 3.7e-4
        return {"rel": 1.5e-3, "max": 0.02}
    if kind == "glu":  # one fp16 rounding: 2.1e-4
        return {"rel": 8e-4, "max": 0.01}
    if kind == "lora":  # products of rounded fp16 intermediates: 4.7e-4
        return {"rel": 2e-3, "max": 0.05}
    if kind == "attn":  # probabilities rounded to fp16 for their products: 3.2e-4
        return {"rel": 1.3e-3, "max": 0.05}
    if kind == "head":  # fp16 logits: 2.1e-4; of two equal maxima either may be the argmax
        return {"rel": 8e-4, "max": 0.05, "differ": 0.01}
    if kind == "dequant":  # each value is one rounding of one product
        return "exact"
    if kind == "stack":  # whole layers in fp16: 2.5e-3
        return {"rel": 0.01, "max": 0.5}
    # the unscaled loss leaves small fp16 gradients: 1.7e-2
    return {"rel": 0.03, "max": 0.9, "differ": 0.01}


# ---------------------------------------------------------------------------------------------
# The same in 64 bits, plain torch
# ---------------------------------------------------------------------------------------------

_PHILOX_M = (0xD2E7470EE14C6C93, 0xCA5A826395121157)
_PHILOX_W = (0x9E3779B97F4A7C15, 0xBB67AE8584CAA73B)


def _mulhilo(m, x):
    """High and low 64 bits of m * x for uint64 arrays x."""
    m0, m1 = np.uint64(m & 0xFFFFFFFF), np.uint64(m >> 32)
    x0, x1 = x & np.uint64(0xFFFFFFFF), x >> np.uint64(32)
    a, b, c = m0 * x0, m1 * x0, m0 * x1
    mid = (a >> np.uint64(32)) + (b & np.uint64(0xFFFFFFFF)) + (c & np.uint64(0xFFFFFFFF))
    hi = m1 * x1 + (b >> np.uint64(32)) + (c >> np.uint64(32)) + (mid >> np.uint64(32))
    return hi, np.uint64(m) * x


def _keep(seed, stream, n, d):
    """The documented dropout mask [n, d]: element e is kept when 32-bit word e % 8 of
    Philox4x64-10 at counter e // 8, key (seed, stream), is at least p 2^32."""
    c = [np.arange((n * d + 7) // 8, dtype=np.uint64)] + [np.zeros(1, np.uint64)] * 3
    k0, k1 = seed, stream
    with np.errstate(over="ignore"):
        for _ in range(10):
            hi0, lo0 = _mulhilo(_PHILOX_M[0], c[0])
            hi1, lo1 = _mulhilo(_PHILOX_M[1], c[2])
            c = [hi1 ^ c[1] ^ np.uint64(k0), lo1, hi0 ^ c[3] ^ np.uint64(k1), lo0]
            k0, k1 = (k0 + _PHILOX_W[0]) % 2**64, (k1 + _PHILOX_W[1]) % 2**64
    c = np.stack(np.broadcast_arrays(*c), 1)
    w = np.stack([c & np.uint64(0xFFFFFFFF), c >> np.uint64(32)], 2).reshape(-1)[: n * d]
    limit = np.uint64(int(float(np.float32(DROPOUT)) * 4294967296.0 + 0.5))
    return torch.from_numpy((w >= limit).reshape(n, d)).cuda()


def _drop(x, seed, stream):
    keep = _keep(seed, stream, *x.shape)
    return torch.where(keep, x / (1.0 - DROPOUT), torch.zeros((), dtype=x.dtype, device=x.device))


def _rms(x, w):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * w.double()


def _rotate(x, cos, sin):
    """NeoX rotary embedding of x [n, heads, 128]."""
    half = HEAD_DIM // 2
    turned = torch.cat([-x[..., half:], x[..., :half]], -1)
    return x * cos[:, None, :] + turned * sin[:, None, :]


def _tables(pos):
    inv = THETA ** (-torch.arange(0, HEAD_DIM, 2, device="cuda").double() / HEAD_DIM)
    a = pos.double()[:, None] * inv[None]
    a = torch.cat([a, a], -1)
    return a.cos(), a.sin()


def _attention(q, k, v, lens):
    """(out [n, heads, 128], lse [heads, n]) of causal attention within each row."""
    outs, lses, a = [], [], 0
    for n in lens:
        mask = torch.ones(n, n, dtype=torch.bool, device="cuda").tril()
        o, l = [], []
        for h in range(HEADS):
            g = h // (HEADS // KV_HEADS)
            s = q[a:a + n, h] @ k[a:a + n, g].t().contiguous() / math.sqrt(HEAD_DIM)
            s = s.masked_fill(~mask, -math.inf)
            l.append(torch.logsumexp(s, -1))
            o.append(torch.softmax(s, -1) @ v[a:a + n, g])
        outs.append(torch.stack(o, 1))
        lses.append(torch.stack(l, 0))
        a += n
    return torch.cat(outs, 0), torch.cat(lses, 1)


def _decode(w):
    """A quantised weight in 64 bits."""
    levels = torch.tensor(quant.NF4_LEVELS, dtype=torch.float64, device="cuda")
    scale = w.code2.double()[w.absmax.long()]
    scale = scale * w.absmax2.double().repeat_interleave(w.super_blocksize)[: scale.numel()]
    scale = (scale + w.offset).repeat_interleave(w.blocksize)
    p = w.packed.long()
    return (levels[torch.stack([p >> 4, p & 15], 1).reshape(-1)] * scale[: 2 * p.numel()]).view(w.shape)


def _layer(x, L, lens, cos, sin, seed, l):
    """One decoder layer with LoRA on q and v, dropout masks of streams 2 l and 2 l + 1."""
    n = x.shape[0]
    y = _rms(x, L.ln1)
    q = y @ _decode(L.q).t() + L.q_bias.double()
    k = y @ _decode(L.k).t() + L.k_bias.double()
    v = y @ _decode(L.v).t() + L.v_bias.double()
    q = q + SCALE * (_drop(y, seed, 2 * l) @ L.q_A.t()) @ L.q_B.t()
    v = v + SCALE * (_drop(y, seed, 2 * l + 1) @ L.v_A.t()) @ L.v_B.t()
    q = _rotate(q.view(n, HEADS, HEAD_DIM), cos, sin)
    k = _rotate(k.view(n, KV_HEADS, HEAD_DIM), cos, sin)
    o, _ = _attention(q, k, v.view(n, KV_HEADS, HEAD_DIM), lens)
    x = x + o.reshape(n, Q_DIM) @ _decode(L.o).t()
    y = _rms(x, L.ln2)
    act = F.silu(y @ _decode(L.gate).t()) * (y @ _decode(L.up).t())
    return x + act @ _decode(L.down).t()


def _exact_stack(m, h, lens, seed):
    """(final norm output, leaf LoRA factors) of the whole stack in 64 bits, under autograd."""
    cos, sin = _tables(_positions(lens))
    leaves = []
    x = h.double()
    for l, L in enumerate(m.layers):
        f = [p.detach().double().requires_grad_(True) for p in (L.q_A, L.q_B, L.v_A, L.v_B)]
        leaves += f
        L64 = model.LayerWeights(L.q, L.k, L.v, L.o, L.gate, L.up, L.down, L.q_bias, L.k_bias,
                                 L.v_bias, L.ln1, L.ln2, *f)
        x = _layer(x, L64, lens, cos, sin, seed, l)
    return _rms(x, m.final_norm), leaves


def _exact_head(h, w, labels):
    """(loss, nll, entropy) in 64 bits, token blocks at a time."""
    nll, ent = [], []
    wt = w.double().t().contiguous()
    for hb, lb in zip(h.split(256), labels.split(256)):
        z = hb @ wt
        lse = torch.logsumexp(z, -1)
        ent.append(lse - (torch.exp(z - lse[:, None]) * z).sum(-1))
        t = z.gather(1, lb.clamp(min=0)[:, None])[:, 0]
        nll.append(torch.where(lb == -100, torch.zeros_like(t), lse - t))
    nll, ent = torch.cat(nll), torch.cat(ent)
    return nll.sum() / max(1, int((labels != -100).sum())), nll, ent


def _exact_lora(case, seed):
    s = _lora_inputs(case, seed)
    cos16, sin16 = (t.double() for t in ops.rope_cache(MAX_POS, HEAD_DIM, THETA, "cuda"))
    cos, sin = cos16[s["pos"]], sin16[s["pos"]]
    n = s["x"].shape[0]
    x = s["x"].double().requires_grad_(True)
    qkv = s["qkv"].double().requires_grad_(True)
    f = {k: s[k].double().requires_grad_(True) for k in ("Aq", "Bq", "Av", "Bv")}
    q, k, v = qkv.split([Q_DIM, KV_DIM, KV_DIM], 1)
    q = q + SCALE * (_drop(x, MASK_SEED, 0) @ f["Aq"].t()) @ f["Bq"].t()
    v = v + SCALE * (_drop(x, MASK_SEED, 1) @ f["Av"].t()) @ f["Bv"].t()
    q = _rotate(q.view(n, HEADS, HEAD_DIM), cos, sin)
    k = _rotate(k.view(n, KV_HEADS, HEAD_DIM), cos, sin)
    v = v.view(n, KV_HEADS, HEAD_DIM)

    def group(t):
        return t.double().view(KV_HEADS, HEADS // KV_HEADS, n, HEAD_DIM).sum(1).transpose(0, 1)

    g = torch.autograd.grad((q, k, v), (qkv, x, f["Aq"], f["Bq"], f["Av"], f["Bv"]),
                            (s["dq"].double(), group(s["dk"]), group(s["dv"])))
    return [t.detach() for t in (q, k, v)] + list(g)


def exact(case, seed):
    kind = case["kind"]
    if kind == "norm":
        s = _norm_inputs(case, seed)
        h = (s["x"].double() + s["res"].double()).requires_grad_(True)
        y = _rms(h, s["weight"])
        (dx,) = torch.autograd.grad((y, h), h, (s["dy"].double(), s["dh"].double()))
        return [y.detach(), h.detach(), dx]
    if kind == "glu":
        s = _glu_inputs(case, seed)
        gu = s["gu"].double().requires_grad_(True)
        gate, up = gu.chunk(2, 1)
        out = F.silu(gate) * up
        (dgu,) = torch.autograd.grad(out, gu, s["dout"].double())
        return [out.detach(), dgu]
    if kind == "lora":
        return _exact_lora(case, seed)
    if kind == "attn":
        s = _attn_inputs(case, seed)
        q, k, v = (s[t].double().requires_grad_(True) for t in ("q", "k", "v"))
        out, lse = _attention(q, k, v, _lens(case))
        g = torch.autograd.grad(out, (q, k, v), s["dout"].double())
        return [out.detach(), lse.detach(), *g]
    if kind == "head":
        s = _head_inputs(case, seed)
        with torch.set_grad_enabled(False):
            loss, nll, ent = _exact_head(s["h"].double(), s["w"], s["labels"])
        if not case["train"]:
            return [loss, nll, ent, None]
        w = s["w"].double()
        wt, dh = w.t().contiguous(), []
        for hb, lb in zip(s["h"].double().split(256), s["labels"].split(256)):
            p = torch.softmax(hb @ wt, -1)
            p.scatter_add_(1, lb.clamp(min=0)[:, None], torch.full_like(hb[:, :1], -1.0))
            dh.append((p * (lb != -100)[:, None]) @ w)
        count = max(1, int((s["labels"] != -100).sum()))
        return [loss, nll, ent, None, torch.cat(dh) * (LOSS_SCALE / count)]
    if kind == "dequant":
        return [torch.cat([_decode(w) for w in group]) for group in _segments(case, seed)]
    lens = _lens(case)
    if kind == "stack":
        s = _stack_inputs(case, seed)
        final, leaves = _exact_stack(s["model"], s["h"], lens, MASK_SEED + 1)
        return [final.detach(), *torch.autograd.grad(final, leaves, s["d_final"].double())]
    s = _step_inputs(case, seed)
    ids = torch.cat([s["ids"][r, :n] for r, n in enumerate(lens)]).cuda()
    labels = torch.cat([torch.cat([s["labels"][r, 1:n], torch.tensor([-100])])
                        for r, n in enumerate(lens)]).cuda()
    final, leaves = _exact_stack(s["model"], s["model"].embed[ids], lens, MASK_SEED + 1)
    loss, nll, ent = _exact_head(final, s["model"].embed, labels)
    grads = torch.autograd.grad(loss, leaves)
    return [loss.detach(), nll.detach(), ent.detach(), None, *grads]
