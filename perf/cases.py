"""Workloads of the HiF8 linear path as programs run it, for timing and for comparing results.

Each case is one call (or one short chain of calls) through the package's public entry points at
sizes of the Wan 1.3B and 14B DiT or generic ones: ``HIF8Linear`` inference from a few dozen rows to
the 75600 tokens of a 14B 720P video, its training step in bf16 and with an fp32 input, ``HIF8FFN``,
the q/k/v projections behind the modulated norm, the attention with the statistic it leaves for the
``o`` projection, the codec, and one whole DiT block.

``listed()`` gives the fixed cases, ``draw(rng)`` more of the same ranges, ``prepare`` what a program
holds before the call, ``run`` one call, ``exact`` the same outputs in float64 by plain torch.
"""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from __graft_entry__ import load_package

DEV = "cuda:0"
FORWARD_MAX, BACKWARD_MAX = 15.0, 224.0
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32, "f16": torch.float16}
SIZES = {"bf16": 2, "f32": 4, "f16": 2}

# The largest drawn call: the 14B FFN up-projection at 720P (2 * 75600 * 5120 * 13824).
MAX_FLOPS = 1.08e13


# ------------------------------------------------------------------------------------- cases


def listed():
    return [
        # a handful of tokens through the 1.3B model's q projection: launches and latency
        dict(name="linear_few_rows_1p3b", kind="linear", rows=64, k=1536, n=1536, x="bf16"),
        # the cross-attention's k (or v) of the 512 text tokens, 14B
        dict(name="linear_text_kv_14b", kind="linear", rows=512, k=5120, n=5120, x="bf16"),
        # FFN down-projection of a short, ragged 480P clip (3 latent frames of 30 x 52), 1.3B
        dict(name="linear_down_short_1p3b", kind="linear", rows=4680, k=8960, n=1536, x="bf16"),
        # the largest linear: 14B FFN up-projection of a 720P video (21 x 45 x 80 tokens)
        dict(name="linear_up_14b_720p", kind="linear", rows=75600, k=5120, n=13824, x="bf16"),
        # the feed-forward network of the 1.3B block on a 480P video (21 x 30 x 52 tokens)
        dict(name="ffn_1p3b_480p", kind="ffn", rows=32760, k=1536, n=8960),
        # modulated LayerNorm and the three projections behind it, same video
        dict(name="qkv_norm_1p3b_480p", kind="qkv", rows=32760, k=1536),
        # full self-attention of that video, with the o projection's statistic
        dict(name="attention_1p3b_480p", kind="attention", batch=1, queries=32760, keys=32760, kept=32760, heads=12,
             shared=False),
        # Skiparse self-attention of a 14B block at 480P: 4 sub-sequences with padding keys masked
        dict(name="attention_skiparse_14b_480p", kind="attention", batch=4, queries=8736, keys=8736, kept=8190,
             heads=40, shared=False),
        # training step of the FFN up-projection: the parameter rewritten, forward and backward
        dict(name="train_up_1p3b_480p", kind="train", rows=32760, k=1536, n=8960, x="bf16", w="bf16"),
        # training step of the self-attention's o projection, whose input is fp32
        dict(name="train_o_f32_1p3b_480p", kind="train", rows=32760, k=1536, n=1536, x="f32", w="bf16"),
        # _quant of a 4096-token activation
        dict(name="quant_4096x5120", kind="codec", op="quant", rows=4096, k=5120, x="bf16", torch_route=False),
        # one 1.3B block at 480P on the way from the full to the Skiparse layout, Q/K/V quantised
        dict(name="block_1p3b_480p", kind="block", dim=1536, ffn=8960, heads=12, t=21, h=30, w=52, layout="token",
             quant_attn=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _features(rng):
    """(in, out) features: the models' projections, or generic ones (some outside every tile)."""
    if rng.random() < 0.6:
        return rng.choice([(1536, 1536), (1536, 8960), (8960, 1536), (5120, 5120), (5120, 13824), (13824, 5120)])
    k, n = _log_int(rng, 256, 6144), _log_int(rng, 256, 6144)
    if rng.random() < 0.75:
        k, n = max(64, k // 64 * 64), max(8, n // 8 * 8)
    return k, n


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "ffn", "qkv", "attention", "attention", "train", "train", "codec",
                       "block"])
    if kind == "linear":
        k, n = _features(rng)
        rows = _log_int(rng, 16, min(75600, int(MAX_FLOPS / (2 * k * n))))
        return dict(kind=kind, rows=rows, k=k, n=n, x=rng.choice(["bf16", "bf16", "bf16", "f32"]))
    if kind == "ffn":
        k, n = rng.choice([(1536, 8960), (5120, 13824), (1024, 4096), (768, 3072)])
        return dict(kind=kind, rows=_log_int(rng, 64, min(32760, int(MAX_FLOPS / (4 * k * n)))), k=k, n=n)
    if kind == "qkv":
        k = rng.choice([1536, 5120, 1024, 2048])
        return dict(kind=kind, rows=_log_int(rng, 64, min(75600, int(MAX_FLOPS / (6 * k * k)))), k=k)
    if kind == "attention":
        heads = rng.choice([12, 40, 8, 16])
        if rng.random() < 0.3:    # cross-attention: one text for every sub-sequence
            return dict(kind=kind, batch=1, queries=_log_int(rng, 256, 80640), keys=512, kept=512, heads=heads,
                        shared=True)
        batch = rng.choice([1, 4])
        top = int(math.sqrt(0.5 * MAX_FLOPS / (4 * batch * heads * 128)))
        queries = _log_int(rng, 256, min(32760, top))
        kept = queries if rng.random() < 0.5 else int(queries * rng.uniform(0.85, 0.99))
        return dict(kind=kind, batch=batch, queries=queries, keys=queries, kept=kept, heads=heads, shared=False)
    if kind == "train":
        k, n = rng.choice([(1536, 1536), (1536, 8960), (8960, 1536), (5120, 5120), (1024, 1024), (1000, 1304)])
        x, w = rng.choice([("bf16", "bf16"), ("bf16", "bf16"), ("f32", "bf16"), ("f32", "f32"), ("bf16", "f32")])
        cost = 32760 * 1536 * 1536 if "f32" in (x, w) else 32760 * 1536 * 8960
        return dict(kind=kind, rows=_log_int(rng, 256, min(32760, max(257, cost // (k * n)))), k=k, n=n, x=x, w=w)
    if kind == "codec":
        op = rng.choice(["quant", "qdq"])
        x = rng.choice(["bf16", "f32"] if op == "quant" else ["bf16", "f32", "f16"])
        return dict(kind=kind, op=op, rows=_log_int(rng, 16, 32760), k=rng.choice([1536, 5120, 4096, 1001, 333]), x=x,
                    torch_route=op == "qdq" and rng.random() < 0.5)
    t, h, w = rng.randint(1, 13), rng.randint(8, 32), rng.randint(8, 52)
    return dict(kind=kind, dim=1536, ffn=8960, heads=12, t=t, h=h, w=w, layout=rng.choice(["full", "token"]),
                quant_attn=rng.random() < 0.5)


# ------------------------------------------------------------------------------------ inputs


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _activation(g, rows, k, dtype):
    """Unit activations with a few outlier channels, as a transformer's residual stream has them."""
    x = _randn(g, rows, k)
    x[:, torch.randint(0, k, (min(16, k),), generator=g, device=DEV)] *= 20
    return x.to(DTYPES[dtype])


def _layer(pkg, g, k, n, dtype=torch.bfloat16):
    lin = pkg.HIF8Linear(k, n, bias=True, device=DEV, dtype=dtype)
    with torch.no_grad():
        lin.weight.copy_(_randn(g, n, k) * 0.02)
        lin.bias.copy_(_randn(g, n) * 0.1)
    return lin


def _grid_tokens(case):
    """(sub-sequences, tokens of each) of a block's attention, padding included."""
    if case["layout"] == "full":
        return 1, case["t"] * case["h"] * case["w"]
    hp, wp = -(-case["h"] // 4) * 4, -(-case["w"] // 4) * 4
    return 4, case["t"] * hp * wp // 4


def prepare(case, seed):
    pkg = load_package()
    g = _gen(seed)
    kind = case["kind"]
    s = dict(case=case, pkg=pkg)
    if kind == "linear":
        s["x"] = _activation(g, case["rows"], case["k"], case["x"])
        s["lin"] = _layer(pkg, g, case["k"], case["n"]).prepack()
    elif kind == "ffn":
        s["x"] = _activation(g, case["rows"], case["k"], "bf16")
        ffn = pkg.HIF8FFN(case["k"], case["n"], device=DEV, dtype=torch.bfloat16)
        with torch.no_grad():
            for lin in (ffn[0], ffn[2]):
                lin.weight.copy_(_randn(g, *lin.weight.shape) * 0.02)
                lin.bias.copy_(_randn(g, *lin.bias.shape) * 0.1)
                lin.prepack()
        s["ffn"] = ffn
    elif kind == "qkv":
        k = case["k"]
        s["x"] = _activation(g, case["rows"], k, "bf16").view(1, case["rows"], k)
        s["shift"], s["scale"] = ((_randn(g, 1, 1, k) * 0.5).to(torch.bfloat16) for _ in range(2))
        s["layers"] = [_layer(pkg, g, k, k).prepack() for _ in range(3)]
    elif kind == "attention":
        b, h = case["batch"], case["heads"]
        kb = 1 if case["shared"] else b
        s["q"] = _randn(g, b, case["queries"], h, 128).to(torch.bfloat16)
        s["k"] = _randn(g, kb, case["keys"], h, 128).to(torch.bfloat16)
        s["v"] = _randn(g, kb, case["keys"], h, 128).to(torch.bfloat16)
        s["idx"] = s["cnt"] = None
        if case["kept"] < case["keys"]:
            mask = torch.zeros(b, case["keys"], dtype=torch.bool, device=DEV)
            for i in range(b):
                mask[i, torch.randperm(case["keys"], generator=g, device=DEV)[:case["kept"]]] = True
            s["mask"] = mask
            s["idx"], s["cnt"] = pkg.key_list(mask)
    elif kind == "train":
        dtype = DTYPES[case["w"]]
        s["lin"] = _layer(pkg, g, case["k"], case["n"], dtype)
        s["master"] = s["lin"].weight.detach().float().clone()
        s["x"] = _activation(g, case["rows"], case["k"], case["x"]).requires_grad_(True)
        s["gy"] = (_randn(g, case["rows"], case["n"]) * 1e-3).to(torch.bfloat16)
    elif kind == "codec":
        s["x"] = _activation(g, case["rows"], case["k"], case["x"])
        s["qtype"] = pkg.QType("hif8")
    else:
        dit = pkg.dit
        grid = (case["t"], case["h"], case["w"])
        token = case["layout"] == "token"
        blk = dit.OSPNextAttentionBlock(
            case["dim"], case["ffn"], case["heads"], cross_attn_norm=True, sparse_ratio=2 if token else 1,
            skiparse_block_type=case["layout"], is_full2skiparse_block=token, quant="hif8",
            quant_attn="hif8" if case["quant_attn"] else None, device=DEV, dtype=torch.bfloat16)
        with torch.no_grad():
            for m in blk.modules():
                if isinstance(m, pkg.HIF8Linear):
                    m.weight.copy_(_randn(g, *m.weight.shape) * 0.02)
                    m.bias.copy_(_randn(g, *m.bias.shape) * 0.1)
                    m.prepack()
            blk.modulation.copy_(_randn(g, *blk.modulation.shape) / case["dim"] ** 0.5)
        s["block"], s["grid"] = blk, grid
        s["mask"] = dit.skiparse_masks(1, grid, 2, DEV)[0] if token else None
        s["x"] = _activation(g, grid[0] * grid[1] * grid[2], case["dim"], "bf16").unsqueeze(0)
        s["e"] = _randn(g, 1, 6, case["dim"]).to(torch.bfloat16)
        s["text"] = _randn(g, 1, 512, case["dim"]).to(torch.bfloat16)
        s["rope"] = dit.SkiparseRopeWrapper(dit.rope_freqs(128).to(DEV))
    return s


# -------------------------------------------------------------------------------------- calls


def run(s):
    case, pkg = s["case"], s["pkg"]
    kind = case["kind"]
    if kind == "train":
        lin = s["lin"]
        with torch.no_grad():    # the optimiser's fp32 weights into the layer's parameter, once a step
            lin.weight.copy_(s["master"])
        y = lin(s["x"])
        return (y.detach(), *torch.autograd.grad(y, (s["x"], lin.weight, lin.bias), s["gy"]))
    with torch.no_grad():
        if kind == "linear":
            return s["lin"](s["x"])
        if kind == "ffn":
            return s["ffn"](s["x"])
        if kind == "qkv":
            return pkg.qkv_from_modulated_norm(s["x"], s["shift"], s["scale"], *s["layers"])
        if kind == "attention":
            st = pkg.QuantState(s["q"].device)
            out = pkg.attention_fwd(s["q"], s["k"], s["v"], s["idx"], s["cnt"], o_state=st, o_as_f32=True,
                                    scale_max=FORWARD_MAX)
            return out, st.scale()
        if kind == "codec":
            if case["op"] == "quant":
                return pkg._quant(s["x"], FORWARD_MAX)
            return pkg.quant_dequant_float(s["x"], s["qtype"], force_py=case["torch_route"])
        return s["block"](s["x"], s["mask"], s["mask"], s["e"], s["grid"], s["grid"], s["rope"], s["text"])


# --------------------------------------------------------------------------------- accounting


def _linear_work(rows, k, n, xbytes):
    return dict(bytes=rows * k * xbytes + n * k + 2 * n + 2 * rows * n, flops=2 * rows * k * n)


def work(case):
    kind = case["kind"]
    if kind == "linear":
        return _linear_work(case["rows"], case["k"], case["n"], SIZES[case["x"]])
    if kind == "ffn":
        m, k, n = case["rows"], case["k"], case["n"]
        return dict(bytes=4 * m * k + 2 * k * n + 2 * (k + n), flops=4 * m * k * n)
    if kind == "qkv":
        m, k = case["rows"], case["k"]
        return dict(bytes=8 * m * k + 3 * k * k + 10 * k, flops=6 * m * k * k)
    if kind == "attention":
        b, h = case["batch"], case["heads"]
        kv = (1 if case["shared"] else b) * case["kept"]
        return dict(bytes=4 * 128 * h * (b * case["queries"] + kv),
                    flops=4 * 128 * h * b * case["queries"] * case["kept"])
    if kind == "train":
        m, k, n = case["rows"], case["k"], case["n"]
        xb, wb = SIZES[case["x"]], SIZES[case["w"]]
        return dict(bytes=2 * m * k * xb + 4 * m * n + n * k * (4 + wb) + n * 2 * wb, flops=6 * m * k * n)
    if kind == "codec":
        n = case["rows"] * case["k"]
        return dict(bytes=2 * n * SIZES[case["x"]], flops=2 * n)
    b, n = _grid_tokens(case)
    d, f = case["dim"], case["ffn"]
    m, real = b * n, case["t"] * case["h"] * case["w"]
    kept = real // b
    flops = 2 * m * (6 * d * d + 2 * d * f) + 2 * 512 * 2 * d * d + 4 * m * d * (kept + 512)
    return dict(bytes=2 * d * (real + m + 512) + 8 * d * d + 2 * d * f, flops=flops)


def tolerance(case):
    kind = case["kind"]
    if kind == "codec":
        return "exact"          # whole HiF8 values: every implementation gives the same bits
    if kind == "block":
        # bf16 roundings ahead of a quantised linear move some HiF8 values by a step
        return dict(rel=5e-2)
    if kind == "attention":
        return dict(rel=9e-3)   # bf16 probabilities and output: 2.3e-3 from float64
    # bf16 output of an fp32 sum over equal operands: 1.7e-3 from float64, also behind the one
    # rounding that ffn and qkv have ahead of a quantised linear
    return dict(rel=7e-3)


# ------------------------------------------------------------------------- float64 restatement


def _hif8(x):
    """HiF8 rounding of finite fp32 values (half away from zero on the tapered grid)."""
    a = x.abs()
    e = (torch.frexp(a)[1] - 1).clamp(min=-23)
    ae = e.abs()
    bits = (ae <= 3).int() + (ae <= 7).int() + (ae <= 15).int()
    step = torch.ldexp(torch.ones_like(a), (e.clamp(min=-22) - bits))
    q = torch.floor(a / step + 0.5) * step
    q = torch.where(a < 2.0 ** -23, torch.zeros_like(q), q)
    q = torch.where(a >= 40960.0, torch.full_like(q, float("inf")), q)
    return torch.copysign(q, x) * (q != 0)


def _fake_quant(x, scale_max):
    """x_q and scale, each operation rounded to x's dtype."""
    amax = x.abs().amax().clamp(min=1e-8)
    scale = amax.reciprocal() * scale_max
    q = _hif8((x * scale).float()).to(x.dtype)
    return q / scale, scale


def _dot(x_q, w_q, bias):
    return x_q.to(torch.bfloat16).double() @ w_q.to(torch.bfloat16).double().t().contiguous() + bias.double()


def _quant_weight(lin):
    return _fake_quant(lin.weight.detach(), FORWARD_MAX)[0]


def _norm_modulate(x, shift, scale):
    xd = x.double()
    mean = xd.mean(-1, keepdim=True)
    n = ((xd - mean) * (xd.var(-1, unbiased=False, keepdim=True) + 1e-6).rsqrt()).to(torch.bfloat16)
    return n * (1 + scale) + shift


def _attention64(q, k, v, mask):
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    for b in range(q.shape[0]):
        kb = b if k.shape[0] > 1 else 0
        rows = mask[b].nonzero().squeeze(-1) if mask is not None else slice(None)
        for h in range(q.shape[2]):
            kt = k[kb, rows, h].double().t().contiguous()
            vh = v[kb, rows, h].double().contiguous()
            for i in range(0, q.shape[1], 8192):
                p = torch.softmax(q[b, i:i + 8192, h].double() @ kt / math.sqrt(128.0), dim=-1)
                out[b, i:i + 8192, h] = p @ vh
    return out


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind == "block":
        # bf16 roundings between its layers decide HiF8 values: no float64 chain is its limit
        return None
    if kind == "codec" and case["torch_route"]:
        return None    # that route is defined by the roundings of its own low-precision steps
    s = prepare(case, seed)
    if kind == "linear":
        lin = s["lin"]
        return _dot(_fake_quant(s["x"], FORWARD_MAX)[0], _quant_weight(lin), lin.bias)
    if kind == "ffn":
        up, down = s["ffn"][0], s["ffn"][2]
        y = _dot(_fake_quant(s["x"], FORWARD_MAX)[0], _quant_weight(up), up.bias).to(torch.bfloat16)
        h = F.gelu(y.double(), approximate="tanh").to(torch.bfloat16)
        return _dot(_fake_quant(h, FORWARD_MAX)[0], _quant_weight(down), down.bias)
    if kind == "qkv":
        y_q = _fake_quant(_norm_modulate(s["x"], s["shift"], s["scale"]), FORWARD_MAX)[0]
        return tuple(_dot(y_q, _quant_weight(lin), lin.bias) for lin in s["layers"])
    if kind == "attention":
        out = _attention64(s["q"], s["k"], s["v"], s.get("mask"))
        return out, FORWARD_MAX / out.abs().max()
    if kind == "train":
        lin, x = s["lin"], s["x"].detach()
        x_q, w_q, g_q = _fake_quant(x, FORWARD_MAX)[0], _quant_weight(lin), _fake_quant(s["gy"], BACKWARD_MAX)[0]
        g = g_q.double()
        return (_dot(x_q, w_q, lin.bias.to(torch.bfloat16)), g @ w_q.double(), g.t().contiguous() @ x_q.double(),
                g.sum(0))
    if case["op"] == "quant":
        return _fake_quant(s["x"], FORWARD_MAX)
    return _hif8(s["x"].float()).to(s["x"].dtype)
