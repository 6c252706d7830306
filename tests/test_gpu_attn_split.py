"""The attention's key ranges (hif8_attention_fwd_split): tiles of the last wave of workgroups
computed over ranges of the keys whose fp32 partials a second kernel adds.

Oracle and tolerance as for the unsplit kernel (test_gpu_attn_kernel.py): float64 softmax attention
over the kept keys, normwise 1e-2 and elementwise 2e-2 of the largest output; against the unsplit
kernel itself, whose bf16 probabilities and output are rounded at the same places, one bf16 step of the
largest output (2^-7).  The o state must be the one an amax pass over the output gives."""
from __future__ import annotations

import ctypes
import math

import pytest

torch = pytest.importorskip("torch")

DEV = "cuda:0"
D = 128


def reference(q, k, v, rows):
    out = torch.zeros(q.shape, dtype=torch.float64, device=q.device)
    for b in range(q.shape[0]):
        kb = b if k.shape[0] > 1 else 0
        if len(rows[b]) == 0:
            continue
        for h in range(q.shape[2]):
            kt = k[kb, rows[b], h].double().t().contiguous()
            p = torch.softmax(q[b, :, h].double() @ kt / math.sqrt(D), -1)
            out[b, :, h] = p @ v[kb, rows[b], h].double().contiguous()
    return out


def unsplit(pkg, q, k, v, idx, cnt, state=None):
    B, Nq, H, _ = q.shape
    out = torch.empty_like(q)
    I4 = ctypes.c_int64 * 4
    rs = I4(q.stride(1), k.stride(1), v.stride(1), out.stride(1))
    bs = I4(q.stride(0), k.stride(0) if k.shape[0] == B else 0, v.stride(0) if v.shape[0] == B else 0, out.stride(0))
    pkg._lib.check(pkg._lib.load().hif8_attention_fwd(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), B, Nq, k.shape[1], H, D, rs, bs,
        idx.data_ptr() if idx is not None else None, idx.stride(0) if idx is not None else 0,
        cnt.data_ptr() if cnt is not None else None, 1.0 / math.sqrt(D), state.ptr if state else None, 2, 15.0,
        pkg._lib.stream_ptr(q.device)), "hif8_attention_fwd")
    return out


# (B, Nq, Nkv, H, shared k/v, kept keys per batch or None).  Few tiles, one wave and a remainder;
# ragged queries and keys; lists whose counts leave some ranges short, empty, or without any key
CASES = [
    (1, 384, 640, 1, False, None),
    (1, 500, 1000, 2, False, None),
    (2, 300, 2050, 3, False, [2050, 130]),
    (4, 700, 1500, 2, False, [1500, 1, 0, 64]),
    (1, 97, 512, 5, True, None),
    (3, 400, 777, 2, True, [777, 300, 65]),
    (1, 384 * 130, 512, 2, False, None),
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("as_f32", [True, False])
def test_key_ranges(pkg, case, as_f32):
    B, Nq, Nkv, H, shared, kept = case
    print(f"[attn split] {case} as_f32={as_f32}", flush=True)
    assert pkg._lib.load().hif8_attention_workspace_bytes(B, Nq, Nkv, H) > 0
    g = torch.Generator().manual_seed(Nq + Nkv + H)
    kb = 1 if shared else B
    q = (torch.randn(B, Nq, H, D, generator=g) * 2).to(torch.bfloat16).to(DEV)
    k = (torch.randn(kb, Nkv, H, D, generator=g) * 2).to(torch.bfloat16).to(DEV)
    v = torch.randn(kb, Nkv, H, D, generator=g).to(torch.bfloat16).to(DEV)
    idx = cnt = None
    rows = [torch.arange(Nkv, device=DEV)] * B
    if kept is not None:
        mask = torch.zeros(B, Nkv, dtype=torch.bool)
        for b, n in enumerate(kept):
            mask[b, torch.randperm(Nkv, generator=g)[:n]] = True
        mask = mask.to(DEV)
        idx, cnt = pkg.key_list(mask)
        rows = [mask[b].nonzero().squeeze(-1) for b in range(B)]
    st = pkg.QuantState(DEV)
    out = pkg.attention_fwd(q, k, v, idx, cnt, o_state=st, o_as_f32=as_f32)
    again = pkg.attention_fwd(q, k, v, idx, cnt)
    whole = unsplit(pkg, q, k, v, idx, cnt)
    assert torch.equal(out.view(torch.int16), again.view(torch.int16))
    want = pkg.absmax_scale(out, 15.0, pkg.QuantState(DEV), as_f32)
    assert st.read() == want.read()
    top = float(whole.double().abs().max())
    assert float((out.double() - whole.double()).abs().max()) <= top * 2.0 ** -7
    if Nq <= 1000:
        ref = reference(q, k, v, rows)
        err = (out.double() - ref).abs()
        assert float(err.max()) <= 2e-2 * float(ref.abs().max())
        assert float(err.norm()) <= 1e-2 * float(ref.norm())


@pytest.mark.gpu
def test_key_ranges_nan(pkg):
    """A NaN query row gives NaN outputs in its own rows alone."""
    q, k, v = (torch.randn(1, 400, 1, D, device=DEV).to(torch.bfloat16) for _ in range(3))
    q[0, 33] = float("nan")
    assert pkg._lib.load().hif8_attention_workspace_bytes(1, 400, 400, 1) > 0
    out = pkg.attention_fwd(q, k, v)
    bad = torch.isnan(out.float()).any(-1).squeeze()
    assert bad[33] and int(bad.sum()) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("split", [True, False])
def test_infinite_scores(pkg, split):
    """Keys of score -inf add nothing beside finite ones, also where they fill whole key tiles or a whole
    key range; where all of a query's keys score -inf its output is NaN (float64 softmax's), and so is the
    o state's amax; without keys it is zero."""
    B, Nq, Nkv, H = 2, 300, 1200, 2
    assert pkg._lib.load().hif8_attention_workspace_bytes(B, Nq, Nkv, H) > 0
    g = torch.Generator().manual_seed(5)
    q, k, v = (torch.randn(B, n, H, D, generator=g).to(torch.bfloat16).to(DEV) for n in (Nq, Nkv, Nkv))
    q[..., 7] = q[..., 7].abs() + 0.25
    rows = [torch.arange(Nkv, device=DEV)] * B

    def run(k, cnt=None):
        st = pkg.QuantState(DEV)
        out = (pkg.attention_fwd(q, k, v, None, cnt, o_state=st, o_as_f32=True) if split
               else unsplit(pkg, q, k, v, None, cnt, st))
        assert st.read()[0] == pkg.absmax_scale(out, 15.0, pkg.QuantState(DEV), True).read()[0]
        return out
    some = k.clone()
    some[0, :700, :, 7] = float("-inf")           # the first tiles and ranges of batch 0
    some[1, 640:704, :, 7] = float("-inf")        # one key tile of batch 1
    ref = reference(q, some, v, rows)
    err = (run(some).double() - ref).abs()
    assert float(err.max()) <= 2e-2 * float(ref.abs().max()) and float(err.norm()) <= 1e-2 * float(ref.norm())
    every = k.clone()
    every[1, :, :, 7] = float("-inf")
    out = run(every)
    assert bool(torch.isnan(reference(q, every, v, rows)[1]).all())
    assert bool(torch.isnan(out[1]).all()) and bool(torch.isfinite(out[0]).all())
    cnt = torch.tensor([0, 5], dtype=torch.int32, device=DEV)
    out = run(every, cnt)
    assert bool((out[0] == 0).all()) and bool(torch.isnan(out[1]).all())


def test_attention_plan_on_256_cus(pkg):
    """hif8_attention_workspace_bytes as planned for 256 CUs (assumed without a GPU)."""
    L = pkg._lib.load()
    part = (384 * 128 + 2 * 384) * 4
    assert L.hif8_attention_workspace_bytes(1, 32760, 32760, 12) == 8 * 32 * part     # 1032 tiles
    assert L.hif8_attention_workspace_bytes(1, 384 * 256, 512, 1) == 0                # one whole wave
    assert L.hif8_attention_workspace_bytes(1, 384, 64, 1) == 0                       # one key tile
    assert L.hif8_attention_workspace_bytes(1, 84672, 84672, 40) == 0                 # 34 waves
    assert L.hif8_attention_workspace_bytes(0, 1, 1, 1) == 0
    for tiles in (1, 8, 60, 130, 250, 300, 1032):
        for nt in (2, 8, 31, 137, 512):
            b = L.hif8_attention_workspace_bytes(1, 384 * tiles, 64 * nt, 1)
            tail = tiles % 256
            assert b % (tail * part) == 0
            sp = b // (tail * part)
            assert sp == 0 or (2 <= sp <= nt // 2 and sp * tail <= 768)
