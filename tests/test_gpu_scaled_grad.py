"""The backward's products with an fp32-held operand on the MFMA GEMM (hif8_linear_wgrad_scaled,
hif8_linear_fwd_scaled): grad_q^T @ x_q of an fp32 x and grad_q @ w_q of an fp32 weight
(hif8_linear.py:97,104), and the k-range plan of small grids.

Oracle: the float64 product of the same quantised operands.  The kernel's products are exact in fp32
and their sums are rounded in fp32, so each output lies within a few fp32 steps of sum |g||x| (2^-20
of it here, 16 steps), plus 2^-8 of itself for a bf16 output."""
from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")

DEV = "cuda:0"


def quantised(pkg, M, N, K, seed):
    g = torch.Generator().manual_seed(seed)
    gq, _ = pkg._quant(torch.randn(M, N, generator=g).to(torch.bfloat16).to(DEV), 224.0)
    x = torch.randn(M, K, generator=g)
    x[:, : max(1, K // 64)] *= 20
    x = x.to(DEV)
    st = pkg.absmax_scale(x, 15.0, pkg.QuantState(DEV))
    return gq, pkg.encode(x, st), st


def bound(got, a, b, out_dtype):
    """got against a @ b in float64."""
    ref = a.double() @ b.double()
    tol = (a.double().abs() @ b.double().abs()) * 2.0 ** -20
    if out_dtype == torch.bfloat16:
        tol = tol + ref.abs() * 2.0 ** -8
    assert got.dtype == out_dtype and got.shape == ref.shape
    err = (got.double() - ref).abs()
    assert bool((err <= tol).all()), float((err / tol).max())
    return float(err.norm() / ref.norm())


# one and two k-steps, a ragged last one; a single column and tile edges; 36 tiles split 2 and 4
# ways; features outside multiples of 8
SHAPES = [(1, 8, 8), (64, 256, 256), (65, 264, 8), (300, 320, 264), (1000, 1536, 1536), (2100, 1536, 1536),
          (257, 100, 36), (4100, 520, 1032)]


@pytest.mark.gpu
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_wgrad_scaled(pkg, M, N, K, out_dtype):
    print(f"[scaled] wgrad M={M} N={N} K={K} {out_dtype}", flush=True)
    gq, codes, st = quantised(pkg, M, N, K, M + N + K)
    x_q = pkg.decode(codes, st, torch.float32)
    got = pkg.hif8_linear.linear_wgrad_scaled(gq, codes, st, out_dtype)
    rel = bound(got, gq.t().contiguous(), x_q, out_dtype)
    if out_dtype == torch.float32:
        fma = pkg.gemm_f32(gq, x_q, N, K, M, (1, N), (K, 1))
        ref = gq.double().t() @ x_q.double()
        old = float((fma.double() - ref).norm() / ref.norm())
        print(f"[scaled] relative error {rel:.2e}, fp32 FMA kernel {old:.2e}", flush=True)
        assert rel <= 1.5 * old + 2.0 ** -24


@pytest.mark.gpu
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [(1, 64, 8), (64, 64, 256), (300, 100, 36), (257, 320, 264), (1100, 1536, 1536),
                                   (513, 8960, 776)])
def test_dgrad_scaled(pkg, M, N, K, out_dtype):
    print(f"[scaled] dgrad M={M} N={N} K={K} {out_dtype}", flush=True)
    g = torch.Generator().manual_seed(M + N + K)
    gq, _ = pkg._quant(torch.randn(M, N, generator=g).to(torch.bfloat16).to(DEV), 224.0)
    packed = pkg.PackedWeight((torch.randn(N, K, generator=g) * 0.02).to(DEV), 15.0)
    got = pkg.hif8_linear.linear_dgrad_scaled(gq, packed, out_dtype)
    bound(got, gq, packed.dequantize(torch.float32), out_dtype)


# the decode-once route (8192 rows, 24576 where N <= 2048) and the fused one just below it, on its 256 x 256
# tile and on each small one; ragged rows, padded features and reductions
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(8192, 2112, 40), (8200, 2304, 264), (24600, 64, 8), (8193, 2100, 36),
                                   (8192, 2112, 2304), (8191, 2112, 40), (8191, 2112, 2304), (24575, 64, 8),
                                   (4097, 320, 8960), (1, 64, 8), (33, 192, 40), (65, 384, 1544), (300, 256, 2568),
                                   (1000, 1600, 1536), (257, 100, 36)])
def test_dgrad_fp32_output(pkg, M, N, K):
    """The gradient of an fp32 input with a bf16 weight: fp32, unrounded, whatever the route."""
    print(f"[scaled] dgrad fp32 M={M} N={N} K={K}", flush=True)
    g = torch.Generator().manual_seed(M + N + K)
    gq, _ = pkg._quant(torch.randn(M, N, generator=g).to(torch.bfloat16).to(DEV), 224.0)
    packed = pkg.PackedWeight((torch.randn(N, K, generator=g) * 0.02).to(torch.bfloat16).to(DEV), 15.0)
    y = pkg.linear_dgrad(gq, packed, torch.float32)
    bound(y, gq, packed.dequantize(torch.bfloat16), torch.float32)
    if not pkg.hif8_linear.decode_once(M, -(-N // 64) * 64):
        # the bf16 output is these sums rounded
        assert torch.equal(y.to(torch.bfloat16), pkg.linear_dgrad(gq, packed))


@pytest.mark.gpu
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_wgrad_scaled_non_finite_input(pkg, value):
    """An Inf or NaN in x makes the scale 0 or NaN and every quotient non-finite: outputs are NaN or
    Inf where the product of the decoded operands is."""
    gq, _, _ = quantised(pkg, 130, 64, 64, 3)
    x = torch.randn(130, 64, device=DEV)
    x[5, 7] = value
    st = pkg.absmax_scale(x, 15.0, pkg.QuantState(DEV))
    codes = pkg.encode(x, st)
    got = pkg.hif8_linear.linear_wgrad_scaled(gq, codes, st, torch.float32)
    want = pkg.gemm_f32(gq, pkg.decode(codes, st, torch.float32), 64, 64, 130, (1, 64), (64, 1))
    assert not torch.isfinite(want).any()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    same = torch.isnan(want) | (got == want)
    assert bool(same.all())


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(130, 64, 64), (2100, 1536, 1536)])   # whole tiles, k ranges
def test_scale_with_overflowing_reciprocal(pkg, M, N, K):
    """An fp32 operand of amax 1e38 under a scale_max of 0.1 has a scale of 1e-39, whose reciprocal is
    infinite: the quotients, zero sums among them, are those of the decoded operand."""
    gen = torch.Generator().manual_seed(M)
    gq = (torch.randn(M, N, generator=gen) * 2.0 ** -10).to(torch.bfloat16).to(DEV)
    x = torch.randn(M, K, generator=gen).clamp(-3, 3) * 2e37
    x[:, 3] = 0
    x[5, 7] = 1e38
    x = x.to(DEV)
    st = pkg.absmax_scale(x, 0.1, pkg.QuantState(DEV))
    assert 0 < st.read()[1] < 2.0 ** -128
    codes = pkg.encode(x, st)
    for out_dtype in (torch.float32, torch.bfloat16):
        got = pkg.hif8_linear.linear_wgrad_scaled(gq, codes, st, out_dtype)
        bound(got, gq.t().contiguous(), pkg.decode(codes, st, torch.float32), out_dtype)
        assert bool((got[:, 3] == 0).all())
    packed = pkg.PackedWeight(x[:N].contiguous(), 0.1)
    g = gq[:, :packed.shape[0]].contiguous()
    if packed.shape[0] % 64 == 0:
        bound(pkg.hif8_linear.linear_dgrad_scaled(g, packed, torch.float32), g, packed.dequantize(torch.float32),
              torch.float32)


@pytest.mark.gpu
def test_wgrad_small_grid_split(pkg):
    """36 tiles over 4100 tokens run as k ranges: bounded against float64, equal to the transposed
    route bit for bit, and the same on a second call."""
    M, N, K = 4100, 1536, 1536
    assert pkg._lib.load().hif8_linear_ksplit_workspace_bytes(N, K, M) > 0
    gq, codes, st = quantised(pkg, M, N, K, 7)
    xq = pkg.decode(codes, st, torch.bfloat16)
    got = pkg.linear_wgrad(gq, xq)
    bound(got, gq.t().contiguous(), xq, torch.bfloat16)
    for other in (pkg.linear_wgrad(gq, xq), pkg.linear_wgrad(gq, xq, transposed=True)):
        assert torch.equal(got.view(torch.int16), other.view(torch.int16))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1536, 1536, 4160), (4352, 4096, 1088)])   # 36 tiles; 272: 16 split 2 ways
def test_workspace_size_does_not_choose_the_sum_order(pkg, M, N, K):
    """hif8_linear_fwd_wq_split and hif8_linear_wgrad split as hif8_linear_split_workspace_bytes says,
    however much more a caller's workspace holds: the bits of the exact size (of no workspace where that
    is 0)."""
    L, s = pkg._lib.load(), pkg._lib.stream_ptr(torch.device(DEV))
    g = torch.Generator().manual_seed(M)
    a, b = (torch.randn(n, K, generator=g).to(torch.bfloat16).to(DEV) for n in (M, N))
    at, bt = a.t().contiguous(), b.t().contiguous()
    need, wide = L.hif8_linear_split_workspace_bytes(M, N, K), L.hif8_linear_ksplit_workspace_bytes(M, N, K)
    assert max(need, wide) > 0
    ws = torch.empty(max(need, wide) + (1 << 20), dtype=torch.uint8, device=DEV)
    for fn in (lambda y, p, n: L.hif8_linear_fwd_wq_split(a.data_ptr(), b.data_ptr(), None, y.data_ptr(), M, N, K, p, n, s),
               lambda y, p, n: L.hif8_linear_wgrad(at.data_ptr(), bt.data_ptr(), y.data_ptr(), K, M, N, p, n, s)):
        exact, large = (torch.empty(M, N, dtype=torch.bfloat16, device=DEV) for _ in range(2))
        assert fn(exact, ws.data_ptr() if need else None, need) == 0
        assert fn(large, ws.data_ptr(), ws.numel()) == 0
        assert torch.equal(exact.view(torch.int16), large.view(torch.int16))


def test_ksplit_plan_on_256_cus(pkg):
    """hif8_linear_ksplit_workspace_bytes as planned for 256 CUs (assumed without a GPU): the tails of
    the split-tail plan as they are there, small grids in ranges of at least 8 k-steps, nothing where
    the CUs are busy or the reduction is short; never an empty range."""
    L = pkg._lib.load()
    tile = 256 * 256 * 4
    assert L.hif8_linear_ksplit_workspace_bytes(13824, 5120, 75600) == 56 * 4 * tile
    assert L.hif8_linear_ksplit_workspace_bytes(4096, 4096, 75648) == 0
    assert L.hif8_linear_ksplit_workspace_bytes(75600, 5120, 13824) == 0
    assert L.hif8_linear_ksplit_workspace_bytes(1536, 1536, 32760) == 36 * 7 * tile
    assert L.hif8_linear_ksplit_workspace_bytes(1536, 1536, 960) == 0          # 15 k-steps
    assert L.hif8_linear_ksplit_workspace_bytes(0, 256, 512) == 0
    for tiles in (1, 5, 36, 100, 200, 255, 400, 700):
        for nk in (16, 17, 40, 65, 129, 512, 1182):
            b = L.hif8_linear_ksplit_workspace_bytes(256 * tiles, 256, 64 * nk)
            parts = b // tile
            if b == 0:
                continue
            tail = tiles % 256
            assert b % tile == 0 and parts % tail == 0 and parts <= 3 * 256
            sp = parts // tail
            per = -(-nk // sp)
            assert (sp - 1) * per < nk and nk >= 8 * sp


class Calls:
    """The library with its launches recorded instead of made (its size queries answered by itself)."""

    def __init__(self, lib):
        self.lib, self.made = lib, {}

    def __getattr__(self, name):
        if name.endswith(("_bytes", "_size")):
            return getattr(self.lib, name)

        def launch(*args):
            self.made[name] = args
            return 0
        return launch


def dgrad_calls(pkg, monkeypatch, M, N, K, out_dtype):
    """The launches of linear_dgrad for a bf16 gradient [M, N] and a bf16 weight [N, K]."""
    calls = Calls(pkg._lib.load())
    monkeypatch.setattr(pkg._lib, "load", lambda: calls)
    monkeypatch.setattr(pkg._lib, "stream_ptr", lambda device: 0)
    monkeypatch.setattr(pkg._lib, "require_gpu_tensor", lambda t, name: None)

    class Packed:
        shape = (N, K)

        class state:
            ptr = 1

        def codes_t(self):
            return torch.empty(K, N, dtype=torch.uint8)
    y = pkg.linear_dgrad(torch.empty(M, N, dtype=torch.bfloat16), Packed(), out_dtype)
    assert y.dtype == out_dtype and y.shape == (M, K)
    return calls.made


@pytest.mark.parametrize("M,N,K", [(8192, 2112, 2304), (8192, 2112, 256)])
def test_dgrad_fp32_output_splits(pkg, monkeypatch, M, N, K):
    """The fp32 input gradient on the decode-once route gets the partials of its k ranges, on grids with a
    short last wave (288 tiles) and below one wave (32 tiles)."""
    want = pkg._lib.load().hif8_linear_ksplit_workspace_bytes(M, K, N)
    made = dgrad_calls(pkg, monkeypatch, M, N, K, torch.float32)
    assert want > 0 and made["hif8_linear_fwd_scaled"][-2] == want


def test_scaled_status_codes_without_gpu(pkg):
    L = pkg._lib.load()
    fake = 0x100000

    def wg(g=fake, st=fake, dt=1, tokens=1024, n=256, k=256, dw=fake):
        return L.hif8_linear_wgrad_scaled(g, fake, st, dw, dt, tokens, n, k, None, 0, None)

    def fw(a=fake, st=fake, dt=1, M=128, N=256, K=512, y=fake):
        return L.hif8_linear_fwd_scaled(a, fake, st, y, dt, M, N, K, None, 0, None)
    assert wg(g=None) == -1 and wg(st=None) == -1 and wg(dt=2) == -1 and wg(tokens=0) == -1
    assert wg(n=260) == -2 and wg(k=100) == -2 and wg(tokens=1 << 22) == -2 and wg(dw=fake + 2) == -3
    assert fw(a=None) == -1 and fw(dt=3) == -1 and fw(N=0) == -1
    assert L.hif8_linear_fwd_f32(None, fake, fake, fake, 64, 64, 64, None) == -1
    assert L.hif8_linear_fwd_f32(fake, fake, fake, fake, 0, 64, 64, None) == -1
    assert L.hif8_linear_fwd_f32(fake, fake, fake, fake, 64, 100, 64, None) == -2
    assert L.hif8_linear_fwd_f32(fake, fake, fake, fake, 64, 64, 100, None) == -2
    assert L.hif8_linear_fwd_f32(fake, fake, fake, fake + 8, 64, 64, 64, None) == -3
    assert fw(K=100) == -2 and fw(N=100) == -2 and fw(K=1 << 22) == -2 and fw(y=fake + 8) == -3
    assert L.hif8_decode_values(None, 16, None, fake, None) == -1
    assert L.hif8_decode_values(fake, 16, None, fake + 4, None) == -3
