"""The fused GEMM on small tiles (hif8_gemm_small.hip), which hif8_linear_fwd and its GELU-statistic and
grouped forms take for few rows or features.

It issues the products of the decode-free GEMM (hif8_linear_fwd_wq, checked against float64 in
test_gpu_w16.py) in the same order, so its outputs are compared with that kernel's bit for bit."""
from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda:0"
# one to six 64-k steps (odd counts, steps past the ring's depth), rows and features at and past the
# edges of the 32 x 32, 64 x 64, 128 x 64 and 128 x 128 tiles, and grids that pick each of them, the last
# pairs at and past the rows where the 256 x 256 kernel takes over on 256 CUs
SHAPES = [(1, 64, 8), (31, 128, 32), (33, 192, 40), (64, 320, 264), (65, 384, 1544), (127, 1024, 2048),
          (300, 256, 2568), (513, 704, 1536), (260, 448, 8960), (1000, 1600, 1536), (600, 640, 5128), (129, 8960, 776),
          (2688, 1536, 1536), (2689, 1536, 1536), (384, 1536, 8960), (385, 1536, 8960)]


def operands(pkg, M, K, N, seed, bias=True):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(M, K, generator=g)
    x[:, :3] *= 20
    w = (torch.randn(N, K, generator=g) * 0.02).to(torch.bfloat16).to(DEV)
    b = (torch.randn(N, generator=g) * 0.1).to(torch.bfloat16).to(DEV) if bias else None
    a, fmt, st = pkg.quantize_activation(x.to(torch.bfloat16).to(DEV), 15.0, "bf16")
    return a, fmt, st, pkg.PackedWeight(w, 15.0), b


def same(x, y):
    return torch.equal(x.view(torch.int16), y.view(torch.int16))


@pytest.mark.parametrize("M,K,N", SHAPES)
@pytest.mark.parametrize("bias", [True, False])
def test_equals_decode_free(pkg, M, K, N, bias):
    print(f"[small] M={M} K={K} N={N} bias={bias}", flush=True)
    a, fmt, st, packed, b = operands(pkg, M, K, N, M + K + N, bias)
    assert same(pkg.linear_fwd(a, fmt, st, packed, b), pkg.linear_fwd_wq(a, packed.dequantize(torch.bfloat16), b))


@pytest.mark.parametrize("M,K,N", [(1, 64, 8), (64, 320, 264), (300, 256, 2568), (1000, 1600, 1536), (513, 704, 1536)])
def test_gelu_statistic(pkg, M, K, N):
    """The outputs and the statistic, wherever in a workgroup's tile the largest output lies."""
    a, _, _, packed, b = operands(pkg, M, K, N, 3 * M + N)
    s_f, s_w = pkg.QuantState(DEV), pkg.QuantState(DEV)
    got = pkg.linear_fwd_gelu_stat(a, packed, b, s_f, 15.0)
    want = pkg.linear_fwd_wq(a, packed.dequantize(torch.bfloat16), b, s_w, 15.0)
    assert same(got, want) and s_f.read() == s_w.read()
    for at in (0, M // 2, M - 1):
        top = a.clone()
        top[at] *= 64
        pkg.linear_fwd_gelu_stat(top, packed, b, s_f, 15.0)
        pkg.linear_fwd_wq(top, packed.dequantize(torch.bfloat16), b, s_w, 15.0)
        assert s_f.read() == s_w.read()


@pytest.mark.parametrize("M", [1, 77, 512])
def test_groups(pkg, M):
    """Groups ending inside tiles of every width, each with its own decode table."""
    g = torch.Generator().manual_seed(M)
    K, ns = 384, (256, 512, 264)
    a, _, _ = pkg.quantize_activation(torch.randn(M, K, generator=g).to(torch.bfloat16).to(DEV), 15.0, "bf16")
    packs = [pkg.PackedWeight((torch.randn(n, K, generator=g) * 0.02 * (i + 1)).to(torch.bfloat16).to(DEV), 15.0)
             for i, n in enumerate(ns)]
    for y, p in zip(pkg.linear_fwd_grouped(a, pkg.GroupedWeight(packs, [None] * 3)), packs):
        assert same(y, pkg.linear_fwd_wq(a, p.dequantize(torch.bfloat16), None))
