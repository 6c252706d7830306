"""hif8_quantize_colsum: the gradient's fake quant with its column sums (the bias gradient,
hif8_linear.py:93,107) in one pass.  The quantised gradient and the state must equal hif8_quantize's byte
for byte; the sums lie within 2^-20 of sum |g_q| of the float64 sums, plus 2^-8 of themselves in bf16.
(A column's sum is a chain of at most 128 rows in a thread, at most 256 lanes of a workgroup and 64 of at
most 1024 workgroups in the shapes here, then 16: under 2^9 fp32 additions, each rounding a partial sum of
at most sum |g_q| by 2^-24 of it, in either direction; 16 such roundings in one direction are allowed.)"""
from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")

DEV = "cuda:0"


# rows around the 8 in flight and the 16 (or more) of a workgroup, with partials of several workgroups;
# columns of one chunk, of part of a strip, of uneven strips; columns that 256, 32, 3 and 2 lanes of a
# workgroup share (up to 1024 columns), with idle threads beside them and lanes past the last row; enough
# of both for larger row blocks
SHAPES = [(1, 8), (7, 64), (8, 2048), (9, 2056), (15, 1536), (16, 1536), (17, 1536), (33, 4104), (63, 1536), (65, 4104),
          (129, 8960), (1000, 13824), (40000, 2048), (70001, 1536), (300, 40), (2049, 8), (75600, 64), (20001, 680),
          (5000, 1024), (33000, 1032)]


@pytest.mark.gpu
@pytest.mark.parametrize("M,N", SHAPES)
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_quant_and_sums(pkg, M, N, out_dtype):
    print(f"[colsum] M={M} N={N} {out_dtype}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(M + N)
    x = (torch.randn(M, N, generator=g, device=DEV) * 1e-3 + 1e-4).to(torch.bfloat16)
    xq, sums = pkg.hif8_linear.quantize_colsum(x, 224.0, out_dtype)
    want, st = pkg.hif8_linear.quantize(x, 224.0)
    assert torch.equal(xq.view(torch.int16), want.view(torch.int16))
    ref = want.double().sum(0)
    tol = want.double().abs().sum(0) * 2.0 ** -20
    if out_dtype == torch.bfloat16:
        tol = tol + ref.abs() * 2.0 ** -8
    assert sums.dtype == out_dtype and bool(((sums.double() - ref).abs() <= tol).all())
    again = pkg.hif8_linear.quantize_colsum(x, 224.0, out_dtype)[1]
    assert torch.equal(again, sums)


@pytest.mark.gpu
@pytest.mark.parametrize("value", [0.0, float("inf"), float("nan")])
def test_degenerate(pkg, value):
    x = torch.zeros(100, 72, device=DEV, dtype=torch.bfloat16)
    x[3, 5] = value
    xq, sums = pkg.hif8_linear.quantize_colsum(x, 224.0, torch.float32)
    want, _ = pkg.hif8_linear.quantize(x, 224.0)
    assert torch.equal(xq.view(torch.int16), want.view(torch.int16))
    assert torch.equal(torch.isfinite(sums), torch.isfinite(want.float().sum(0)))


@pytest.mark.gpu
def test_backward_takes_it(pkg):
    """HIF8Linear's bias gradient and the others are those of the separate passes."""
    torch.manual_seed(2)
    lin = pkg.HIF8Linear(256, 264, device=DEV, dtype=torch.bfloat16)
    x = torch.randn(500, 256, device=DEV).to(torch.bfloat16).requires_grad_(True)
    gy = torch.randn(500, 264, device=DEV).to(torch.bfloat16)
    lin(x).backward(gy)
    gq, _ = pkg._quant(gy, 224.0)
    ref = gq.double().sum(0)
    assert bool(((lin.bias.grad.double() - ref).abs() <= ref.abs() * 2.0 ** -8 + gq.double().abs().sum(0) * 2.0 ** -20).all())
    assert torch.equal(x.grad, pkg.linear_dgrad(gq, lin._packed_weight()))


def test_status_codes_without_gpu(pkg):
    L = pkg._lib.load()
    f = 0x100000

    def q(x=f, M=64, N=64, st=f, dt=0, out=f, ws=f, nb=1 << 30):
        return L.hif8_quantize_colsum(x, M, N, 224.0, st, f, out, dt, ws, nb, None)
    assert q(x=None) == -1 and q(st=None) == -1 and q(out=None) == -1 and q(ws=None) == -1 and q(dt=2) == -1
    assert q(M=0) == -1 and q(N=60) == -2 and q(x=f + 2) == -3 and q(ws=f + 4) == -3 and q(nb=16) == -1
    assert L.hif8_quantize_colsum_workspace_bytes(64, 64) == 4 * 64 * 4
    assert L.hif8_quantize_colsum_workspace_bytes(0, 64) == 0
