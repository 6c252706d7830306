"""hif8_quantize (amax, scale and quantisation in two launches, the state settled by the second) against
hif8_state_init + hif8_absmax_scale + hif8_encode / hif8_fake_quant / hif8_fake_quant_to_bf16: the same
output bytes and the same state, starting from a state full of garbage."""
from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")

DEV = "cuda:0"
SPAN = 4 * 256 * 256 * 16       # elements from which the quantisation takes spans on 256 CUs


def inputs(n, dtype, special, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(n, generator=g) * 3
    if special == "zeros":
        x.zero_()
    elif special == "tiny":
        x *= 1e-12
    elif special == "huge":
        x *= 1e30
    elif special:
        x[(n - 1) // 2] = float(special)
    return x.to(dtype).to(DEV)


def both(pkg, x, kind, sem, as_f32=False):
    lib = pkg._lib
    L, s = lib.load(), lib.stream_ptr(x.device)
    dt = lib.DTYPE_BF16_AS_F32 if as_f32 else lib.dtype_code(x.dtype)
    st = pkg.absmax_scale(x, 15.0, pkg.QuantState(DEV), as_f32)
    if kind == lib.OUT_CODES:
        want = pkg.encode(x, st, as_f32)
    elif kind == lib.OUT_SAME:
        want = pkg.fake_quant(x, st, sem)
    else:
        want = pkg.fake_quant_to_bf16(x, st, sem, as_f32)
    got = torch.empty_like(want)
    buf = torch.full((lib.state_size(),), 0xA5, dtype=torch.uint8, device=DEV)
    lib.check(L.hif8_quantize(x.data_ptr(), dt, x.numel(), 15.0, buf.data_ptr(), got.data_ptr(), kind, sem, s), "q")
    assert torch.equal(got.view(torch.uint8), want.view(torch.uint8))
    head = 32 + 512 + 1024                       # scalars and decode tables
    a, b = buf[:head].clone(), st.buf[:head].clone()
    assert torch.equal(a, b)
    # counters zero: the state serves the other entry points
    st2 = pkg.QuantState.unset(x.device)
    st2.buf = buf
    y = (torch.randn(70000, device=DEV) * 2).to(torch.bfloat16)
    assert pkg.absmax_scale(y, 15.0, st2).read() == pkg.absmax_scale(y, 15.0, pkg.QuantState(DEV)).read()


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 15, 16, 4097, 256 * 64 + 1, 300000, SPAN - 16, SPAN, SPAN + 1037])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("kind", [0, 1, 3])
def test_sizes(pkg, n, dtype, kind):
    both(pkg, inputs(n, dtype, None, n), kind, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("special", ["zeros", "tiny", "huge", "inf", "-inf", "nan"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_degenerate_scales(pkg, special, dtype):
    for kind, sem in ((0, 0), (1, 0), (1, 1), (3, 0), (3, 1)):
        both(pkg, inputs(5003, dtype, special, 1), kind, sem)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1000, SPAN + 48])
def test_bf16_as_f32(pkg, n):
    x = inputs(n, torch.bfloat16, None, 3)
    for kind in (0, 3):
        both(pkg, x, kind, 0, as_f32=True)
    got, st = pkg.hif8_linear.quantize(x, 15.0, as_f32=True)      # OUT_SAME: the fp32 x_q of x.float()
    want, ref = pkg.hif8_linear.quantize(x.float(), 15.0)
    assert got.dtype == torch.float32 and torch.equal(got, want) and st.read() == ref.read()


@pytest.mark.parametrize("dtype,as_f32", [("bfloat16", False), ("float32", False), ("bfloat16", True)])
@pytest.mark.parametrize("kind", [0, 1, 3])
def test_output_holds_what_the_kernel_writes(pkg, monkeypatch, dtype, as_f32, kind):
    """quantize allocates the bytes that hif8_quantize writes for its dtype and kind (hif8_mi355x.h): codes
    1 an element, OUT_BF16 2, OUT_SAME 2 for a bf16 tensor and 4 for fp32 arithmetic, bf16 storage or not."""
    lib, calls = pkg._lib, []

    class Recorder:
        def hif8_quantize(self, *args):
            calls.append(args)
            return 0
    monkeypatch.setattr(lib, "load", Recorder)
    monkeypatch.setattr(lib, "require_gpu_tensor", lambda t, name: None)
    monkeypatch.setattr(lib, "stream_ptr", lambda device: 0)
    monkeypatch.setattr(lib, "unset_state", lambda device: torch.empty(4096, dtype=torch.uint8))
    x = torch.zeros(5, 32, dtype=getattr(torch, dtype))
    out, _ = pkg.hif8_linear.quantize(x, 15.0, kind, as_f32=as_f32)
    (_, code, n, _, _, ptr, _, _, _), = calls
    writes = {0: 1, 3: 2, 1: 2 if code == lib.DTYPE_BF16 else 4}[kind]
    assert ptr == out.data_ptr() and n == x.numel() and out.element_size() == writes and out.shape == x.shape


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 17, 4099, SPAN + 333])
@pytest.mark.parametrize("special", [None, "inf", "nan", "zeros"])
def test_with_codes(pkg, n, special):
    """The bf16 x_q and the codes of one pass: those of the two separate passes."""
    x = inputs(n, torch.float32, special, n)
    xq, codes, st = pkg.hif8_linear.quantize_with_codes(x, 15.0)
    want = pkg.absmax_scale(x, 15.0, pkg.QuantState(DEV))
    assert torch.equal(codes, pkg.encode(x, want)) and st.read()[0] == want.read()[0]
    assert torch.equal(xq.view(torch.int16), pkg.fake_quant_to_bf16(x, want).view(torch.int16))


def test_status_codes_without_gpu(pkg):
    L = pkg._lib.load()
    f = 0x100000

    def q(x=f, dt=0, n=16, st=f, out=f, kind=1, sem=0):
        return L.hif8_quantize(x, dt, n, 15.0, st, out, kind, sem, None)
    assert q(x=None) == -1 and q(st=None) == -1 and q(out=None) == -1 and q(n=0) == -1 and q(dt=7) == -1
    assert L.hif8_quantize_with_codes(f, 1, 16, 15.0, f, f, None, None) == -1
    assert L.hif8_quantize_with_codes(f, 0, 16, 15.0, f, f, f, None) == -1        # a bf16 tensor's x_q is bf16
    assert L.hif8_quantize_with_codes(f, 1, 16, 15.0, f, f, f + 4, None) == -3
    assert q(kind=2) == -1 and q(sem=2) == -1 and q(kind=0, sem=1) == -1 and q(x=f + 2) == -3 and q(out=f + 8) == -3
