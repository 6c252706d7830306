"""The two-level fold of the amax passes (fold_amax): the maximum is found wherever it sits, on grids
below, at and above the two-level threshold and with uneven groups of workgroups, and the state's
counters are zero again after each pass."""
from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda:0"
PER_WG = 256 * 64      # elements of one workgroup's step of the bf16 amax pass


def amax_bits(x):
    return int((x.view(torch.int16).int() & 0x7FFF).max())


@pytest.mark.parametrize("wgs", [1, 2, 31, 63, 64, 65, 95, 96, 97, 255, 256, 700])
def test_amax_any_position(pkg, wgs):
    n = PER_WG * wgs - 5
    x = torch.full((n,), 0.5, device=DEV, dtype=torch.bfloat16)
    st = pkg.QuantState(DEV)
    for i in range(6):
        at = (n - 1) * i // 5
        x[at] = -(3.0 + i)
        pkg.absmax_scale(x, 15.0, st)
        x[at] = 0.5
        assert st.read()[0] == amax_bits(torch.tensor([3.0 + i], dtype=torch.bfloat16))
        head = st.buf[:8].view(torch.int32)
        assert int(head[0]) == 0 and int(head[1]) == 0       # counter, running maximum


@pytest.mark.parametrize("rows", [3, 255, 257, 1000, 4099])
def test_norm_passes_settle_the_same_state(pkg, rows):
    """The modulated norm's amax pass on grids of several sizes: the state of an amax pass over its y."""
    g = torch.Generator().manual_seed(rows)
    x = torch.randn(rows, 512, generator=g).to(torch.bfloat16).to(DEV)
    e = (torch.randn(2, 1, 512, generator=g) * 0.5).to(torch.bfloat16).to(DEV)
    for _ in range(3):
        _, st, y = pkg.modulated_norm_quant(x, e[0], e[1], return_y=True)
        assert st.read() == pkg.absmax_scale(y, 15.0, pkg.QuantState(DEV)).read()
