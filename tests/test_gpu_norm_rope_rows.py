"""q/k RMSNorm + rope (hif8_rms_norm_rope and its quantising forms) over more rows than the grid's waves:
the rows a wave takes in turn, their rope rows and, up to 2048 features, the loads a row ahead.

Oracle: the same kernel on pieces of `seq` rows, where no wave takes a second row and the rope row is the
row itself (test_gpu_dit_norm_rope.py checks that against torch's ops and the codec); equal bit for bit."""
from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda:0"


# 1, 3, 4 (the last with loads ahead), 5, 10 and 16 chunks a lane; rows: one past the 2048 workgroups' 8192
# waves, and several turns with a ragged last one
@pytest.mark.parametrize("dim", [512, 1536, 2048, 2560, 5120, 8192])
@pytest.mark.parametrize("seq,batch,rep", [(2731, 3, 1), (2731, 3, 3), (5003, 4, 2), (1, 8193, 8193)])
@pytest.mark.parametrize("sem", [0, 1])
def test_rows_in_turn(pkg, dim, seq, batch, rep, sem):
    L = pkg._lib.load()
    s = pkg._lib.stream_ptr(torch.device(DEV))
    g = torch.Generator(device=DEV).manual_seed(dim + seq)
    rows = seq * batch
    x = (torch.randn(rows, dim, generator=g, device=DEV) * 3).to(torch.bfloat16)
    w = torch.rand(dim, generator=g, device=DEV) + 0.5
    cs, sn = (torch.randn(batch // rep * seq, 64, generator=g, device=DEV) for _ in range(2))
    whole, q = torch.empty_like(x), torch.empty_like(x)
    st = pkg.QuantState(torch.device(DEV))
    tail = (rows, dim, 128, seq, rep, 1e-6)
    for rc in (L.hif8_rms_norm_rope(x.data_ptr(), w.data_ptr(), cs.data_ptr(), sn.data_ptr(), whole.data_ptr(), *tail, s),
               L.hif8_rms_norm_rope_amax(x.data_ptr(), w.data_ptr(), cs.data_ptr(), sn.data_ptr(), *tail, 15.0, st.ptr, s),
               L.hif8_rms_norm_rope_fake_quant(x.data_ptr(), w.data_ptr(), cs.data_ptr(), sn.data_ptr(), *tail, st.ptr, sem,
                                               q.data_ptr(), None, s)):
        assert rc == 0
    step = seq if seq > 1 else 4096   # seq 1: every row takes table row 0 of a table with one row
    want, want_q = torch.empty_like(x), torch.empty_like(x)
    amax = 0
    for r0 in range(0, rows, step):
        n = min(step, rows - r0)
        sq, rp = (seq, 1) if seq > 1 else (1, n)
        t0 = (r0 // seq // rep) * seq * 64 * 4
        args = (cs.data_ptr() + t0, sn.data_ptr() + t0)
        at = r0 * dim * 2
        piece = pkg.QuantState(torch.device(DEV))
        tail = (n, dim, 128, sq, rp, 1e-6)
        assert L.hif8_rms_norm_rope(x.data_ptr() + at, w.data_ptr(), *args, want.data_ptr() + at, *tail, s) == 0
        assert L.hif8_rms_norm_rope_amax(x.data_ptr() + at, w.data_ptr(), *args, *tail, 15.0, piece.ptr, s) == 0
        amax = max(amax, piece.read()[0])
        assert L.hif8_rms_norm_rope_fake_quant(x.data_ptr() + at, w.data_ptr(), *args, *tail, st.ptr, sem,
                                               want_q.data_ptr() + at, None, s) == 0
    assert torch.equal(whole.view(torch.int16), want.view(torch.int16))
    assert torch.equal(q.view(torch.int16), want_q.view(torch.int16))
    assert st.read()[0] == amax
