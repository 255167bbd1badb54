"""q16k calls of one or two slots under graph capture: they leave the work buffer alone and may be captured and replayed;
one more slot is refused. Run with -m gpu."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from panvram_amd import _native as N

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rc", [0, 1])
def test_short_q16k_calls_are_captured(fx, oracle_ref, rc):
    import panvram_amd
    c = panvram_amd.Cohort.open(fx["dirs"]["q16k"], device="cuda", dataset="q16k", reference=fx["ref"])
    arcs = [O.Archive(f"{fx['dirs']['q16k']}/{nm}.q16k.rr3") for nm in c.names]
    L, dev = N.lib(), c.device
    a, s = 1, 30_001
    lengths = (1, 5000, 16384)
    work = torch.empty(int(L.pv_windows_work_bytes(c._Dref, 1, 40_000)), dtype=torch.uint8, device=dev)
    ta, ts = torch.tensor([a], device=dev), torch.tensor([s], device=dev)
    mask = torch.tensor([rc], dtype=torch.uint8, device=dev)
    rec = [torch.zeros(32, dtype=torch.uint8, device=dev) for _ in lengths]
    status = torch.zeros(1, dtype=torch.int32, device=dev)
    rows = [(torch.zeros(W, dtype=torch.uint8, device=dev), torch.zeros(W, dtype=torch.uint8, device=dev)) for W in lengths]
    over = torch.zeros(16385, dtype=torch.uint8, device=dev)
    other = torch.zeros(40_000, dtype=torch.uint8, device=dev)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    codes, refused = [], []
    with torch.cuda.graph(g, stream=side):
        st = torch.cuda.current_stream().cuda_stream

        def fetch(W, row, r):
            err = N.errbuf()
            return L.pv_fetch_hip(c._Dref, a, s, W, rc, 0, row.data_ptr(), r.data_ptr(), work.data_ptr(), work.numel(), st, err, len(err)), err.value

        def windows(W, row):
            err = N.errbuf()
            return L.pv_windows_hip(c._Dref, ta.data_ptr(), ts.data_ptr(), 1, W, mask.data_ptr(), 0, 1, row.data_ptr(), status.data_ptr(),
                                    work.data_ptr(), work.numel(), st, err, len(err)), err.value
        for W, (x, y), r in zip(lengths, rows, rec):
            codes += [fetch(W, x, r), windows(W, y)]
        refused += [fetch(16385, over, rec[0]), windows(16385, over)]
    assert all(code == 0 for code, _ in codes), codes
    assert all(code == N.PV_EARG and b"captured" in msg for code, msg in refused), refused
    want = [O.windows(arcs, oracle_ref, np.array([a]), np.array([s]), W, rc=np.array([rc], np.uint8))[0] for W in lengths]
    for k in range(3):
        for x, y in rows:
            x.fill_(7)
            y.fill_(7)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        for (x, y), w, r in zip(rows, want, rec):
            assert np.array_equal(x.cpu().numpy(), w) and np.array_equal(y.cpu().numpy(), w), (k, w.size)
            assert int(r[24:28].view(torch.int32)) == 0
        assert int(status) == 0 and not over.any()
        # the program's own calls between the replays, with the same buffers
        err = N.errbuf()
        assert L.pv_fetch_hip(c._Dref, 0, 12_000, 40_000 - 7, rc, 0, other.data_ptr(), rec[0].data_ptr(),
                              work.data_ptr(), work.numel(), torch.cuda.current_stream().cuda_stream, err, len(err)) == 0, err.value
        torch.cuda.synchronize()
