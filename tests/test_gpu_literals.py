"""The wave decoder's literal windows (nine literals each, at most 21 a run) at every length a long literal run can end
at: cohorts of many short insertions, without and with N / IUPAC bytes in them, at each block size, and runs of many
windows. Every block equals the CPU oracle. Run with -m gpu."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests import cohortgen as G


def _cohort(d, Q, odd, lo, hi, per):
    G.make("mini", str(d), threads=4, ref={"lengths": [120_000, 60_000]},
           asm={"Q": Q, "sv_min": lo, "sv_max": hi, "sv_per_contig": per, "ins_odd": odd, "n_asm": 2, "seed": 211 + Q + hi})
    return sorted(str(p) for p in d.glob("*.rr3"))


@pytest.mark.gpu
@pytest.mark.parametrize("Q", [1024, 2048, 4096, 16384])
@pytest.mark.parametrize("odd,lo,hi,per", [(0.0, 9, 60, 300), (0.02, 9, 60, 300), (0.0, 150, 900, 60), (0.002, 150, 900, 60)])
def test_literal_windows_equal_oracle(tmp_path, Q, odd, lo, hi, per):
    import panvram_amd
    paths = _cohort(tmp_path, Q, odd, lo, hi, per)
    fa = str(tmp_path / "reference.fa")
    c = panvram_amd.Cohort.open(str(tmp_path), device="cuda", dataset=None, reference=fa)
    assert c.block_size == Q
    ref, arcs = O.reference_bases(fa), [O.Archive(p) for p in paths]
    a, s = [], []
    for i, A in enumerate(arcs):
        for b in range(A.nblocks):
            a.append(i)
            s.append(min(b * Q, A.nbases - Q))
    a, s = np.array(a, dtype=np.int64), np.array(s, dtype=np.int64)
    want = O.windows(arcs, ref, a, s, Q)
    ta, ts = torch.from_numpy(a).cuda(), torch.from_numpy(s).cuda()
    for light in (True, False):
        c.light_decode = light
        assert np.array_equal(c.windows(ta, ts, Q).cpu().numpy(), want), light
    c.light_decode = True
    k = 20_000 // len(a) + 1                        # the large call's kernels
    x = c.windows(ta.repeat(k), ts.repeat(k), Q).view(k, len(a), Q)
    assert all(torch.equal(x[i], x[0]) for i in range(1, k)) and np.array_equal(x[0].cpu().numpy(), want)


def test_literal_entries(mini):
    """The model table's pair section against its own literal rows: lo << 4 | freq << 20, and 0 for a frequency under 16
    or of 4096."""
    from panvram_amd import _native as N
    L, err, h = N.lib(), N.errbuf(), ctypes.c_void_p()
    argv = (ctypes.c_char_p * len(mini["paths"]))(*[p.encode() for p in mini["paths"]])
    assert L.pv_cohort_open(mini["ref"].encode(), ctypes.cast(argv, ctypes.c_void_p), len(mini["paths"]), 0, 0, ctypes.byref(h), err, len(err)) == 0
    try:
        p, n = ctypes.c_void_p(), ctypes.c_uint64()
        assert L.pv_cohort_array(h, N.ARR_TAB, ctypes.byref(p), ctypes.byref(n)) == 0
        tab = np.frombuffer((ctypes.c_uint8 * n.value).from_address(p.value), dtype=np.uint8).reshape(-1, 10240).copy()
    finally:
        L.pv_cohort_close(h)
    for t in tab:
        rows = t[:736].view(np.uint16).reshape(46, 8)[10:26].astype(np.int64)      # the 16 order-2 literal contexts
        pair = t[4096:6144].view(np.uint32).reshape(16, 16, 2)

        def entry(r, s):
            f = rows[r, s + 1] - rows[r, s]
            return 0 if f < 16 or f >= 4096 else int(rows[r, s] << 4 | f << 20)
        for r in range(16):
            for l in range(16):
                s1, s2 = l >> 2, l & 3
                assert (int(pair[r, l, 0]), int(pair[r, l, 1])) == (entry(r, s1), entry((r & 3) * 4 + s1, s2))
