"""The light lanes (one lane per block) at the edges of what they take: blocks of many short ops, payloads up to and past
the lanes' limit, literal bytes that are N or escapes, rare lengths and distances (past a bucket entry's symbols),
reverse-complemented pieces - at each block size, with the reference as bytes and packed. The kernels differ by the
call's (window, covering block) slots: one window of at most 64 (one wave, the model table in LDS), more windows or slots
(one kernel), over 16,384 (2,048 at q16k: kernels of their own), and over that with windows of 256 slots or more (waves
of one assembly hold the table in LDS, waves across two do not). Everything equals the CPU oracle. Run with -m gpu."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests import cohortgen as G

pytestmark = pytest.mark.gpu


def _open(d, Q, **asm):
    import panvram_amd
    G.make("mini", str(d), threads=4, ref={"lengths": [1_500_000, 700_000], "iupac_runs": 40},
           asm={"Q": Q, "n_asm": 2, "sv_min": 1, "sv_max": 900, "sv_per_contig": 20, "seed": 307 + Q, **asm})
    fa = str(d / "reference.fa")
    ref = O.reference_bases(fa)
    full = [O.Archive(str(p)).full(ref) for p in sorted(d.glob("*.rr3"))]
    return full, lambda packed: panvram_amd.Cohort.open(str(d), device="cuda", dataset=None, reference=fa, packed_reference=packed,
                                                        compact_blocks=packed)


@pytest.mark.parametrize("Q", [1024, 2048, 4096, 16384])
@pytest.mark.parametrize("snv,indel,odd", [(5e-4, 5e-5, 0.0), (2e-3, 4e-4, 0.05), (8e-3, 2e-3, 0.01)])
def test_lanes_equal_oracle(tmp_path, Q, snv, indel, odd):
    full, opened = _open(tmp_path, Q, snv_rate=snv, indel_rate=indel, ins_odd=odd)
    many = (2048 if Q == 16384 else 16384) // 2 + 500     # windows of two slots: past the one-kernel path
    for packed in (False, True):
        c = opened(packed)
        for a, want in enumerate(full):                   # one window: the whole assembly, and a ragged part of it
            n = len(want)
            assert np.array_equal(c.windows(torch.tensor([a]), torch.tensor([0]), n)[0].cpu().numpy(), want)
            assert np.array_equal(c.windows(torch.tensor([a]), torch.tensor([777]), n - 1300)[0].cpu().numpy(), want[777:n - 523])
            for W in (5, Q, Q + 1, 40 * Q + 3, 63 * Q):   # one window of 2 to 64 slots
                s = (a + 1) * 12_345
                assert np.array_equal(c.windows(torch.tensor([a]), torch.tensor([s]), W)[0].cpu().numpy(), want[s:s + W]), (packed, a, W)
        rng = np.random.default_rng(5)
        for n, W in ((3, 5), (40, 3 * Q + 1), (many, Q - 1)):     # small calls, then a large one
            a = rng.integers(0, len(full), n)
            s = np.array([rng.integers(0, len(full[i]) - W) for i in a])
            x = c.windows(torch.from_numpy(a).cuda(), torch.from_numpy(s).cuda(), W).cpu().numpy()
            want = np.stack([full[i][t:t + W] for i, t in zip(a, s)])
            assert np.array_equal(x, want), (packed, n, W)


@pytest.mark.parametrize("Q", [1024, 2048, 4096])
def test_long_windows_of_a_large_call_equal_oracle(tmp_path, Q):
    """64 windows of 301 slots (19,264), the assemblies in turn: a wave of 64 slots lies in one window or across two."""
    full, opened = _open(tmp_path, Q, snv_rate=2e-3, indel_rate=4e-4, ins_odd=0.02)
    W = 300 * Q - 7
    for packed in (False, True):
        c = opened(packed)
        a = np.arange(64) % 2
        s = np.array([(k * 9_973) % (len(full[i]) - W) for k, i in enumerate(a)])
        x = c.windows(torch.from_numpy(a).cuda(), torch.from_numpy(s).cuda(), W).cpu().numpy()
        for row, i, t in zip(x, a, s):
            assert np.array_equal(row, full[i][t:t + W]), (packed, i, t)
