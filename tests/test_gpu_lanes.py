"""The light lanes (one lane per block) at the edges of what they take: blocks of many short ops, payloads up to and past
the lanes' limit, literal bytes that are N or escapes, rare lengths and distances (past a bucket entry's symbols),
reverse-complemented pieces - at each block size, in small calls, large calls and calls of one long window (whose waves
hold the model table in LDS). Everything equals the CPU oracle. Run with -m gpu."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests import cohortgen as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Q", [1024, 4096, 16384])
@pytest.mark.parametrize("snv,indel,odd", [(5e-4, 5e-5, 0.0), (2e-3, 4e-4, 0.05), (8e-3, 2e-3, 0.01)])
def test_lanes_equal_oracle(tmp_path, Q, snv, indel, odd):
    import panvram_amd
    G.make("mini", str(tmp_path), threads=4, ref={"lengths": [1_500_000, 700_000], "iupac_runs": 40},
           asm={"Q": Q, "snv_rate": snv, "indel_rate": indel, "ins_odd": odd, "n_asm": 2, "sv_min": 1, "sv_max": 900, "sv_per_contig": 20,
                "seed": 307 + Q})
    fa = str(tmp_path / "reference.fa")
    paths = sorted(str(p) for p in tmp_path.glob("*.rr3"))
    ref, arcs = O.reference_bases(fa), [O.Archive(p) for p in paths]
    full = [A.full(ref) for A in arcs]
    for packed in (False, True):
        c = panvram_amd.Cohort.open(str(tmp_path), device="cuda", dataset=None, reference=fa, packed_reference=packed, compact_blocks=packed)
        for a, want in enumerate(full):                   # one window: the whole assembly, and a ragged part of it
            n = len(want)
            assert np.array_equal(c.windows(torch.tensor([a]), torch.tensor([0]), n)[0].cpu().numpy(), want)
            assert np.array_equal(c.windows(torch.tensor([a]), torch.tensor([777]), n - 1300)[0].cpu().numpy(), want[777:n - 523])
        rng = np.random.default_rng(5)
        for n, W in ((3, 5), (40, 3 * Q + 1), (20_000 * 1024 // Q + 2100, Q - 1)):     # small calls, then a large one
            a = rng.integers(0, len(full), n)
            s = np.array([rng.integers(0, len(full[i]) - W) for i in a])
            x = c.windows(torch.from_numpy(a).cuda(), torch.from_numpy(s).cuda(), W).cpu().numpy()
            want = np.stack([full[i][t:t + W] for i, t in zip(a, s)])
            assert np.array_equal(x, want), (packed, n, W)
