"""The calls whose speed counts: what programs ask of a resident cohort, from one short slice to whole chromosomes.

A case names one call of `panvram_amd.Cohort` and its sizes. Three synthetic cohorts stand behind them, written by the
generator that the tests and bench.py use (tests/cohortgen) and opened once per process, as a program keeps them:

  human    the 3.1 Gbp chromosome-like reference and 32 haplotypes (SNVs, indels, 200 structural variants of 1-100 kbp
           each) at q4k: the headline cohort's shape
  mid      256 Mbp in 16 contigs, 32 fragmented, half soft-masked haplotypes at q4k
  mid16    the same at q16k

`mid` is also held with the 2-bit reference and the compact block table (`packed`). What changes with the seed is what
a program changes from call to call: the slices' places, the coordinates, the generator's draws, the assembly.
Every output is bytes, token ids or whole numbers, so another implementation's are equal.
"""
import functools
import os
import tempfile

import torch

import panvram_amd
from tests import cohortgen

_COHORTS = {
    "human": dict(preset="headline", asm={"n_asm": 32}, dataset="q4k"),
    "mid": dict(preset="mid", dataset="q4k"),
    "mid16": dict(preset="mid16", dataset="q16k"),
    "packed": dict(preset="mid", dataset="q4k", packed_reference=True, compact_blocks=True),
}
# block size and mean payload bytes per block of each cohort (for the bytes a call cannot do without)
_BLOCK = {"human": (4096, 13.4), "mid": (4096, 12.3), "mid16": (16384, 38.1), "packed": (4096, 12.3)}
_IDS = (11, 12, 13, 14, 15)


@functools.lru_cache(maxsize=None)
def _cohort(name):
    kw = dict(_COHORTS[name])
    preset, asm = kw.pop("preset"), kw.pop("asm", None)
    shm = "/dev/shm"
    with tempfile.TemporaryDirectory(prefix="panvram_", dir=shm if os.access(shm, os.W_OK) else None) as d:
        cohortgen.make(preset, d, asm=asm)
        return panvram_amd.Cohort.open(d, device="cuda", **kw)      # holds what it needs of the files


def listed():
    return [
        # a variant caller or a genome browser asks for one short slice and waits for it
        {"name": "fetch_1000", "op": "fetch", "cohort": "human", "W": 1000},
        # the same on the large-block archive, at the slice length its users take
        {"name": "fetch_5000_q16k", "op": "fetch", "cohort": "mid16", "W": 5000},
        # one gene-cluster sized slice, reverse strand: the longest single fetch of the latency draw (1 .. 2^20)
        {"name": "fetch_1M_rc", "op": "fetch", "cohort": "human", "W": 1 << 20, "rc": True},
        # a training step's batch, decoded when it is needed and its status looked at: the headline batch
        {"name": "sample_1024x8192", "op": "sample", "cohort": "human", "n": 1024, "W": 8192, "check": True, "coords": True},
        # the same batch in a loop that keeps several calls in flight: tokens, half the windows reverse-complemented
        {"name": "sample_1024x8192_tok", "op": "sample", "cohort": "mid", "n": 1024, "W": 8192, "rc": 0.5, "tokens": True, "coords": True},
        # the batch out of the small resident form (2-bit reference, compact block table), with case
        {"name": "sample_1024x8192_packed", "op": "sample", "cohort": "packed", "n": 1024, "W": 8192},
        # a language-model loader's batch of odd size: int64 token ids, an odd context length
        {"name": "sample_500x2049_ids", "op": "sample", "cohort": "mid", "n": 500, "W": 2049, "rc": 0.5, "ids": True},
        # long contexts from the large-block archive
        {"name": "sample_1024x65536_q16k", "op": "sample", "cohort": "mid16", "n": 1024, "W": 65536},
        # the largest batch: a pre-training loader that fills half a gigabyte at a time
        {"name": "sample_65536x8192", "op": "sample", "cohort": "human", "n": 65536, "W": 8192},
        # a batch of slices at coordinates the program has (a panel of loci over all haplotypes), q16k
        {"name": "windows_65536x5000_q16k", "op": "windows", "cohort": "mid16", "n": 65536, "W": 5000, "check": True},
        # a whole chromosome's worth of one haplotype into device memory
        {"name": "windows_1x2^28", "op": "windows", "cohort": "human", "n": 1, "W": 1 << 28, "check": True},
        # a whole 256 Mbp assembly into pinned host memory
        {"name": "decode_256M", "op": "decode", "cohort": "mid"},
    ]


def _log(rng, lo, hi):
    """A whole number in [lo, hi], even over its logarithm, odd as often as not."""
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    op = rng.choice(["fetch", "fetch", "sample", "sample", "sample", "windows", "windows", "span"])
    cohort = rng.choice(["human", "mid", "mid16", "packed"])
    if op == "fetch":
        return {"op": "fetch", "cohort": cohort, "W": _log(rng, 64, 1 << 20), "rc": rng.random() < 0.5, "tokens": rng.random() < 0.3}
    if op == "span":
        return {"op": "windows", "cohort": cohort, "n": rng.randint(1, 3), "W": _log(rng, 1 << 20, 1 << 26), "check": rng.random() < 0.5}
    case = {"op": op, "cohort": cohort, "W": _log(rng, 256, 65536), "check": rng.random() < 0.5}
    form = rng.choice(["bytes", "bytes", "tokens", "ids"])
    case["n"] = _log(rng, 16, min(65536, (1 << 29) // (case["W"] * (8 if form == "ids" else 1))))
    if form != "bytes":
        case[form] = True
    if rng.random() < 0.5:
        case["rc"] = rng.choice([0.25, 0.5])
    if op == "sample" and rng.random() < 0.3:
        case["coords"] = True
    return case


def prepare(case, seed):
    c = _cohort(case["cohort"])
    s = dict(case, c=c)
    gen = torch.Generator(device=c.device).manual_seed(seed)
    if case["op"] == "sample":
        s["gen"] = gen
        return s
    if case["op"] == "decode":
        s["a"] = seed % len(c)
        longest = max(c.info(a)["bases"] for a in range(len(c)))          # one buffer takes any assembly
        s["out"] = torch.zeros(longest, dtype=torch.uint8, pin_memory=True)
        return s
    W = case["W"]
    if case["op"] == "fetch":
        pick = torch.Generator().manual_seed(seed)
        s["a"] = seed % len(c)
        room = [(k, t[2]) for k, t in enumerate(c.contigs(s["a"])) if t[2] >= W]
        s["ctg"], length = room[int(torch.randint(len(room), (1,), generator=pick))]
        s["start"] = int(torch.randint(length - W + 1, (1,), generator=pick))
        return s
    n = case["n"]
    bases = torch.tensor([c.info(a)["bases"] for a in range(len(c))], device=c.device)
    s["asm"] = torch.randint(len(c), (n,), generator=gen, device=c.device)
    place = torch.rand(n, dtype=torch.float64, generator=gen, device=c.device)
    s["start"] = (place * (bases[s["asm"]] - W)).to(torch.int64)
    s["mask"] = torch.rand(n, generator=gen, device=c.device) < case["rc"] if case.get("rc") else None
    return s


def run(state):
    c, op, tokens = state["c"], state["op"], state.get("tokens", False)
    ids = _IDS if state.get("ids") else None
    if op == "fetch":
        return c.fetch(state["a"], state["ctg"], state["start"], state["W"], reverse_complement=state.get("rc", False), tokens=tokens)
    if op == "sample":
        return c.sample(state["n"], state["W"], generator=state["gen"], reverse_complement=state.get("rc", False), tokens=tokens,
                        return_coords=state.get("coords", False), check=state.get("check", False), token_ids=ids)
    if op == "windows":
        return c.windows(state["asm"], state["start"], state["W"], reverse_complement=state["mask"], tokens=tokens,
                         check=state.get("check", False), token_ids=ids)
    c.decode(state["a"], out=state["out"])
    return state["out"]


def work(case):
    """Each window's covering blocks (payload and 16 bytes of block table), the reference bytes it copies (a quarter of
    a byte per base in the packed form), the draws and what is returned. The decode has no floating-point work."""
    Q, payload = _BLOCK[case["cohort"]]
    n, W = case.get("n", 1), case.get("W", 256_000_000)
    blocks = W / Q + 1
    read = blocks * (payload + 16) + W * (0.25 if case["cohort"] == "packed" else 1.0)
    wrote = W * (8 if case.get("ids") else 1) + (32 if case.get("coords") else 0)
    return {"bytes": n * (read + wrote + (8 if case["op"] == "sample" else 16)), "flops": 0.0}


def tolerance(case):
    return "exact"
