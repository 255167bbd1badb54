"""Calls from several threads on one stream: a `fetch` or `windows` call passes slot records from one launch to the next
through a work buffer, so each thread has its own. And no call waits for what its stream has queued."""
import threading
import time
import types

import numpy as np
import pytest
import torch

from oracle import oracle as O


def test_each_thread_has_its_work_buffer(monkeypatch):
    """Two threads on one stream: the work pointers given to the library differ, and each thread's stays the same."""
    from panvram_amd import cohort as M
    calls = []

    class Lib:
        def pv_windows_work_bytes(self, D, n, W):
            return 1536

        def pv_fetch_hip(self, *a):
            calls.append((threading.get_ident(), a[8]))
            return 0

    lib = Lib()
    monkeypatch.setattr(M.N, "lib", lambda: lib)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: types.SimpleNamespace(cuda_stream=0))
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    c = M.Cohort.__new__(M.Cohort)
    c.names, c._by_name, c._ctgs, c._ctg_index = ["a"], {"a": 0}, [[("c", "c", 1000, 0, 60)]], [{"c": 0}]
    c.device, c._idx, c._Dref, c._h, c.light_decode, c.kernel_events = torch.device("cpu"), 0, None, None, True, None
    c._local, c._stream_work, c._views, c._fast = threading.local(), {}, {}, {}
    meet, failed = threading.Barrier(2), []

    def work():
        try:
            for _ in range(2):
                c.fetch(0, 0, 5, 100)
                meet.wait(30)                                      # both are alive at every call
        except Exception as e:
            failed.append(e)
            meet.abort()

    ts = [threading.Thread(target=work) for _ in range(2)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not failed, failed
    by = {}
    for who, ptr in calls:
        by.setdefault(who, set()).add(ptr)
    a, b = by.values()
    assert len(a) == len(b) == 1 and None not in a | b and a != b


@pytest.mark.gpu
@pytest.mark.parametrize("ds", ["q1k", "q4k", "q16k"])
def test_threads_on_one_stream_equal_oracle(fx, oracle_ref, ds):
    """Four threads on the default stream, each with lengths of its own and `fetch` and `windows` in turn."""
    import panvram_amd
    c = panvram_amd.Cohort.open(fx["dirs"][ds], device="cuda", dataset=ds, reference=fx["ref"])
    arcs = [O.Archive(f"{fx['dirs'][ds]}/{nm}.{ds}.rr3") for nm in c.names]
    full = [A.full(oracle_ref) for A in arcs]
    bad = []

    def work(t):
        try:
            rng = np.random.default_rng(100 + t)
            W = (37, 1500, 5000, 16000)[t]
            for k in range(150):
                a = int(rng.integers(len(c)))
                rows = [(i, x) for i, x in enumerate(c.contigs(a)) if x[2] >= W]
                i, x = rows[int(rng.integers(len(rows)))]
                s = int(rng.integers(x[2] - W + 1))
                want = full[a][x[3] + s:x[3] + s + W]
                if k % 3:
                    got = c.fetch(a, i, s, W).cpu().numpy()
                else:
                    got = c.windows(torch.tensor([a]), torch.tensor([x[3] + s]), W)[0].cpu().numpy()
                if not np.array_equal(got, want):
                    bad.append((t, k, a, i, s, W))
        except Exception as e:
            bad.append((t, repr(e)))

    ts = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad, bad[:5]


@pytest.mark.gpu
def test_noalloc_short_q16k_calls_share_nothing(fx, oracle_ref):
    """pv_windows_hip_noalloc at q16k with one window of at most a block, on three streams at once: no call uses the
    scratch array, so each row is its own."""
    import panvram_amd
    from panvram_amd import _native as N
    c = panvram_amd.Cohort.open(fx["dirs"]["q16k"], device="cuda", dataset="q16k", reference=fx["ref"])
    full = [O.Archive(f"{fx['dirs']['q16k']}/{nm}.q16k.rr3").full(oracle_ref) for nm in c.names]
    rng = np.random.default_rng(9)
    calls = []
    for k in range(90):
        a, W = int(rng.integers(len(c))), (1, 700, 16384)[k % 3]
        s = int(rng.integers(len(full[a]) - W + 1))
        calls.append((a, s, W, torch.tensor([a], device="cuda"), torch.tensor([s], device="cuda"),
                      torch.empty((1, W), dtype=torch.uint8, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")))
    streams = [torch.cuda.Stream() for _ in range(3)]
    torch.cuda.synchronize()
    err = N.errbuf()
    for k, (a, s, W, ta, ts, out, status) in enumerate(calls):
        assert N.lib().pv_windows_hip_noalloc(c._Dref, ta.data_ptr(), ts.data_ptr(), 1, W, None, 0, 1, out.data_ptr(), status.data_ptr(),
                                              streams[k // 3 % 3].cuda_stream, err, len(err)) == 0, err.value
    torch.cuda.synchronize()
    for a, s, W, _, _, out, status in calls:
        assert int(status) == 0 and np.array_equal(out[0].cpu().numpy(), full[a][s:s + W]), (a, s, W)


@pytest.mark.gpu
@pytest.mark.parametrize("ds,n", [("q4k", 8192 + 100), ("q16k", 1024 + 100)])
def test_first_large_call_on_a_busy_stream_returns(fx, oracle_ref, ds, n):
    """The first calls on a stream that make side streams return while earlier work still runs there (a spin kernel of
    about half a second), and the bytes are right; so are those of later calls, which find the stream dry."""
    import panvram_amd
    from panvram_amd import _native as N
    c = panvram_amd.Cohort.open(fx["dirs"][ds], device="cuda", dataset=ds, reference=fx["ref"])
    L, err, W = N.lib(), N.errbuf(), 300
    arcs = [O.Archive(f"{fx['dirs'][ds]}/{nm}.{ds}.rr3") for nm in c.names]
    rng = np.random.default_rng(3)
    asm = rng.integers(0, len(c), n)
    start = np.array([rng.integers(0, arcs[a].nbases - W) for a in asm])
    want = O.windows(arcs, oracle_ref, asm, start, W)
    ta, ts = torch.from_numpy(asm).cuda(), torch.from_numpy(start).cuda()
    wb = int(L.pv_windows_work_bytes(c._Dref, n, W))
    work = [torch.empty(wb, dtype=torch.uint8, device="cuda") for _ in range(2)]
    out = [torch.empty((n, W), dtype=torch.uint8, device="cuda") for _ in range(6)]
    status = torch.zeros(1, dtype=torch.int32, device="cuda")
    warm, busy = torch.cuda.Stream(), torch.cuda.Stream()

    def call(stream, k, w):
        assert L.pv_windows_hip(c._Dref, ta.data_ptr(), ts.data_ptr(), n, W, None, 0, 1, out[k].data_ptr(), status.data_ptr(),
                                work[w].data_ptr(), wb, stream.cuda_stream, err, len(err)) == 0, err.value

    torch.cuda.synchronize()
    call(warm, 0, 0)                                # the kernels are loaded
    with torch.cuda.stream(busy):
        torch.cuda._sleep(1000)
        torch.cuda.synchronize()
        t = time.perf_counter()
        torch.cuda._sleep(1_000_000)
        torch.cuda.synchronize()
        ticks = int(1_000_000 * 0.5 / (time.perf_counter() - t))
        torch.cuda._sleep(ticks)
        done = torch.cuda.Event()
        done.record()
    t = time.perf_counter()
    for k in (1, 2, 3):
        call(busy, k, 1)
    took = time.perf_counter() - t
    assert not done.query() and took < 0.25, took
    torch.cuda.synchronize()
    for k in (4, 5):                                # (the stream is dry: the trial is made here)
        call(busy, k, 1)
        torch.cuda.synchronize()
    assert int(status) == 0
    for x in out:
        assert np.array_equal(x.cpu().numpy(), want)


@pytest.mark.gpu
@pytest.mark.parametrize("ds,n", [("q4k", 8192 + 100), ("q16k", 1024 + 100)])
def test_large_calls_of_threads_equal_oracle(fx, oracle_ref, ds, n):
    """Three threads whose large calls share a stream, from the first call on it (one of them tries and replaces the side
    streams while the others use them), on several streams in turn, so that some share a hardware queue with theirs."""
    import panvram_amd
    c = panvram_amd.Cohort.open(fx["dirs"][ds], device="cuda", dataset=ds, reference=fx["ref"])
    arcs = [O.Archive(f"{fx['dirs'][ds]}/{nm}.{ds}.rr3") for nm in c.names]
    rng, W, jobs = np.random.default_rng(5), 300, []
    for _ in range(3):
        asm = rng.integers(0, len(c), n)
        start = np.array([rng.integers(0, arcs[a].nbases - W) for a in asm])
        jobs.append((torch.from_numpy(asm).cuda(), torch.from_numpy(start).cuda(), torch.from_numpy(O.windows(arcs, oracle_ref, asm, start, W)).cuda()))
    streams = [torch.cuda.Stream() for _ in range(5)]
    torch.cuda.synchronize()
    bad, meet = [], threading.Barrier(3)

    def work(t):
        try:
            a, s, want = jobs[t]
            for st in streams:
                with torch.cuda.stream(st):
                    meet.wait(60)
                    for k in range(5):
                        if not torch.equal(c.windows(a, s, W, check=k % 2 == 0), want):
                            bad.append((t, k))
        except Exception as e:
            bad.append((t, repr(e)))
            meet.abort()

    ts = [threading.Thread(target=work, args=(t,)) for t in range(3)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad, bad[:5]
