"""Ops called without ws= on several streams, host threads and graph captures at once: each has a
workspace of its own, so every result has the bits of the same call made alone."""

import threading

import numpy as np
import pytest
import torch

from llmnputest_amd import ops, synth

pytestmark = pytest.mark.gpu

# (kind, rows, N, K): prompt blocks (operands laid out in the workspace between two launches) and
# launches that split K (records and arrival counters there)
CASES = [("q4", 300, 2560, 2560), ("q8", 200, 4096, 1024), ("q4", 129, 4096, 4096),
         ("q4", 8, 2560, 8192), ("q4", 100, 512, 8192)]


def _job(case, dev, seed):
    kind, m, n, k = case
    rng = np.random.default_rng(seed)
    t = (synth.q4_tiles if kind == "q4" else synth.q8_tiles)(rng, n, k).reshape(-1)
    w = torch.from_numpy(t).to(dev)
    x = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).to(dev).to(torch.bfloat16)
    return lambda out=None: ops.gemm(w, kind, x, n // 32, k // 256, out=out)


@pytest.fixture
def jobs(dev):
    js = [_job(c, dev, 11 + i) for i, c in enumerate(CASES)]
    want = [j() for j in js]
    torch.cuda.synchronize()
    return js, want


def test_default_workspace_per_stream(jobs):
    js, want = jobs
    streams = [torch.cuda.Stream() for _ in js]
    got = [[] for _ in js]
    for s in streams:
        s.wait_stream(torch.cuda.current_stream())
    for _ in range(20):
        for j, s, g in zip(js, streams, got):
            with torch.cuda.stream(s):
                g.append(j())
    torch.cuda.synchronize()
    assert all(torch.equal(o, w) for g, w in zip(got, want) for o in g)


def test_default_workspace_per_thread(jobs):
    """Host threads that share one stream: the two launches of a call interleave with another's."""
    js, want = jobs
    got = [[] for _ in js]

    def work(i):
        for _ in range(40):
            got[i].append(js[i]())
    ts = [threading.Thread(target=work, args=(i,)) for i in range(len(js))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    torch.cuda.synchronize()
    assert all(len(g) == 40 for g in got)
    assert all(torch.equal(o, w) for g, w in zip(got, want) for o in g)


def test_default_workspace_per_capture(jobs):
    """Two graphs captured one after the other on the same stream, the later replayed first and
    both among eager calls and synchronisations."""
    js, want = jobs
    outs = [torch.empty_like(w) for w in want]
    graphs = []
    for part in (range(0, 3), range(3, len(js))):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            for i in part:
                js[i](out=outs[i])
        graphs.append(g)
    side = torch.cuda.Stream()
    for rep in range(4):
        for o in outs:
            o.fill_(float("nan"))
        side.wait_stream(torch.cuda.current_stream())
        graphs[1].replay()
        with torch.cuda.stream(side):
            graphs[0].replay()
        eager = [j() for j in js]
        torch.cuda.synchronize()
        for o, e, w in zip(outs, eager, want):
            assert torch.equal(o, w) and torch.equal(e, w), rep


def test_default_workspace_is_bounded(dev, monkeypatch):
    """A request beyond what a stream keeps is allocated for its call alone; no more than
    DEFAULT_WS_STREAMS streams of a thread keep one; a thread's go with it."""
    monkeypatch.setattr(ops, "DEFAULT_WS_BYTES", 1 << 20)
    job = _job(("q4", 300, 2560, 2560), dev, 5)
    want = job()
    s = torch.cuda.current_stream()
    kept = ops.default_workspace().buf.numel()
    assert kept >= 1 << 20
    monkeypatch.setattr(ops, "DEFAULT_WS_BYTES", 0)
    with torch.cuda.stream(torch.cuda.Stream()):
        torch.cuda.current_stream().wait_stream(s)
        got = job()
        assert ops.default_workspace().buf.numel() == 1 << 20
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    for _ in range(40):
        with torch.cuda.stream(torch.cuda.Stream()):
            ops.default_workspace()
    assert len(ops._defaults.by_stream) <= ops.DEFAULT_WS_STREAMS
    seen = []
    t = threading.Thread(target=lambda: seen.append((ops.default_workspace().buf.data_ptr(),
                                                     len(ops._defaults.by_stream))))
    t.start()
    t.join()
    assert seen[0][1] == 1


def test_capture_id(dev):
    from llmnputest_amd import _lib
    fn = _lib.lib().q4nx_stream_capture_id
    ids = []
    assert fn(torch.cuda.current_stream().cuda_stream) == 0
    for _ in range(2):
        g = torch.cuda.CUDAGraph()
        t = torch.zeros(4, device=dev)
        with torch.cuda.graph(g):
            t.add_(1)
            ids.append(fn(torch.cuda.current_stream().cuda_stream))
        assert fn(torch.cuda.current_stream().cuda_stream) == 0
    assert ids[0] and ids[1] and ids[0] != ids[1]
