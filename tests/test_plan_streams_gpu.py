"""Runs of one plan on several arrays at a time, on several streams, in several graphs and from several threads: the
buffers that a run writes belong to its stream or capture, so each array gets what a run alone gives it."""
import threading

import pytest

import bkma_amd as B

pytestmark = pytest.mark.gpu

# mode, (B, C, L, K): several tiles per row and several owners in a row (matrix, lane and VALU forms)
CONVS = [(B.CONV_F32, (64, 128, 4096, 5)), (B.CONV_F64, (16, 33, 4096, 5)), (B.CONV_F64, (64, 4, 4096, 7)),
         (B.CONV_F32, (64, 6, 4096, 7))]


def _conv(mode, shape):
    import torch
    Bn, C, L, K = shape
    t, code = (torch.float32, B.F32) if mode == B.CONV_F32 else (torch.float64, B.F64)
    g = torch.Generator(device="cuda").manual_seed(C)
    r = lambda *s: torch.randn(*s, generator=g, dtype=t, device="cuda")  # noqa: E731
    plan = B.Conv1dPlan(mode, code, Bn, C, L, K, r(C, C, K) / (C * K) ** 0.5, r(C))
    return plan, lambda n: [r(Bn, C, L) for _ in range(n)]


def _alone(run, arrays):
    """What each array is after run() by itself on the current stream."""
    import torch
    out = []
    for a in arrays:
        b = a.clone()
        run(b)
        torch.cuda.synchronize()
        out.append(b)
    return out


def _check_streams(run, arrays, streams, rounds=3):
    import torch
    want = _alone(run, arrays)
    for _ in range(rounds):
        got = [a.clone() for a in arrays]
        torch.cuda.synchronize()
        for a, s in zip(got, streams):
            with torch.cuda.stream(s):
                run(a)
        torch.cuda.synchronize()
        assert all(torch.equal(a, w) for a, w in zip(got, want))


def _check_graphs(run, arrays, rounds=3):
    """A graph for each array, captured in turn, replayed beside each other and beside eager runs."""
    import torch
    want = _alone(run, arrays)
    bufs, graphs = [a.clone() for a in arrays], []
    for b in bufs:
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            run(b)
        graphs.append(g)
    streams = [torch.cuda.Stream() for _ in bufs]
    for _ in range(rounds):
        for b, a in zip(bufs, arrays):
            b.copy_(a)
        eager = arrays[0].clone()
        torch.cuda.synchronize()
        for g, s in zip(graphs, streams):
            with torch.cuda.stream(s):
                g.replay()
        run(eager)
        torch.cuda.synchronize()
        assert torch.equal(eager, want[0]) and all(torch.equal(b, w) for b, w in zip(bufs, want))


def _check_threads(run, arrays):
    import torch
    want = _alone(run, arrays)
    got = [a.clone() for a in arrays]
    torch.cuda.synchronize()

    def work(a):
        with torch.cuda.stream(torch.cuda.Stream()):
            run(a)

    ts = [threading.Thread(target=work, args=(a,)) for a in got]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    torch.cuda.synchronize()
    assert all(torch.equal(a, w) for a, w in zip(got, want))


@pytest.mark.parametrize("case", CONVS, ids=lambda c: f"{'f32' if c[0] == B.CONV_F32 else 'f64'}-{'x'.join(map(str, c[1]))}")
def test_conv(cuda, case):
    import torch
    plan, inputs = _conv(*case)
    arrays = inputs(12)  # more streams than buffers: the others take whole rows
    _check_streams(plan.run, arrays, [torch.cuda.Stream() for _ in arrays])
    _check_graphs(plan.run, arrays[:3])
    _check_threads(plan.run, arrays[:4])


# (n0, n1, n2), dt * n1, what: strips and LDS segments through halo snapshots, large shifts through a second array (the
# first stream) and through snapshots (the others), whole lines, column pairs beside strips, old LINE_LDS segments
PLANS = [((64, 9000, 6), 3.0, "strip"), ((16, 20000, 4), 100.0, "regs"), ((200, 500, 3), 2.0, "whole"),
         ((1024, 160, 64), 1.0, "pair"), ((8, 9000, 6), 3.0, "old")]


@pytest.mark.parametrize("case", PLANS, ids=lambda c: f"{c[2]}-{'x'.join(map(str, c[0]))}")
@pytest.mark.parametrize("dtype", [B.F64, B.F32], ids=["f64", "f32"])
def test_advection(cuda, dtype, case):
    import torch
    (n0, n1, n2), s, what = case
    p = B.make_params(n0, n1, n2, dt=s / n1, minRealVx=-1.0, maxRealVx=1.0)
    c = None
    if what in ("strip", "regs", "old"):
        c = B.TunedConfig()
        c.strategy, c.prefetch, c.steps_per_pass = B.STRATEGY_LINE_LDS, {"strip": 6, "regs": 5, "old": 0}[what], 3
        c.seg_rows = 500 if what == "old" else 0
    plan = B.AdvPlan(p, dtype, config=c)
    name = plan.describe()[1]
    print(name, flush=True)
    assert ("seg" in name) == (what in ("strip", "regs", "old"))
    t = torch.float64 if dtype == B.F64 else torch.float32
    arrays = [torch.rand((n0, n1, n2), dtype=t, device="cuda") for _ in range(10)]  # two streams more than buffers
    for steps in (6, 7):
        run = lambda a: plan.run(a, steps)  # noqa: B023, E731
        _check_streams(run, arrays, [torch.cuda.Stream() for _ in arrays], rounds=2)
    _check_graphs(run, arrays[:3])
    _check_threads(run, arrays[:4])


def test_second_array_also_holds_the_snapshots(cuda):
    """Large shifts: the plan keeps one array's size, not the halos' (0.7 of it here) beside it."""
    import torch
    p = B.make_params(64, 262144, 4, dt=1e-3, minRealVx=-1.0, maxRealVx=1.0)
    size = 64 * 262144 * 4 * 4
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    plan = B.AdvPlan(p, B.F32)
    taken = free - torch.cuda.mem_get_info()[0]
    assert "seg" in plan.describe()[1] and 0.5 * size < taken < 1.2 * size
    plan.close()


def test_conv_runs_allocate_nothing(cuda):
    """On whatever stream, and in a capture."""
    import torch
    plan, inputs = _conv(B.CONV_F32, (256, 64, 4096, 33))
    arrays = inputs(6)
    streams = [torch.cuda.Stream() for _ in arrays]
    torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    for a, s in zip(arrays[:3], streams):
        with torch.cuda.stream(s):
            plan.run(a)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        plan.run(arrays[3])
        plan.run(arrays[3])
    for a, s in zip(arrays[4:], streams[4:]):
        with torch.cuda.stream(s):
            plan.run(a)
    torch.cuda.synchronize()
    size = 256 * 64 * 32 * 4  # of the columns that one buffer holds, at least
    assert free - torch.cuda.mem_get_info()[0] < size
