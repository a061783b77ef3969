"""The forms of a ragged batch and what autotuning chooses in them: the groups of tiles (every problem has one), whose
FP32 passes may round at every step or once per pass, and the persistent launch (an explicit configuration, or a
problem whose shifts no tile holds), against the oracle's restatement."""
import numpy as np
import pytest

import bkma_amd as B
import oracle as O

pytestmark = pytest.mark.gpu


def _batch(dtype, specs, **kw):
    import torch
    t = torch.float64 if dtype == B.F64 else torch.float32
    arrays = [torch.zeros((n0, n1, n2), dtype=t, device="cuda") for n0, n1, n2, _ in specs]
    params = [B.make_params(n0, n1, n2, dt=dt, minRealVx=-1, maxRealVx=1) for n0, n1, n2, dt in specs]
    batch = B.AdvBatch(arrays, params, dtype, **kw)
    info = batch.describe()
    print(info, flush=True)
    for j, a in enumerate(arrays):
        B.fill_uniform(a, 900 + j)
    torch.cuda.synchronize()
    return batch, info, arrays, [a.cpu().numpy() for a in arrays]


def _check(batch, arrays, refs, specs, dtype, nsteps, ns, graph=True):
    import torch
    batch.run(nsteps, graph=graph)
    torch.cuda.synchronize()
    _ = arrays[0].clone().sum().item()  # eager work between the runs
    for j, (a, r, (n0, n1, n2, dt)) in enumerate(zip(arrays, refs, specs)):
        po = O.make_params(n0, n1, n2, dt=dt, minRealVx=-1, maxRealVx=1)
        if dtype == B.F64:
            O.advect_f64(r, po, nsteps)
        else:
            O.advect_f32_blocked(r, po, nsteps, ns)
        assert np.array_equal(a.cpu().numpy(), r), (nsteps, j, specs[j])


# Whole lines and segments, strips and LDS tiles; the second list holds large shifts, which few steps fit.
TILES = [[(300, 640, 8, 1e-3), (50, 100, 1, 2e-3), (200, 1000, 4, 1e-3), (9, 6001, 2, 1e-3)],
         [(64, 8192, 8, 2e-3), (20, 16384, 1, 1e-3), (40, 640, 64, 1e-3)]]


@pytest.mark.parametrize("specs", TILES, ids=["small_shifts", "large_shifts"])
@pytest.mark.parametrize("dtype", [B.F64, B.F32], ids=["f64", "f32"])
def test_autotuned_tiles(cuda, dtype, specs):
    batch, info, arrays, refs = _batch(dtype, specs, autotune=True)
    assert info["grid"] > 0 and info["steps_per_pass"] in ((1,) if dtype == B.F64 else (1, 2, 3, 4, 8, 16, 32))
    for nsteps in (37, 1, 37):
        _check(batch, arrays, refs, specs, dtype, nsteps, info["steps_per_pass"])
    batch.close()


# Whole lines, chained segments, and one problem whose shifts (-410 to 358 cells) exceed its segments of 1024 rows less
# the halos, which then are not chained: an item each.
PERSISTENT = [(3, 8192, 8, 2e-3), (2, 16384, 1, 1e-3), (4, 640, 64, 1e-3), (5, 100, 1, 2e-3), (16, 16384, 8, 2.5e-2)]


@pytest.mark.parametrize("threads", [256, 1024])
@pytest.mark.parametrize("dtype", [B.F64, B.F32], ids=["f64", "f32"])
def test_persistent_graphs_and_unchained_segments(cuda, dtype, threads):
    """Runs of more and fewer steps than a graph holds (32), replayed, and without graphs."""
    budget = 65536 if dtype == B.F64 else 32768
    batch, info, arrays, refs = _batch(dtype, PERSISTENT, config=(budget, threads, 1))
    assert info["lds_budget"] == budget and info["steps_per_pass"] == 1
    assert info["items"] - info["segmented_items"] == 5 and info["segmented_items"] > 16 * 16384 // 256
    for nsteps, graph in ((33, True), (2, True), (33, True), (3, False)):
        _check(batch, arrays, refs, PERSISTENT, dtype, nsteps, 1, graph)
    batch.close()


def test_graphs_end_with_a_pass(cuda):
    """Three steps per pass: a run of more steps than a graph holds makes the same passes with graphs as without."""
    specs = [(4, 640, 8, 1e-3), (2, 16384, 1, 1e-3)]
    for graph in (True, False):
        batch, info, arrays, refs = _batch(B.F32, specs, config=(98304, 256, 3))
        _check(batch, arrays, refs, specs, B.F32, 70, 3, graph)
        batch.close()


@pytest.mark.parametrize("dtype", [B.F64, B.F32], ids=["f64", "f32"])
def test_persistent_autotuned(cuda, dtype):
    """A shift of 2000 cells leaves a tile's segment too few rows, so the batch stays with the persistent launch and its
    own candidates."""
    specs = [(3, 20000, 1, 0.1), (30, 6000, 2, 1e-3), (12, 300, 8, 1e-3)]
    batch, info, arrays, refs = _batch(dtype, specs, autotune=True)
    assert info["lds_budget"] in (32768, 65536, 98304, B.query_lds_bytes() - 1024) and 1 <= info["steps_per_pass"] <= 4
    for nsteps in (5, 33, 5):
        _check(batch, arrays, refs, specs, dtype, nsteps, info["steps_per_pass"])
    batch.close()


@pytest.mark.parametrize("autotune", [False, True], ids=["default", "autotuned"])
@pytest.mark.parametrize("dtype", [B.F64, B.F32], ids=["f64", "f32"])
def test_short_and_long_runs_in_turn(cuda, dtype, autotune):
    """Many small problems: runs of a step or two take the persistent launch, longer ones the groups."""
    specs = [(20 + 3 * j, 64 * (1 + j % 11), (1, 8, 64)[j % 3], 5e-4 + 4e-5 * j) for j in range(30)]
    batch, info, arrays, refs = _batch(dtype, specs, autotune=autotune)
    for nsteps in (1, 2, 3, 5, 1, 34, 2, 1):
        _check(batch, arrays, refs, specs, dtype, nsteps, info["steps_per_pass"])
    batch.close()
