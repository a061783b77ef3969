"""The forms of a ragged batch and what autotuning chooses in them: the groups of tiles (every problem has one), whose
FP32 passes may round at every step or once per pass, against the oracle's restatement."""
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
