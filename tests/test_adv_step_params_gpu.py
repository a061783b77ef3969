"""Executor steps (bkma_adv_run) with parameters at the ends of what the whole-array kernels cover: bit-identical to
the oracle's executors whatever the parameters."""
import numpy as np
import pytest

import bkma_amd as B
import oracle as O

pytestmark = pytest.mark.gpu


def _params(shape, change=None, **kw):
    p, po = B.make_params(*shape, **kw), O.make_params(*shape, **kw)
    for k, f in (change or {}).items():
        for q in (p, po):
            setattr(q, k, f * getattr(q, k))
    return p, po


def _step(shape, dtype, impl, p, po):
    import torch
    host = O.uniform(int(np.prod(shape)), 77, dtype).reshape(shape)
    d = torch.from_numpy(host).cuda()
    if impl == B.ADAPTIVE_WG:
        B.adv_run(impl, d, p, B.create_optim_params(*shape, pref_wg_size=64, elem_size=host.itemsize))
    else:
        B.adv_run(impl, d, p)
    got = d.cpu().numpy()
    (O.advect_f64 if dtype == np.float64 else O.advect_f32_plain)(host, po, 1)
    bits = np.uint64 if dtype == np.float64 else np.uint32
    assert np.array_equal(got.view(bits), host.view(bits))


@pytest.mark.parametrize("shift", [-4 + 2e-6, 4 - 2e-6, -3 - 2e-6, 3 - 2e-6])
@pytest.mark.parametrize("width", [64, 128])
def test_shift_that_rounds_out_of_the_column_kernels(cuda, shift, width):
    """x far from the origin: 2e-6 of a cell is less than the coordinates resolve, so that all rows of the first slab
    take the whole shift, which the column kernel has no body for."""
    shape = (1024, 64, width)
    p, po = _params(shape, dt=1.0 / 64, minRealVx=shift, maxRealVx=0.0, minRealX=2.0 ** 30, maxRealX=2.0 ** 30 + 1)
    _step(shape, np.float64, B.ADAPTIVE_WG, p, po)
