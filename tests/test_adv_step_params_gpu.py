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


# Derived fields that do not agree, x so far away that a cell is two units in the last place, shifts of many lines.
ODD = {"dx": dict(change={"dx": 1.01}), "inv_dx": dict(change={"inv_dx": 1.3}), "width": dict(change={"realWidthX": 0.5}),
       "far": dict(minRealX=2.0 ** 44, maxRealX=2.0 ** 44 + 1), "dvx": dict(change={"dvx": 300.0})}


@pytest.mark.parametrize("odd", sorted(ODD))
@pytest.mark.parametrize("impl", [B.ADAPTIVE_WG, B.ND_RANGE], ids=["adaptivewg", "ndrange"])
@pytest.mark.parametrize("shape", [(1100, 64, 64), (5, 256, 3)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
def test_parameters_that_no_regular_grid_has(cuda, dtype, shape, impl, odd):
    kw = dict(ODD[odd])
    p, po = _params(shape, change=kw.pop("change", None), dt=1.7 / shape[1], minRealVx=-1.0, maxRealVx=1.0, **kw)
    _step(shape, dtype, impl, p, po)


@pytest.mark.parametrize("dtype", [B.F64, B.F32], ids=["f64", "f32"])
def test_plans_and_batches_where_coordinates_do_not_resolve_the_cells(cuda, dtype):
    """Rows of one slab take many shifts: whole lines in LDS that evaluate every foot, no tile form (column streams
    and segments write NaN for a row outside their planned window)."""
    import torch
    shape = n0, n1, n2 = 6, 1000, 3
    p, po = _params(shape, dt=1.0 / n1, minRealVx=-1.0, maxRealVx=1.0, minRealX=2.0 ** 43, maxRealX=2.0 ** 43 + 1)
    host = O.uniform(n0 * n1 * n2, 5, np.float64 if dtype == B.F64 else np.float32).reshape(shape)
    plan = B.AdvPlan(p, dtype)
    cfg, name = plan.describe()
    assert "regs" not in name and "strip" not in name
    a, b = torch.from_numpy(host).cuda(), torch.from_numpy(host).cuda()
    plan.run(a, 3)
    batch = B.AdvBatch([b], [p], dtype)
    batch.run(3)
    torch.cuda.synchronize()
    for got, ns in ((a, cfg.steps_per_pass), (b, batch.describe()["steps_per_pass"])):
        ref = host.copy()
        if dtype == B.F64:
            O.advect_f64(ref, po, 3)
        else:
            O.advect_f32_blocked(ref, po, 3, max(1, ns))
        assert np.array_equal(got.cpu().numpy(), ref)
