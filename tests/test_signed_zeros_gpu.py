"""Signs of zero: the reference's sum starts at 0., so six products that are all -0. give 0.  Arrays of zeros of random
signs, in which about one row in 64 of a slab at rest has six such products, through the tile forms of steps, plans
and batches, bit for bit against the oracle."""
import numpy as np
import pytest

import bkma_amd as B
import oracle as O

pytestmark = pytest.mark.gpu

# (n0, n1, n2), strategy's prefetch (5: LDS tiles, 6: strips), a piece of the plan's name
PLANS = [((4, 300, 5), 5, "regs5,whole"), ((4, 8192, 3), 5, "regs5,seg"), ((4, 100, 1), 6, "strip4"),
         ((4, 1000, 1), 6, "strip6"), ((2, 3000, 8), 6, "strip8"), ((2, 8192, 4), 6, "seg"), ((4, 1024, 6), 6, "strip")]


def _zeros(shape, dtype):
    s = O.uniform(int(np.prod(shape)), 11).reshape(shape) < 0.5
    return np.where(s, -0.0, 0.0).astype(np.float64 if dtype == B.F64 else np.float32)


def _params(shape, at_rest):
    # v = 0 in the slab n0 / 2, or in all; on x in [0.1, 1.1) its rows round to two shifts
    kw = dict(dt=1e-3, minRealVx=0.0, maxRealVx=0.0) if at_rest else dict(dt=1e-3, minRealVx=-1.0, maxRealVx=1.0,
                                                                          minRealX=0.1, maxRealX=1.1)
    return B.make_params(*shape, **kw), O.make_params(*shape, **kw)


def _same(d, host, dtype, po, executor=False):
    ref = host.copy()
    if dtype == B.F64:
        O.advect_f64(ref, po, 1)
    else:
        (O.advect_f32_plain if executor else O.advect_f32_mixed)(ref, po, 1)
    assert not np.signbit(ref[host.shape[0] // 2]).all() and np.signbit(host).any()
    assert np.array_equal(np.signbit(d.cpu().numpy()), np.signbit(ref)) and not ref.any()


@pytest.mark.parametrize("at_rest", [True, False], ids=["at_rest", "moving"])
@pytest.mark.parametrize("case", PLANS, ids=lambda c: f"{c[2]}-{'x'.join(map(str, c[0]))}")
@pytest.mark.parametrize("dtype", [B.F64, B.F32], ids=["f64", "f32"])
def test_plans(cuda, dtype, case, at_rest):
    import torch
    shape, prefetch, want = case
    p, po = _params(shape, at_rest)
    c = B.TunedConfig()
    c.strategy, c.prefetch, c.steps_per_pass = B.STRATEGY_LINE_LDS, prefetch, 2
    plan = B.AdvPlan(p, dtype, config=c)
    assert want in plan.describe()[1]
    host = _zeros(shape, dtype)
    d = torch.from_numpy(host).cuda()
    plan.run(d, 1)
    _same(d, host, dtype, po)


@pytest.mark.parametrize("dtype", [B.F64, B.F32], ids=["f64", "f32"])
@pytest.mark.parametrize("at_rest", [True, False], ids=["at_rest", "moving"])
def test_steps_and_batches(cuda, dtype, at_rest):
    import torch
    for shape in ((4, 1024, 1), (4, 300, 5), (1100, 64, 64)):
        p, po = _params(shape, at_rest)
        host = _zeros(shape, dtype)
        d, e = torch.from_numpy(host).cuda(), torch.from_numpy(host).cuda()
        B.adv_run(B.ADAPTIVE_WG, d, p, B.create_optim_params(*shape, pref_wg_size=64, elem_size=host.itemsize))
        _same(d, host, dtype, po, executor=True)
        B.AdvBatch([e], [p], dtype).run(1)
        torch.cuda.synchronize()
        _same(e, host, dtype, po)
