"""Default plans of tiles run single steps on a plan of their own: runs of one step and of more in turn, bit for bit
against the oracle, with the name and configuration of the plan's long passes."""
import numpy as np
import pytest

import bkma_amd as B
import oracle as O

pytestmark = pytest.mark.gpu

# strips on whole lines of one and several columns, strips with LDS tiles beside them, large shifts in segments
CASES = [((50, 300, 1), 1.0), ((64, 64, 33), 1.0), ((9, 1000, 5), 3.0), ((21, 300, 6), 9.0), ((4, 20000, 4), 300.0)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[0])) + f"-s{c[1]}")
@pytest.mark.parametrize("dtype", [B.F64, B.F32], ids=["f64", "f32"])
def test_single_steps_between_longer_runs(cuda, dtype, case):
    import torch
    shape, s = case
    p, po = (m.make_params(*shape, dt=s / shape[1], minRealVx=-1, maxRealVx=1) for m in (B, O))
    plan = B.AdvPlan(p, dtype)
    cfg, name = plan.describe()
    print(name, flush=True)
    assert "line_lds<" in name and cfg.steps_per_pass > 1
    ref = O.uniform(int(np.prod(shape)), 21, np.float64 if dtype == B.F64 else np.float32).reshape(shape)
    d = torch.from_numpy(ref.copy()).cuda()
    for n in (1, 1, 5, 1, cfg.steps_per_pass + 1):
        plan.run(d, n)
        if dtype == B.F64:
            O.advect_f64(ref, po, n)
        else:
            O.advect_f32_blocked(ref, po, n, cfg.steps_per_pass)
        assert np.array_equal(d.cpu().numpy(), ref), n
    plan.close()


def test_names_are_whole(cuda):
    """An autotuned plan of strips and tiles, and another kernel for short runs: more than 128 characters."""
    plan = B.AdvPlan(B.make_params(4096, 10000, 1, dt=1e-3, minRealVx=-1, maxRealVx=1), B.F64, autotune=True)
    name = plan.describe()[1]
    plan.close()
    assert name.endswith(">") and name.count("<") == name.count(">") == name.count("+") + 1
