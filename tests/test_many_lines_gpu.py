"""Arrays whose tiles or lines need more threads than one launch may have (2^32): several launches."""
import numpy as np
import pytest

import bkma_amd as B
import oracle as O

pytestmark = pytest.mark.gpu


# (lines, cells, cells per lane): a work-group of 1024 threads per line, and 16 threads per line
@pytest.mark.parametrize("n0,n1,vec", [(2 ** 22 + 3, 4096, 4), (2 ** 28 + 5, 16, 1)], ids=["line", "row16"])
def test_more_lines_in_registers_than_a_launch_holds(cuda, n0, n1, vec):
    """LINE_SHFL over 69 and 17 GB of FP32: lines at both ends and around the end of the first launch."""
    import torch
    if torch.cuda.mem_get_info()[0] < 100 << 30:
        pytest.skip("needs 100 GB of device memory")
    p = B.make_params(n0, n1, 1, dt=0.8 / n1, minRealVx=-1.0, maxRealVx=1.0)
    c = B.TunedConfig()
    c.strategy, c.vec, c.waves_per_wg, c.steps_per_pass = B.STRATEGY_LINE_SHFL, vec, 16 if vec == 4 else 0, 2
    plan = B.AdvPlan(p, B.F32, config=c)
    d = torch.zeros((n0, n1, 1), dtype=torch.float32, device="cuda")
    rows = [0, 1, n0 // 3, n0 - 7, n0 - 6, n0 - 5, n0 - 4, n0 - 3, n0 - 2, n0 - 1]
    host = O.uniform(len(rows) * n1, 4, np.float32).reshape(len(rows), n1, 1)
    d[rows] = torch.from_numpy(host).cuda()
    plan.run(d, 2)
    got = d[rows].cpu().numpy()
    plan.close()
    del d
    torch.cuda.empty_cache()
    for k, i0 in enumerate(rows):
        po = O.make_params(1, n1, 1, dt=0.8 / n1, minRealVx=-1.0, maxRealVx=1.0)
        po.minRealVx = -1.0 + i0 * p.dvx
        ref = host[k:k + 1].copy()
        O.advect_f32_blocked(ref, po, 2, 2)
        assert np.array_equal(got[k:k + 1], ref), i0


@pytest.mark.parametrize("what", ["step", "plan"])
def test_more_slabs_than_a_launch_holds(cuda, what):
    """2^24 + 3 lines of 1000 cells, FP32 (67 GB), a work-group of 256 threads each: the first and last lines and
    those around the end of the first launch against the oracle."""
    import torch
    n0, n1 = 2 ** 24 + 3, 1000
    if torch.cuda.mem_get_info()[0] < 100 << 30:
        pytest.skip("needs 100 GB of device memory")
    p = B.make_params(n0, n1, 1, dt=1e-3, minRealVx=-1.0, maxRealVx=1.0)
    d = torch.zeros((n0, n1, 1), dtype=torch.float32, device="cuda")
    rows = [0, 1, 2 ** 22, 2 ** 23 + 5, 2 ** 24 - 2, 2 ** 24 - 1, 2 ** 24, 2 ** 24 + 1, 2 ** 24 + 2]
    host = O.uniform(len(rows) * n1, 3, np.float32).reshape(len(rows), n1, 1)
    d[rows] = torch.from_numpy(host).cuda()
    if what == "step":
        B.adv_run(B.ADAPTIVE_WG, d, p, B.create_optim_params(n0, n1, 1, pref_wg_size=256, elem_size=4))
    else:
        c = B.TunedConfig()
        c.strategy, c.prefetch, c.steps_per_pass = B.STRATEGY_LINE_LDS, 5, 2
        plan = B.AdvPlan(p, B.F32, config=c)
        assert "regs5" in plan.describe()[1] and plan.describe()[1].endswith("wg256>")
        plan.run(d, 2)
    got = d[rows].cpu().numpy()
    del d
    torch.cuda.empty_cache()
    for k, i0 in enumerate(rows):
        po = O.make_params(1, n1, 1, dt=1e-3, minRealVx=-1.0, maxRealVx=1.0)
        po.minRealVx = -1.0 + i0 * p.dvx  # the line's own velocity
        ref = host[k:k + 1].copy()
        if what == "step":
            O.advect_f32_plain(ref, po, 1)
        else:
            O.advect_f32_blocked(ref, po, 2, 2)
        assert np.array_equal(got[k:k + 1], ref), i0
