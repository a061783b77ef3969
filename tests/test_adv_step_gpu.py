"""GPU parity of the whole-array advection step that AdaptiveWg (LDS scratch) and NDRange calls take: bit-identical
to the oracle's executors for FP64 and FP32 storage in the register form (64 and 128 columns, one shift and two
shifts per slab), the LDS tiles, and the shapes around both that stay with the executors' own kernels; values that
are not finite stay where the six taps put them."""
import numpy as np
import pytest

import bkma_amd as B
import oracle as O

pytestmark = pytest.mark.gpu

# (n0, n1, n2, dt * n1, minRealVx, maxRealVx, minRealX)
CASES = [
    (1024, 64, 64, 0.9, -1.0, 1.0, 0.0),     # register form, 64 columns, shortest line
    (600, 100, 128, 2.9, -1.0, 1.0, 0.0),    # 128 columns, shifts up to 3
    (1300, 64, 64, 1.0, -2.5, 2.5, 0.1),     # slabs whose rows round to two shifts
    (1301, 64, 128, 1.0, -2.5, 2.5, 0.1),
    (1300, 100, 64, 3.2, -1.0, 1.0, 0.0),    # a shift beyond the register form: tiles
    (1030, 64, 65, 1.0, -1.0, 1.0, 0.0),     # columns that do not fill a wavefront: tiles
    (5, 2049, 3, 1.0, -1.0, 1.0, 0.0),
    (100, 16, 1, 0.016, -1.0, 1.0, 0.0),
    (2, 5120, 4, 5.0, -1.0, 1.0, 0.0),       # longest whole-line tile
    (2, 5121, 4, 5.0, -1.0, 1.0, 0.0),       # beyond it: the executor's kernel
    (40, 15, 5, 1.0, -1.0, 1.0, 0.0),        # below the shortest: the executor's kernel
    (6, 64, 5, 31.0, -1.0, 1.0, 0.0),        # shifts of half a line: the executor's kernel
]


@pytest.mark.parametrize("impl", ["adaptivewg", "ndrange"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:3])) + f"-s{c[3]}-v{c[4]}")
@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
def test_step_bit_exact(cuda, dtype, case, impl):
    import torch
    n0, n1, n2, dtn, vmin, vmax, x0 = case
    if impl == "ndrange" and n1 > 1024:
        pytest.skip("NDRange lines have at most 1024 rows")
    kw = dict(dt=dtn / n1, minRealVx=vmin, maxRealVx=vmax, minRealX=x0, maxRealX=x0 + 1)
    p, po = B.make_params(n0, n1, n2, **kw), O.make_params(n0, n1, n2, **kw)
    host = O.uniform(n0 * n1 * n2, 31 + n1, dtype).reshape(n0, n1, n2)
    d = torch.from_numpy(host).cuda()
    o = B.create_optim_params(n0, n1, n2, pref_wg_size=64, elem_size=host.itemsize)
    for _ in range(3):
        if impl == "adaptivewg":
            B.adv_run(B.ADAPTIVE_WG, d, p, o)
        else:
            B.adv_run(B.ND_RANGE, d, p)
    torch.cuda.synchronize()
    ref = host.copy()
    (O.advect_f64 if dtype == np.float64 else O.advect_f32_plain)(ref, po, 3)
    assert np.array_equal(d.cpu().numpy(), ref)


@pytest.mark.parametrize("case", [CASES[0], CASES[2], CASES[6]], ids=["one_shift", "two_shifts", "tiles"])
def test_step_keeps_values_that_are_not_finite_in_place(cuda, case):
    import torch
    n0, n1, n2, dtn, vmin, vmax, x0 = case
    kw = dict(dt=dtn / n1, minRealVx=vmin, maxRealVx=vmax, minRealX=x0, maxRealX=x0 + 1)
    p, po = B.make_params(n0, n1, n2, **kw), O.make_params(n0, n1, n2, **kw)
    host = O.uniform(n0 * n1 * n2, 5).reshape(n0, n1, n2)
    host[:, n1 // 3, ::2] = np.inf
    host[:, n1 - 1, 1::2] = np.nan
    d = torch.from_numpy(host).cuda()
    B.adv_run(B.ADAPTIVE_WG, d, p, B.create_optim_params(n0, n1, n2, pref_wg_size=128))
    ref = host.copy()
    O.advect_f64(ref, po, 1)
    assert np.array_equal(d.cpu().numpy(), ref, equal_nan=True)
