"""GPU parity of the LINE_LDS form that keeps its coefficients in registers (TunedConfig.prefetch = 5): FP64
storage bit-identical to the oracle's FP64 steps, FP32 storage to its restatement with one rounding per pass, at
the edges of the tiles: row counts around the five rows of a thread, columns that do not fill a tile, lines
around the longest whole-line tile (5120 rows), segments with halos, slabs whose rows round to two shifts, and
lines too short for the form (which run the other LINE_LDS kernels)."""
import numpy as np
import pytest

import bkma_amd as B
import oracle as O

pytestmark = pytest.mark.gpu

ROWS = 5


def _config(ns):
    c = B.TunedConfig()
    c.strategy = B.STRATEGY_LINE_LDS
    c.prefetch = ROWS
    c.steps_per_pass = ns
    return c


def _check(shape, dtype, nsteps, ns, config, **kw):
    import torch
    n0, n1, n2 = shape
    p, po = B.make_params(n0, n1, n2, **kw), O.make_params(n0, n1, n2, **kw)
    host = O.uniform(n0 * n1 * n2, 17 + n1 + ns, np.float32 if dtype == B.F32 else np.float64).reshape(shape)
    d = torch.from_numpy(host).cuda()
    plan = B.AdvPlan(p, dtype, config=config)
    cfg, name = plan.describe()
    print(name, flush=True)
    assert cfg.steps_per_pass == ns
    plan.run(d, nsteps)
    torch.cuda.synchronize()
    plan.close()
    ref = host.copy()
    if dtype == B.F32:
        O.advect_f32_blocked(ref, po, nsteps, ns)
    else:
        O.advect_f64(ref, po, nsteps)
    bits = np.uint32 if dtype == B.F32 else np.uint64
    got = d.cpu().numpy()
    assert np.array_equal(got.view(bits), ref.view(bits)), np.abs(got.astype(np.float64) - ref).max()
    return name


# (n0, n1, n2, dt, steps per pass, kind of tile)
CASES = [
    (40, 16, 9, 3e-3, 6, "whole"),       # shortest line, odd columns
    (300, 17, 1, 2e-3, 4, "whole"),      # several slabs per tile, one row past three threads
    (7, 64, 5, 1e-3, 70, "whole"),       # more steps than the default pass
    (9, 999, 1, 1e-3, 3, "whole"),
    (3, 1001, 3, 2e-3, 3, "whole"),      # three of four columns per thread
    (2, 1024, 100, 1e-3, 8, "whole"),    # last column tile narrower
    (1, 130, 2, 2e-2, 5, "whole"),       # two columns, shift of ~2.6 cells
    (2, 5119, 1, 1e-3, 4, "whole"),
    (1, 5120, 4, 4e-3, 2, "whole"),      # longest whole line, shift ~20 cells
    (2, 5121, 1, 1e-3, 4, "seg"),        # just beyond it
    (2, 5200, 2, 1e-3, 5, "seg"),
    (3, 6000, 7, 3e-3, 3, "seg"),        # odd columns in two column threads
    (2, 16384, 4, 1e-3, 4, "seg"),       # shift ~16 cells
    (2, 8192, 64, 2e-3, 2, "seg"),       # several column tiles
    (2, 40001, 1, 3e-3, 3, "seg"),       # shift ~120 cells, uneven segments
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:3])) + f"-dt{c[3]}-ns{c[4]}")
@pytest.mark.parametrize("dtype", [B.F64, B.F32], ids=["f64", "f32"])
def test_tile_bit_exact(cuda, dtype, case):
    n0, n1, n2, dt, ns, kind = case
    name = _check((n0, n1, n2), dtype, 2 * ns + 1, ns, _config(ns), dt=dt, minRealVx=-1, maxRealVx=1)
    assert ("whole_line" in name) == (kind == "whole") and ",regs5," in name


@pytest.mark.parametrize("shape", [(13, 300, 1), (13, 300, 6), (13, 6000, 1), (13, 6000, 4)])
@pytest.mark.parametrize("dtype", [B.F64, B.F32], ids=["f64", "f32"])
def test_tile_rows_of_two_shifts(cuda, dtype, shape):
    """Shifts by halves from -3.5 to 2.5 on x in [0.1, 1.1): at the integers the rows round to both sides."""
    n1 = shape[1]
    _check(shape, dtype, 7, 3, _config(3), dt=1.0 / n1, minRealVx=-3.5, maxRealVx=3.0, minRealX=0.1, maxRealX=1.1)


def test_tile_too_short_lines_run_the_other_form(cuda):
    name = _check((5, 15, 3), B.F64, 5, 2, _config(2), dt=2e-3, minRealVx=-1, maxRealVx=1)
    assert name.startswith("line_lds<") and "regs" not in name
    with pytest.raises(B.BkmaUnsupported):  # which fuses at most 4 steps
        B.AdvPlan(B.make_params(5, 15, 3, dt=2e-3), B.F64, config=_config(5))


@pytest.mark.parametrize("shape,dt", [((300, 100, 100), 1e-3), ((5, 12000, 60), 2e-3), ((64, 1000, 1), 1e-3),
                                      ((3, 500, 640), 1e-3)])
@pytest.mark.parametrize("dtype", [B.F64, B.F32], ids=["f64", "f32"])
def test_default_plans(cuda, dtype, shape, dt):
    p = B.make_params(*shape, dt=dt, minRealVx=-1, maxRealVx=1)
    plan = B.AdvPlan(p, dtype)
    cfg, name = plan.describe()
    plan.close()
    assert name.startswith("line_lds<") and (",regs5," in name or ",strip" in name)
    _check(shape, dtype, 11, cfg.steps_per_pass, None, dt=dt, minRealVx=-1, maxRealVx=1)


# Whole-line and segmented tiles of every width, several problems to a launch; the last two share one.
BATCH = [(3, 8192, 8, 2e-3), (2, 16384, 1, 1e-3), (4, 640, 64, 1e-3), (5, 100, 1, 2e-3), (3, 6001, 2, 1e-3),
         (7, 33, 2, 1e-3), (2, 5200, 3, 1e-3), (40, 64, 8, 2e-3), (9, 80, 8, 1e-3)]


@pytest.mark.parametrize("graph", [True, False], ids=["graph", "eager"])
@pytest.mark.parametrize("dtype", [B.F64, B.F32], ids=["f64", "f32"])
def test_batch_of_tiles_rounds_every_step(cuda, dtype, graph):
    """The default batch fuses steps in its tiles, with the results of one step per pass, on every run: 37 steps
    (a graph of 32 and one of 5), then 1, then 37 again."""
    import torch
    tdt = torch.float64 if dtype == B.F64 else torch.float32
    arrays = [torch.empty((n0, n1, n2), dtype=tdt, device="cuda") for n0, n1, n2, _ in BATCH]
    params = [B.make_params(n0, n1, n2, dt=dt, minRealVx=-1, maxRealVx=1) for n0, n1, n2, dt in BATCH]
    batch = B.AdvBatch(arrays, params, dtype)
    assert batch.describe()["steps_per_pass"] == 1
    for j, a in enumerate(arrays):
        B.fill_uniform(a, 600 + j)
    torch.cuda.synchronize()
    refs = [a.cpu().numpy() for a in arrays]
    for nsteps in (37, 1, 37):
        batch.run(nsteps, graph=graph)
        torch.cuda.synchronize()
        for j, (n0, n1, n2, dt) in enumerate(BATCH):
            po = O.make_params(n0, n1, n2, dt=dt, minRealVx=-1, maxRealVx=1)
            if dtype == B.F64:
                O.advect_f64(refs[j], po, nsteps)
            else:
                O.advect_f32_blocked(refs[j], po, nsteps, 1)
            assert np.array_equal(arrays[j].cpu().numpy(), refs[j]), (nsteps, BATCH[j])
    batch.close()
