"""GPU parity of the strip form of LINE_LDS (TunedConfig.prefetch = 6: several steps in a wavefront's registers
between two exchanges): FP64 storage bit-identical to the oracle's FP64 steps, FP32 storage to its restatement with
one rounding per pass, at the edges of the form: every number of rows per lane, lines that wrap around their strips,
a last strip that is not full, segments, slabs whose rows round to two shifts, slabs with larger shifts beside them
(which run the LDS form in the same pass), the smallest and largest shift, columns moved 16 bytes at a time or one by
one, values that are not finite, and default plans that run few steps on the column pair."""
import numpy as np
import pytest

import bkma_amd as B
import oracle as O

pytestmark = pytest.mark.gpu


def _check(shape, dtype, nsteps, ns, explicit=True, poison=None, **kw):
    import torch
    n0, n1, n2 = shape
    p, po = B.make_params(n0, n1, n2, **kw), O.make_params(n0, n1, n2, **kw)
    host = O.uniform(n0 * n1 * n2, 29 + n1 + ns, np.float32 if dtype == B.F32 else np.float64).reshape(shape)
    for at, value in poison or ():
        host[at] = value
    d = torch.from_numpy(host).cuda()
    c = None
    if explicit:
        c = B.TunedConfig()
        c.strategy, c.prefetch, c.steps_per_pass = B.STRATEGY_LINE_LDS, 6, ns
    plan = B.AdvPlan(p, dtype, config=c)
    cfg, name = plan.describe()
    print(name, nsteps, flush=True)
    plan.run(d, nsteps)
    torch.cuda.synchronize()
    plan.close()
    ref = host.copy()
    if dtype == B.F32:
        O.advect_f32_blocked(ref, po, nsteps, cfg.steps_per_pass)
    else:
        O.advect_f64(ref, po, nsteps)
    bits = np.uint32 if dtype == B.F32 else np.uint64
    got = d.cpu().numpy()
    if poison:
        assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.isnan(ref).any()
        ok = ~np.isnan(ref)
        assert np.array_equal(got[ok].view(bits), ref[ok].view(bits))
    else:
        assert np.array_equal(got.view(bits), ref.view(bits)), np.abs(got.astype(np.float64) - ref).max()
    return cfg, name


# (n0, n1, n2, dt, steps per pass, piece of the plan's name)
CASES = [
    (40, 16, 1, 3e-3, 6, "strip4x1,whole_line"),    # the line wraps 16 times around its strip
    (7, 67, 5, 2e-3, 9, "strip4x1,whole_line"),
    (5, 300, 1, 1e-3, 20, "whole_line"),
    (300, 777, 3, 1e-3, 13, "whole_line"),
    (64, 1000, 1, 1e-3, 64, "strip6x4,whole_line"),
    (300, 1000, 4, 1e-3, 8, "strip6x3,whole_line"),
    (9, 1001, 100, 1e-3, 3, "strip"),               # 16-byte columns
    (3, 1003, 33, 1e-3, 3, "strip"),                # odd columns
    (2, 3000, 8, 1e-3, 20, "strip8x8,whole_line"),
    (2, 5000, 1, 1e-3, 30, "seg"),
    (3, 9000, 6, 5e-4, 40, "seg"),                  # four of the six columns, then two
    (2, 20011, 16, 2e-4, 5, "seg"),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:3])) + f"-dt{c[3]}-ns{c[4]}")
@pytest.mark.parametrize("dtype", [B.F64, B.F32], ids=["f64", "f32"])
def test_strip_bit_exact(cuda, dtype, case):
    n0, n1, n2, dt, ns, want = case
    _, name = _check((n0, n1, n2), dtype, 2 * ns + 1, ns, dt=dt, minRealVx=-1, maxRealVx=1)
    assert want in name and "strip" in name


@pytest.mark.parametrize("shape", [(13, 300, 6), (13, 300, 1), (13, 6000, 4), (13, 6000, 1)],
                         ids=["whole_cols", "whole_lines", "seg_cols", "seg_lines"])
@pytest.mark.parametrize("dtype", [B.F64, B.F32], ids=["f64", "f32"])
@pytest.mark.parametrize("lo,hi,parts", [(-3.5, 3.0, 1), (-5.0, 6.0, 1), (-9.0, 4.0, 2), (-8.0, 9.5, 3)])
def test_strip_shifts(cuda, dtype, shape, lo, hi, parts):
    """Shifts by halves or so around the integers, on x in [0.1, 1.1), within the strips' range and beyond it."""
    n1 = shape[1]
    _, name = _check(shape, dtype, 11, 5, dt=1.0 / n1, minRealVx=lo, maxRealVx=hi, minRealX=0.1, maxRealX=1.1)
    assert "strip" in name and name.count("|") == parts - 1


@pytest.mark.parametrize("shape", [(5, 700, 3), (3, 6000, 4)], ids=["whole", "seg"])
def test_strip_not_finite_values_stay_in_their_cone(cuda, shape):
    n0, n1, n2 = shape
    _check(shape, B.F64, 7, 7, dt=1e-3, minRealVx=-1, maxRealVx=1,
           poison=[((0, 0, 0), np.nan), ((1, n1 // 2, n2 - 1), np.inf), ((n0 - 1, n1 - 1, 1), -np.inf)])


@pytest.mark.parametrize("dtype,shape,steps", [(B.F64, (1024, 160, 64), (1, 4, 8, 9)), (B.F64, (1100, 160, 125), (4, 5)),
                                               (B.F32, (384, 160, 130), (1, 5, 6))],
                         ids=["f64-full", "f64-nearly", "f32-ragged"])
def test_default_plan_of_few_steps(cuda, dtype, shape, steps):
    """Default plans of strips where the column kernels also fill the GPU: runs on both sides of the line between
    them have the results of the plan's passes."""
    for n in steps:
        cfg, name = _check(shape, dtype, n, 1, explicit=False, dt=1e-3, minRealVx=-1, maxRealVx=1)
        assert "strip" in name and cfg.steps_per_pass >= 8


@pytest.mark.parametrize("dtype", [B.F64, B.F32], ids=["f64", "f32"])
def test_step_on_an_address_between_16_bytes(cuda, dtype):
    """One executor step (the same staging code) in an array that starts at 8 (FP32: 4) bytes past a 16-byte line."""
    import torch
    n0, n1, n2 = 9, 130, 8
    p, po = (m.make_params(n0, n1, n2, dt=1e-3, minRealVx=-1, maxRealVx=1) for m in (B, O))
    np_dt = np.float32 if dtype == B.F32 else np.float64
    host = O.uniform(n0 * n1 * n2, 3, np_dt).reshape(n0, n1, n2)
    buf = torch.zeros(n0 * n1 * n2 + 2, dtype=torch.float32 if dtype == B.F32 else torch.float64, device="cuda")
    d = buf[1:-1].view(n0, n1, n2)
    d.copy_(torch.from_numpy(host))
    o = B.create_optim_params(n0, n1, n2, pref_wg_size=64, elem_size=host.itemsize)
    B.adv_run(B.ADAPTIVE_WG, d, p, o)
    torch.cuda.synchronize()
    (O.advect_f32_plain if dtype == B.F32 else O.advect_f64)(host, po, 1)
    assert np.array_equal(d.cpu().numpy(), host) and buf[0].item() == 0 and buf[-1].item() == 0


# Tiles of many kinds and sizes: several launches per pass, and enough work that they take turns on several streams.
LANES = [(300, 1000, 4, 1e-3), (40, 6000, 1, 1e-3), (2000, 64, 2, 1e-3), (60, 777, 8, 1e-3), (100, 200, 16, 1e-3),
         (9, 3000, 33, 1e-3), (30, 6000, 2, 3e-3)]


@pytest.mark.parametrize("dtype", [B.F64, B.F32], ids=["f64", "f32"])
def test_batch_on_several_streams_stays_between_the_callers_work(cuda, dtype):
    """A long run of a batch between a copy into its arrays and one out of them, on a stream of the caller's, twice."""
    import torch
    npdt, tdt = (np.float64, torch.float64) if dtype == B.F64 else (np.float32, torch.float32)
    arrays = [torch.empty(c[:3], dtype=tdt, device="cuda") for c in LANES]
    params = [B.make_params(*c[:3], dt=c[3], minRealVx=-1, maxRealVx=1) for c in LANES]
    batch = B.AdvBatch(arrays, params, dtype)
    hosts = [O.uniform(a.numel(), 50 + j, npdt).reshape(tuple(a.shape)) for j, a in enumerate(arrays)]
    sources = [torch.from_numpy(h).cuda() for h in hosts]
    torch.cuda.synchronize()
    s, got = torch.cuda.Stream(), []
    for _ in range(2):
        with torch.cuda.stream(s):
            for a, src in zip(arrays, sources):
                a.copy_(src)
            batch.run(130, stream=s)
            got.append([a.clone() for a in arrays])
    torch.cuda.synchronize()
    batch.close()
    for j, (c, ref) in enumerate(zip(LANES, hosts)):
        po = O.make_params(*c[:3], dt=c[3], minRealVx=-1, maxRealVx=1)
        if dtype == B.F64:
            O.advect_f64(ref, po, 130)
        else:
            O.advect_f32_blocked(ref, po, 130, 1)
        for g in got:
            assert np.array_equal(g[j].cpu().numpy(), ref), j


@pytest.mark.parametrize("dtype", [B.F64, B.F32], ids=["f64", "f32"])
@pytest.mark.parametrize("n0,n1", [(5, 512), (256, 1024)])
def test_default_plan_of_few_lines(cuda, dtype, n0, n1):
    """Few contiguous lines: runs on both sides of the line between LINE_SHFL and strips, and beyond one pass."""
    for n in (32, 33, 257):
        cfg, name = _check((n0, n1, 1), dtype, n, 1, explicit=False, dt=1e-3, minRealVx=-1, maxRealVx=1)
        assert name.startswith("line_shfl<") and "strip" in name and cfg.steps_per_pass == 256


@pytest.mark.parametrize("dtype", [B.F64, B.F32], ids=["f64", "f32"])
@pytest.mark.parametrize("shape,lo,hi", [((3, 20000, 4), -100.0, 100.0), ((13, 6000, 3), -4.0, 30.0)], ids=["tiles", "both"])
@pytest.mark.parametrize("nsteps", [4, 5, 8, 12, 13])
def test_passes_through_a_second_array(cuda, dtype, shape, lo, hi, nsteps):
    """Large shifts, four steps per pass: one pass, even and odd numbers of passes, a shorter last one."""
    _, name = _check(shape, dtype, nsteps, 4, dt=1.0 / shape[1], minRealVx=lo, maxRealVx=hi)
    assert "seg" in name and ("strip" in name) == (lo == -4.0)
