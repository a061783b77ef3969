"""The autotuner's choice by run length: which of the fastest tile plan and the fastest other plan takes short and long
runs (on the host, from times), and that a plan made of both has the results of its passes at every length."""
import ctypes
import os

import numpy as np
import pytest

import bkma_amd as B
import oracle as O

PROBES = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "libbkma_probes.so")
ANY = 2 ** 64 - 1


def _choose(t, o, shared):
    B.lib()  # first: the probes share its HIP runtime
    P = ctypes.CDLL(PROBES)
    P.probe_choose_runs.restype = ctypes.c_longlong
    out = (ctypes.c_int * 2)()
    n = len(t)
    up_to = P.probe_choose_runs((ctypes.c_float * n)(*t), (ctypes.c_float * n)(*o), n, ctypes.c_ulonglong(shared), out)
    return bool(out[0]), bool(out[1]), up_to


def _steps():
    B.lib()
    P = ctypes.CDLL(PROBES)
    n = -1 - ctypes.CDLL(PROBES).probe_choose_runs(None, None, 0, ctypes.c_ulonglong(0), None)
    s = (ctypes.c_ulonglong * n)()
    P.probe_run_steps(s)
    return list(s)


def _times(staging, step, passes=None):
    """Runs of one pass of any length (passes = None), or of passes of `passes` steps."""
    return [staging * (1 if passes is None else -(-n // passes)) + step * n for n in _steps()]


def test_choices():
    # the headline's FP32 times: strips 20 steps 8.5 ms and 50 steps 17.8, pairs 1.95 ms per pass of five
    strips, pairs = _times(2.4, 0.307), _times(1.35, 0.12, 5)
    assert _choose(strips, pairs, 5) == (False, False, 0)
    # where the results are the same, pairs take the short runs only
    short, long_, up_to = _choose(strips, pairs, ANY)
    assert (short, long_) == (False, True) and 20 <= up_to <= 48
    # strips ahead from the second pass of the pairs on: pairs for a pass only
    strips = _times(0.6, 0.05)
    assert _choose(strips, _times(0.3, 0.05, 5), 5) == (False, True, 5)
    # one plan ahead at all lengths, and level ones: no split
    assert _choose(strips, [2 * x for x in strips], ANY) == (True, True, 0)
    assert _choose([2 * x for x in strips], strips, 5) == (False, False, 0)
    assert _choose(strips, [x * (1.001 if i % 2 else 0.999) for i, x in enumerate(strips)], ANY)[2] == 0
    # tiles for the short runs, as far as both plans make one pass of them
    assert _choose(_times(0.1, 0.19), _times(1.0, 0.02, 8), 8) == (True, False, 5)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [B.F64, B.F32], ids=["f64", "f32"])
def test_lines_in_registers_take_long_passes(cuda, dtype):
    """LINE_SHFL candidates differ in their steps per pass only, which pay their staging a tenth or so apart."""
    plan = B.AdvPlan(B.make_params(1 << 17, 1024, 1, dt=1e-3, minRealVx=-1, maxRealVx=1), dtype, autotune=True)
    cfg, name = plan.describe()
    plan.close()
    assert name.startswith("line_shfl<") and cfg.steps_per_pass == 256


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [B.F64, B.F32], ids=["f64", "f32"])
@pytest.mark.parametrize("shape", [(1024, 160, 64), (130, 256, 1), (6, 20000, 4)], ids=lambda s: "x".join(map(str, s)))
def test_autotuned_plans_at_every_length(cuda, dtype, shape):
    import torch
    p, po = (m.make_params(*shape, dt=1.5 / shape[1], minRealVx=-1, maxRealVx=1) for m in (B, O))
    plan = B.AdvPlan(p, dtype, autotune=True)
    cfg, name = plan.describe()
    print(name, flush=True)
    host = O.uniform(int(np.prod(shape)), 8, np.float64 if dtype == B.F64 else np.float32).reshape(shape)
    for n in (1, 2, 4, 5, 6, 9, 33):
        d = torch.from_numpy(host).cuda()
        plan.run(d, n)
        ref = host.copy()
        if dtype == B.F64:
            O.advect_f64(ref, po, n)
        else:
            O.advect_f32_blocked(ref, po, n, max(1, cfg.steps_per_pass))
        assert np.array_equal(d.cpu().numpy(), ref), n
    plan.close()
