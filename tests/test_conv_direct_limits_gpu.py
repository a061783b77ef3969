"""FP64 and FP32 Conv1d modes at the most channels and the longest kernels that their LDS tiles (160 KB) hold: the last
that fits agrees with the oracle, the next is refused."""
import numpy as np
import pytest

import bkma_amd as B
import oracle as O

pytestmark = pytest.mark.gpu

# (B, C, L, K): few columns per tile and 16 of them (FP64, one channel per lane), matrix tiles 16 and 48 banks apart
LARGEST = {B.CONV_F64: [(1, 320, 40, 1), (2, 512, 40, 1), (1, 1137, 20, 1), (1, 5, 4100, 4033)],
           B.CONV_F32: [(1, 640, 33, 1), (2, 600, 130, 1), (1, 515, 40, 3), (1, 512, 70, 2), (1, 5, 8200, 8129)]}
BEYOND = {B.CONV_F64: [(1, 1139, 20, 1), (1, 5, 4100, 4034)],
          B.CONV_F32: [(1, 641, 33, 1), (1, 850, 20, 1), (1, 5, 8200, 8130)]}


def _cases(of):
    return [pytest.param(m, s, id=f"{'f64' if m == B.CONV_F64 else 'f32'}-{'x'.join(map(str, s))}") for m in of for s in of[m]]


def _plan(mode, shape, w, b):
    import torch
    return B.Conv1dPlan(mode, B.F64 if mode == B.CONV_F64 else B.F32, *shape, torch.from_numpy(w).cuda(),
                        torch.from_numpy(b).cuda())


def _weights(mode, shape):
    _, C, _, K = shape
    rng = np.random.default_rng(C + K)
    t = np.float64 if mode == B.CONV_F64 else np.float32
    return rng, (rng.standard_normal((C, C, K)) / np.sqrt(C * K)).astype(t), rng.standard_normal(C).astype(t)


@pytest.mark.parametrize("mode,shape", _cases(BEYOND))
def test_refused(cuda, mode, shape):
    _, w, b = _weights(mode, shape)
    with pytest.raises(B.BkmaUnsupported, match="C too large"):
        _plan(mode, shape, w, b)


@pytest.mark.parametrize("mode,shape", _cases(LARGEST))
def test_largest(cuda, mode, shape):
    import torch
    Bn, C, L, K = shape
    rng, w, b = _weights(mode, shape)
    x = rng.standard_normal((Bn, C, L)).astype(w.dtype)
    d = torch.from_numpy(x).cuda()
    _plan(mode, shape, w, b).run(d)
    got, ref, n = d.cpu().numpy(), x.astype(np.float64), L - K + 1
    O.conv_torch_f64(ref, w.astype(np.float64), b.astype(np.float64))
    if mode == B.CONV_F64:
        assert np.array_equal(got, ref)
        return
    bound = np.abs(x).astype(np.float64)
    O.conv_torch_f64(bound, np.abs(w).astype(np.float64), np.abs(b).astype(np.float64))
    assert np.array_equal(got[:, :, n:], x[:, :, n:])
    assert np.all(np.abs(got[:, :, :n].astype(np.float64) - ref[:, :, :n]) <= (C * K + 2) * 2.0 ** -24 * bound[:, :, :n])
