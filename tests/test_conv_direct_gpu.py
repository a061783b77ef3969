"""The FP64 and FP32 Conv1d modes over the forms that conv_direct.hip chooses: channels per lane or per thread,
matrix cores, tiles that the row does not fill, chunks of several tiles per owner, rows and arrays off 16-byte
boundaries, kernels as long as the row.  FP64 is bit-identical to the oracle; FP32 stays within the bound of an
FP32 sum of n = C K products in any order, (n + 2) 2^-24 (sum |w||x| + |bias|) per output."""
import numpy as np
import pytest

import bkma_amd as B
import oracle as O

pytestmark = pytest.mark.gpu

# (B, C, L, K)
SHAPES = [(5, 1, 64, 1), (7, 6, 256, 5), (3, 5, 2001, 11), (600, 7, 700, 5), (2, 9, 128, 3), (2, 11, 130, 6),
          (2, 12, 131, 3), (1, 13, 65, 1), (2, 16, 1030, 4), (2, 17, 64, 64), (1, 17, 300, 2), (300, 33, 333, 7),
          (3, 64, 700, 9), (2, 65, 90, 3), (2, 128, 4100, 5), (1, 256, 90, 7), (1, 280, 70, 5), (600, 32, 132, 3)]


def _run(mode, shape, offset=0):
    import torch
    Bn, C, L, K = shape
    f32 = mode == B.CONV_F32
    npdt = np.float32 if f32 else np.float64
    rng = np.random.default_rng(C * 1000 + K)
    x = rng.standard_normal((Bn, C, L)).astype(npdt)
    w = (rng.standard_normal((C, C, K)) / np.sqrt(C * K)).astype(npdt)
    b = (0.1 * rng.standard_normal(C)).astype(npdt)
    buf = torch.zeros(x.size + offset, dtype=torch.float32 if f32 else torch.float64, device="cuda")
    tx = buf[offset:].view(Bn, C, L)
    tx.copy_(torch.from_numpy(x))
    plan = B.Conv1dPlan(mode, B.F32 if f32 else B.F64, Bn, C, L, K, torch.from_numpy(w).cuda(),
                        torch.from_numpy(b).cuda())
    plan.run(tx)
    torch.cuda.synchronize()
    got = tx.cpu().numpy()
    assert np.array_equal(got[:, :, L - K + 1:], x[:, :, L - K + 1:])
    ref = x.astype(np.float64)
    O.conv_torch_f64(ref, w.astype(np.float64), b.astype(np.float64))
    return got, ref, x, w, b


@pytest.mark.parametrize("offset", [0, 1], ids=["aligned", "off_by_one"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_f64_bit_exact(cuda, shape, offset):
    got, ref, *_ = _run(B.CONV_F64, shape, offset)
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("offset", [0, 1], ids=["aligned", "off_by_one"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_f32_within_its_sum_bound(cuda, shape, offset):
    got, ref, x, w, b = _run(B.CONV_F32, shape, offset)
    Bn, C, L, K = shape
    S = np.abs(x).astype(np.float64)
    O.conv_torch_f64(S, np.abs(w).astype(np.float64), np.abs(b).astype(np.float64))
    n = L - K + 1
    err = np.abs(got[:, :, :n].astype(np.float64) - ref[:, :, :n])
    assert np.all(err <= (C * K + 2) * 2.0 ** -24 * S[:, :, :n])


@pytest.mark.parametrize("mode,shape", [(B.CONV_F32, (2, 20, 150, 3)), (B.CONV_F32, (2, 5, 150, 3)),
                                        (B.CONV_F64, (2, 20, 150, 3)), (B.CONV_F64, (2, 5, 150, 3))],
                         ids=["f32_matrix", "f32_valu", "f64_lane", "f64_valu"])
def test_values_that_are_not_finite_stay_in_their_windows(cuda, mode, shape):
    """An infinite input reaches the outputs whose window holds it, in every channel, and no other."""
    import torch
    Bn, C, L, K = shape
    f32 = mode == B.CONV_F32
    tdt = torch.float32 if f32 else torch.float64
    x = torch.ones(shape[:3], dtype=tdt, device="cuda")
    x[0, 2, 70] = float("inf")
    w = torch.full((C, C, K), 0.5, dtype=tdt, device="cuda")
    B.Conv1dPlan(mode, B.F32 if f32 else B.F64, Bn, C, L, K, w, torch.zeros(C, dtype=tdt, device="cuda")).run(x)
    torch.cuda.synchronize()
    inf = torch.isinf(x[:, :, :L - K + 1]).cpu().numpy()
    want = np.zeros_like(inf)
    want[0, :, 70 - K + 1:71] = True
    assert np.array_equal(inf, want) and not torch.isnan(x).any()


# Three blocks of 16 channels (FP32, 33 to 48) up to the longest kernel of the form and beyond it; channel counts
# that no number of channels per thread divides.
THREE_BLOCKS = [(3, 33, 70, 1), (200, 40, 301, 3), (2, 48, 1030, 5), (1, 47, 400, 64), (1, 48, 400, 65)]
ODD = [(300, 7, 300, 5), (40, 11, 513, 3), (9, 13, 129, 2)]


@pytest.mark.parametrize("mode,shape", [(B.CONV_F32, s) for s in THREE_BLOCKS + ODD[:2]] + [(B.CONV_F64, s) for s in ODD],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_channel_splits(cuda, mode, shape):
    got, ref, x, w, b = _run(mode, shape)
    if mode == B.CONV_F64:
        assert np.array_equal(got, ref)
        return
    Bn, C, L, K = shape
    S = np.abs(x).astype(np.float64)
    O.conv_torch_f64(S, np.abs(w).astype(np.float64), np.abs(b).astype(np.float64))
    n = L - K + 1
    err = np.abs(got[:, :, :n].astype(np.float64) - ref[:, :, :n])
    assert np.all(err <= (C * K + 2) * 2.0 ** -24 * S[:, :, :n])


# Around the channel counts that leave the matrix cores (12, 17 to 21), kernels beyond 1024 among them, and tiles of
# 128, 64 and 32 columns on work-groups that they fill unevenly.
FORMS = [(9, 12, 300, 3), (1, 12, 1100, 1030), (4, 17, 200, 5), (3, 21, 130, 1), (3, 22, 131, 3), (1, 20, 1060, 1025),
         (70, 128, 1000, 2), (344, 64, 190, 1), (5, 99, 300, 3), (1, 300, 40, 3)]


@pytest.mark.parametrize("shape", FORMS, ids=lambda s: "x".join(map(str, s)))
def test_f32_forms_within_their_sum_bound(cuda, shape):
    got, ref, x, w, b = _run(B.CONV_F32, shape)
    Bn, C, L, K = shape
    S = np.abs(x).astype(np.float64)
    O.conv_torch_f64(S, np.abs(w).astype(np.float64), np.abs(b).astype(np.float64))
    n = L - K + 1
    err = np.abs(got[:, :, :n].astype(np.float64) - ref[:, :, :n])
    assert np.all(err <= (C * K + 2) * 2.0 ** -24 * S[:, :, :n])
