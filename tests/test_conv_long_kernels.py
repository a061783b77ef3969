"""The owners of the direct convolutions (FP64 and FP32 Conv1d modes): kernels that reach past the next tile,
K - 1 > TN, take the columns after an owner's chunk, which belong to another owner, from the copy made before the
launch; chunk bounds for tile counts up to 2^31 - 1."""
import ctypes
import os

import numpy as np
import pytest

import bkma_amd as B
import oracle as O

PROBES = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "libbkma_probes.so")


@pytest.mark.parametrize("tn", [32, 64, 128, 256])
@pytest.mark.parametrize("chunk", [1, 2, 3, 7, 64])
def test_windows_read_no_column_of_another_owner(tn, chunk):
    """On the host: no window reads a live column that another owner writes, nor past the copied columns."""
    B.lib()  # first: the probes share its HIP runtime
    P = ctypes.CDLL(PROBES)
    P.probe_conv_chunk_faults.restype = ctypes.c_longlong
    for tiles in (1, 2, 3, 8, 9):
        for k in (1, 2, tn, tn + 1, tn + 2, 2 * tn + 1, 2 * tn + 2, 5 * tn):
            assert P.probe_conv_chunk_faults(5, tiles, tn, k, chunk) == 0, (tiles, k)


@pytest.mark.parametrize("chunk", [1, 262144, 262145, 2 ** 30, 2 ** 31 - 1])
def test_chunks_of_the_largest_tile_count(chunk):
    """On the host: chunk bounds stay within 2^31 - 1 tiles, also those of the owners past the last one."""
    B.lib()
    P = ctypes.CDLL(PROBES)
    P.probe_conv_chunk.restype = None
    total, f, e = 2 ** 31 - 1, ctypes.c_int(), ctypes.c_int()
    last = -(-total // chunk) - 1
    for owner in (0, last // 2, last, last + 1, last + 7):
        P.probe_conv_chunk(min(owner, 2 ** 31 - 1), chunk, total, ctypes.byref(f), ctypes.byref(e))
        assert f.value == min(owner * chunk, total) and e.value == min((owner + 1) * chunk, total)


@pytest.mark.gpu
def test_largest_batch(cuda):
    """2^31 - 1 batch elements of one cell: every one is written."""
    import torch
    n = 2 ** 31 - 1
    if torch.cuda.mem_get_info()[0] < 40 << 30:
        pytest.skip("needs 40 GB of device memory")
    x = torch.ones((n, 1, 1), dtype=torch.float32, device="cuda")
    one = torch.ones(1, dtype=torch.float32, device="cuda")
    B.Conv1dPlan(B.CONV_F32, B.F32, n, 1, 1, 1, 2 * one.view(1, 1, 1), 0.5 * one).run(x)
    assert x.min().item() == 2.5 and x.max().item() == 2.5
    del x
    torch.cuda.empty_cache()


# (B, C, L, K): several tiles per row and several tiles per owner, K - 1 > TN.
VALU = [(600, 4, 1200, 300), (3000, 2, 1100, 290)]
MATRIX = [(600, 13, 600, 140)]


@pytest.mark.gpu
@pytest.mark.parametrize("mode,shape", [(B.CONV_F64, s) for s in VALU] + [(B.CONV_F32, s) for s in VALU + MATRIX],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else "f64" if v == B.CONV_F64 else "f32")
def test_kernels_longer_than_a_tile(cuda, mode, shape):
    """FP64 bit for bit, FP32 within the bound of a sum of n = C K products, (n + 2) 2^-24 (sum |w||x| + |bias|);
    three runs, since a column read too late shows only now and then."""
    import torch
    Bn, C, L, K = shape
    f32 = mode == B.CONV_F32
    npdt, code = (np.float32, B.F32) if f32 else (np.float64, B.F64)
    rng = np.random.default_rng(K)
    w = (rng.standard_normal((C, C, K)) / np.sqrt(C * K)).astype(npdt)
    b = (0.1 * rng.standard_normal(C)).astype(npdt)
    x = rng.standard_normal((Bn, C, L)).astype(npdt)
    ref = x.astype(np.float64)
    O.conv_torch_f64(ref, w.astype(np.float64), b.astype(np.float64))
    plan = B.Conv1dPlan(mode, code, Bn, C, L, K, torch.from_numpy(w).cuda(), torch.from_numpy(b).cuda())
    n = L - K + 1
    if f32:
        bound = np.abs(x).astype(np.float64)
        O.conv_torch_f64(bound, np.abs(w).astype(np.float64), np.abs(b).astype(np.float64))
        bound *= (C * K + 2) * 2.0 ** -24
    for _ in range(3):
        tx = torch.from_numpy(x).cuda()
        plan.run(tx)
        got = tx.cpu().numpy()
        assert np.array_equal(got[:, :, n:], x[:, :, n:])
        if f32:
            assert np.all(np.abs(got[:, :, :n].astype(np.float64) - ref[:, :, :n]) <= bound[:, :, :n])
        else:
            assert np.array_equal(got, ref)
