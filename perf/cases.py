"""The workloads that this framework is timed on, through its Python binding.

A case is a dict of plain values.  Kinds:
  step   one bkma_adv_run call (the reference's per-step executor call)
  plan   one AdvPlan.run of `steps` steps (the time loop of a driver)
  batch  one AdvBatch.run of `steps` steps over a ragged set of problems
  conv   one Conv1dPlan.run (textbook Conv1d, in place)

Every path works in place: run() returns the state's own arrays, and a second
run() goes on from there, as a time loop does.  Nothing grows without bound
then: the interpolation never amplifies a mode, and the convolution weights
are those of a lossless filter bank (or of a contraction).
"""
import math
import os
import random
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "parallel-advection_amd"))
import bkma_amd as B  # noqa: E402

DEV = "cuda:0"
TORCH = {"f64": torch.float64, "f32": torch.float32, "bf16": torch.bfloat16}
CODE = {"f64": B.F64, "f32": B.F32, "bf16": B.BF16}
MODE = {"f64": B.CONV_F64, "f32": B.CONV_F32, "bf16": B.CONV_BF16, "bf16x3": B.CONV_BF16X3,
        "bf16x6": B.CONV_BF16X6, "fp8": B.CONV_FP8}
SIZE = {"f64": 8, "f32": 4, "bf16": 2}


def listed():
    return [
        # The reference driver's own input file: one AdaptiveWg step on 256 short contiguous lines.
        # The whole array is 2 MB, so the call's latency is what a user sees.
        dict(name="step_small_f64", kind="step", dtype="f64", n0=256, n1=1024, n2=1, dt=1e-3, pref=512),
        # A drop-in time loop over a strided array, one executor call per step.
        dict(name="step_strided_f64", kind="step", dtype="f64", n0=2048, n1=1024, n2=64, dt=1e-3, pref=256),
        # The same small problem as a plan over its 100 steps.
        dict(name="plan_small_f64", kind="plan", dtype="f64", n0=256, n1=1024, n2=1, dt=1e-3, steps=100),
        # The headline workload: a large strided array, FP32 storage, 50 steps.
        dict(name="plan_strided_f32", kind="plan", dtype="f32", n0=2048, n1=1024, n2=512, dt=1e-3, steps=50),
        # FP64 on a grid with no power of two in it.
        dict(name="plan_ragged_f64", kind="plan", dtype="f64", n0=300, n1=1000, n2=100, dt=1e-3, steps=20),
        # Lines far longer than the LDS, large shifts, few columns.
        dict(name="plan_long_f32", kind="plan", dtype="f32", n0=256, n1=262144, n2=4, dt=1e-3, steps=20),
        # Contiguous lines of a length that is no multiple of a wavefront.
        dict(name="plan_lines_f64", kind="plan", dtype="f64", n0=4096, n1=10000, n2=1, dt=1e-3, steps=20),
        # Many independent problems of different shapes advanced together.
        dict(name="batch_ragged_f32", kind="batch", dtype="f32", problems=48, n0max=256, n1max=8192, shapes=3, steps=32),
        # Conv1d layer, BF16 activations.
        dict(name="conv_bf16", kind="conv", mode="bf16", io="bf16", B=1024, C=128, L=4096, K=5),
        # Wide Conv1d layer quantized to FP8, FP32 activations.
        dict(name="conv_fp8", kind="conv", mode="fp8", io="f32", B=512, C=256, L=8192, K=7),
        # The same layer as conv_bf16 in plain FP32, a quarter of the batch.
        dict(name="conv_f32", kind="conv", mode="f32", io="f32", B=256, C=128, L=4096, K=5),
        # FP64 (the reference's real type) on one of the reference benchmark's shapes: few channels.
        dict(name="conv_f64", kind="conv", mode="f64", io="f64", B=16384, C=6, L=256, K=5),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5)))))))


# Conv1d layers that have matrix-core kernels: mode, storage, channels, taps.
_MFMA = [("bf16", "bf16", 128, 5), ("bf16", "f32", 128, 5), ("bf16", "f32", 128, 3), ("bf16", "f32", 64, 5),
         ("bf16x3", "f32", 128, 5), ("bf16x3", "bf16", 128, 5), ("bf16x6", "f32", 128, 5), ("bf16x6", "f32", 64, 5),
         ("fp8", "f32", 256, 7), ("fp8", "bf16", 256, 7), ("fp8", "f32", 128, 5)]


def draw(rng):
    kind = rng.choice(["step", "step", "plan", "plan", "plan", "plan", "batch", "conv", "conv", "conv", "conv"])
    if kind == "step":
        n1, n2 = _log(rng, 64, 4096), rng.choice([1, _log(rng, 2, 63), _log(rng, 64, 512)])
        cells = _log(rng, 1 << 17, 1 << 27)
        return dict(kind=kind, dtype=rng.choice(["f64", "f64", "f32"]), n0=max(1, cells // (n1 * n2)), n1=n1, n2=n2,
                    dt=rng.choice([5e-4, 1e-3, 2e-3]), pref=rng.choice([128, 256, 512, 1024]))
    if kind == "plan":
        wide = rng.random() < 0.4
        n1, dt = _log(rng, 64, 4096 if wide else 65536), rng.choice([5e-4, 1e-3, 2e-3])
        if wide:  # the widest rows with small shifts, rows of any width among them
            n2 = _log(rng, 64, 512 if n1 * dt < 2 else 128)
            n2 -= n2 % rng.choice([2, 4, 4]) if n2 > 128 else 0
        else:
            n2 = rng.choice([1, _log(rng, 2, 63)])
        cells = _log(rng, 1 << 18, 1 << 28)
        return dict(kind=kind, dtype=rng.choice(["f64", "f32"]), n0=max(1, cells // (n1 * n2)), n1=n1, n2=n2, dt=dt,
                    steps=_log(rng, 1, 50))
    if kind == "batch":
        return dict(kind=kind, dtype=rng.choice(["f32", "f32", "f64"]), problems=_log(rng, 4, 48), n0max=_log(rng, 64, 256),
                    n1max=_log(rng, 1024, 8192), shapes=rng.randrange(1 << 20), steps=_log(rng, 4, 32))
    if rng.random() < 0.5:
        mode, io, c, k = rng.choice(_MFMA)
        length = _log(rng, 128, 8192)
        length -= length % rng.choice([1, 4, 8, 8])
        batch = max(1, _log(rng, 1 << 22, 1 << 28) // (c * length))
    else:
        mode = io = rng.choice(["f32", "f64"])
        c, k, length = _log(rng, 1, 128), rng.choice([1, 3, 5, 7, 11]), _log(rng, 64, 4096)
        batch = max(1, _log(rng, 1 << 20, 1 << 25) // (c * length))
    return dict(kind=kind, mode=mode, io=io, B=batch, C=c, L=length, K=k)


def _shapes(case):
    """The problems of a batch: (n0, n1, n2, dt) of each."""
    r = random.Random(case["shapes"])
    out = []
    for _ in range(case["problems"]):
        n1 = 64 * max(1, round(math.exp(r.uniform(0, math.log(case["n1max"] / 64)))))
        out.append((r.randint(16, case["n0max"]), n1, r.choice([1, 8, 64]), r.uniform(5e-4, 2e-3)))
    return out


def work(case):
    if case["kind"] == "conv":
        b, c, n, k = case["B"], case["C"], case["L"], case["K"]
        wsize = 8 if case["io"] == "f64" else 4
        return {"bytes": b * c * (n + n - k + 1) * SIZE[case["io"]] + (c * c * k + c) * wsize,
                "flops": 2 * b * c * c * k * (n - k + 1)}
    if case["kind"] == "batch":
        cells = sum(n0 * n1 * n2 for n0, n1, n2, _ in _shapes(case))
    else:
        cells = case["n0"] * case["n1"] * case["n2"]
    return {"bytes": 2 * cells * SIZE[case["dtype"]], "flops": 12 * cells * case.get("steps", 1)}


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _field(g, n0, n1, n2, dtype):
    """A smooth profile along the lines with noise on it."""
    x = (torch.arange(n1, dtype=torch.float64, device=DEV) * (2 * math.pi / n1)).sin().reshape(1, n1, 1)
    f = torch.rand((n0, n1, n2), generator=g, dtype=torch.float32, device=DEV).to(dtype)
    return f.add_(x.to(dtype))


def _weights(case, seed):
    """Weights [C][C][K] and bias [C] in FP64 on the host: variance 1/(C K), and the layer neither amplifies nor
    (from four channels on) damps its input, however often it is applied."""
    c, k = case["C"], case["K"]
    g = torch.Generator()
    g.manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g, dtype=torch.float64)  # noqa: E731
    bias = 0.01 * r(c)
    if c < 4:
        w = r(c, c, k)
        h = torch.fft.fft(w, n=256, dim=2).permute(2, 0, 1)
        return w / torch.linalg.matrix_norm(h, 2).max(), bias
    h = [torch.linalg.qr(r(c, c))[0]]  # product of an orthogonal matrix and k-1 factors (I - P) + z P
    for _ in range(k - 1):
        v = torch.linalg.qr(r(c, c // 2))[0]
        hp = [t @ v @ v.T for t in h]
        h = [(h[i] - hp[i] if i < len(h) else 0) + (hp[i - 1] if i else 0) for i in range(len(h) + 1)]
    return torch.stack(h, dim=2).contiguous(), bias


def _conv_inputs(case, seed):
    g = _gen(seed)
    x = torch.empty((case["B"], case["C"], case["L"]), dtype=TORCH[case["io"]], device=DEV).normal_(generator=g)
    w, b = _weights(case, seed)
    wt = torch.float64 if case["mode"] == "f64" else torch.float32
    return x, w.to(wt).to(DEV), b.to(wt).to(DEV)


def _params(case):
    return B.make_params(case["n0"], case["n1"], case["n2"], dt=case["dt"], minRealVx=-1.0, maxRealVx=1.0)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "conv":
        x, w, b = _conv_inputs(case, seed)
        plan = B.Conv1dPlan(MODE[case["mode"]], CODE[case["io"]], case["B"], case["C"], case["L"], case["K"], w, b)
        return {"kind": kind, "x": x, "plan": plan}
    if kind == "batch":
        g = _gen(seed)
        shapes = _shapes(case)
        arrays = [_field(g, n0, n1, n2, TORCH[case["dtype"]]) for n0, n1, n2, _ in shapes]
        params = [B.make_params(n0, n1, n2, dt=dt, minRealVx=-1.0, maxRealVx=1.0) for n0, n1, n2, dt in shapes]
        return {"kind": kind, "x": arrays, "steps": case["steps"], "batch": B.AdvBatch(arrays, params, CODE[case["dtype"]])}
    x = _field(_gen(seed), case["n0"], case["n1"], case["n2"], TORCH[case["dtype"]])
    p = _params(case)
    if kind == "step":
        o = B.create_optim_params(case["n0"], case["n1"], case["n2"], pref_wg_size=case["pref"], elem_size=SIZE[case["dtype"]])
        return {"kind": kind, "x": x, "params": p, "optim": o}
    return {"kind": kind, "x": x, "steps": case["steps"], "plan": B.AdvPlan(p, CODE[case["dtype"]])}


def run(state):
    kind, x = state["kind"], state["x"]
    if kind == "step":
        B.adv_run(B.ADAPTIVE_WG, x, state["params"], state["optim"])
    elif kind == "batch":
        state["batch"].run(state["steps"])
    elif kind == "plan":
        state["plan"].run(x, state["steps"])
    else:
        state["plan"].run(x)
    return x


def _advect(f, n0, n1, n2, dt, steps):
    """`steps` steps of f [n0][n1][n2] in FP64: v uniform on [-1, 1) by i0, x periodic on [0, 1), six-point rule."""
    dx, dvx = 1.0 / n1, 2.0 / n0
    inv_dx = 1.0 / dx
    x = torch.arange(n1, dtype=torch.float64, device=DEV) * dx
    f = f.to(torch.float64)
    chunk = max(1, (1 << 25) // (n1 * n2))
    for lo in range(0, n0, chunk):
        hi = min(n0, lo + chunk)
        v = -1.0 + torch.arange(lo, hi, dtype=torch.float64, device=DEV) * dvx
        foot = torch.fmod(1.0 + x[None, :] - (dt * v)[:, None], 1.0)
        left = torch.floor(foot * inv_dx)
        t = inv_dx * (foot - left * dx)  # position of the foot between its two nodes
        c = [-1 / 24 * t * (t - 1) * (t + 1) * (t - 2) * (t - 1),
             1 / 24 * t * (t - 1) * (t - 2) * (5 * t * t + t - 8),
             -1 / 12 * (t - 1) * (t - 2) * (t + 1) * (5 * t * t - 3 * t - 6),
             1 / 12 * t * (t + 1) * (t - 2) * (5 * t * t - 7 * t - 4),
             -1 / 24 * t * (t - 1) * (t + 1) * (5 * t * t - 11 * t - 2),
             1 / 24 * t * (t - 1) * t * (t + 1) * (t - 2)]
        c = [ck[:, :, None] for ck in c]
        at = [((left.to(torch.int64) + n1 - 2 + k) % n1) for k in range(6)]
        row = torch.arange(hi - lo, device=DEV)[:, None]
        g = f[lo:hi]
        for _ in range(steps):
            new = c[0] * g[row, at[0]]
            for k in range(1, 6):
                new.addcmul_(c[k], g[row, at[k]])
            g = new
        f[lo:hi] = g
    return f


def exact(case, seed):
    kind = case["kind"]
    if kind == "conv":
        x, w, b = _conv_inputs(case, seed)
        w, b, k = w.double(), b.double(), case["K"]
        n = case["L"] - k + 1
        out = x.double()
        chunk = max(1, (1 << 27) // (case["C"] * case["L"]))
        for lo in range(0, case["B"], chunk):
            src = x[lo:lo + chunk].double()
            y = b[None, :, None].expand(src.shape[0], case["C"], n).contiguous()
            for j in range(k):
                y += torch.matmul(w[:, :, j].contiguous(), src[:, :, j:j + n].contiguous())
            out[lo:lo + chunk, :, :n] = y
        return out
    if kind == "batch":
        g = _gen(seed)
        shapes = _shapes(case)
        fields = [_field(g, n0, n1, n2, TORCH[case["dtype"]]) for n0, n1, n2, _ in shapes]
        return [_advect(f, n0, n1, n2, dt, case["steps"]) for f, (n0, n1, n2, dt) in zip(fields, shapes)]
    f = _field(_gen(seed), case["n0"], case["n1"], case["n2"], TORCH[case["dtype"]])
    return _advect(f, case["n0"], case["n1"], case["n2"], case["dt"], case.get("steps", 1))
