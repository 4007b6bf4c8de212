"""Timed workloads of the framework: what each one is, its inputs, one pass, its result in 64 bits.

Inputs are synthetic (a seeded phantom generated on the GPU); every pass goes through
public entry points: ``ConvPlan``, ``DoseBatch``, ``LearnedCorrector``, ``ResidualCNN``,
``MonteCarlo``, ``TissueComposition``, ``resample_device`` and the C ABI's ``pvd_tac_fit``.
"""
from __future__ import annotations

import ctypes
import json
import math
import os
import random

import numpy as np
import torch

CIN = (16, 32, 32, 32, 32, 32)                 # input channels of the network's layers, as stored


def listed():
    return [
        # One SPECT-sized volume, 64^3 at 4.42 mm with a compact Y-90 kernel: the smallest dose
        # call, five short launches, where latency counts.
        {"name": "dose_small", "kind": "dose", "nx": 64, "ny": 64, "nz": 64, "k": 11, "mode": "reference",
         "times": 1, "density": False},
        # The benchmark's headline: a CT-sized volume, 31^3 kernel, density correction.
        {"name": "dose_ct", "kind": "dose", "nx": 256, "ny": 256, "nz": 200, "k": 31, "mode": "reference",
         "times": 1, "density": True},
        # A cropped patient volume of odd extents with the calculators' default 64^3 kernel
        # grid (even: no mirror symmetry about a voxel, the general complex spectrum) and the
        # time integral of four scans.
        {"name": "dose_series_odd", "kind": "dose", "nx": 217, "ny": 245, "nz": 163, "k": 64, "mode": "reference",
         "times": 4, "density": True},
        # Full-resolution torso at 0.98 mm, 61^3 kernel, six scans: the largest volume.
        {"name": "dose_torso", "kind": "dose", "nx": 512, "ny": 512, "nz": 400, "k": 61, "mode": "linear",
         "times": 6, "density": True},
        # A cohort of phantoms of uneven sizes, four scans each, in one captured graph.
        {"name": "batch_uneven", "kind": "batch", "volumes": 8, "lo": 96, "hi": 320, "sizes": 11, "k": 25,
         "mode": "reference", "times": 4, "density": True},
        # The learned correction of one 128^3 Y-90 volume, end to end (plain dose, network,
        # bounded correction): the benchmark's second figure.
        {"name": "correct_128", "kind": "correct", "nx": 128, "ny": 128, "nz": 128, "region": False},
        # Gradients of the network on one 128^3 phantom: the forward, loss and backward of a
        # training step.
        {"name": "train_128", "kind": "train", "nx": 128, "ny": 128, "nz": 128},
        # Monte Carlo training target of one 64^3 phantom (the trainer's default histories).
        {"name": "mc_64", "kind": "mc", "nx": 64, "ny": 64, "nz": 64, "nuclide": "Y90", "voxel_mm": 2.0,
         "histories": 16},
        # HU -> metal fill, tissue classes and density of a full-resolution CT with implants.
        {"name": "tissue_ct", "kind": "tissue", "nx": 512, "ny": 512, "nz": 400, "implants": 2},
        # A dose map from the 2 mm kernel grid back onto a 0.98 mm CT grid (the calculators'
        # default interpolation).
        {"name": "resample_linear_up", "kind": "resample", "nx": 251, "ny": 251, "nz": 196, "in_mm": 2.0,
         "out_mm": 0.98, "interp": "linear"},
        # The same by the cubic spline of resample_dose_map, onto a coarser, odd grid.
        {"name": "resample_cubic", "kind": "resample", "nx": 301, "ny": 301, "nz": 233, "in_mm": 1.37,
         "out_mm": 2.0, "interp": "cubic"},
        # Mono-exponential time-activity fits of every voxel of a CT-sized series.
        {"name": "tac_mono", "kind": "tac", "nx": 256, "ny": 256, "nz": 200, "times": 4, "model": "mono"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["dose", "dose", "dose", "batch", "correct", "train", "mc", "tissue", "resample", "resample",
                       "tac"])
    if kind == "dose":
        # 64 .. 512 voxels along each axis, any kernel grid the calculators are used with
        n = [_log_int(rng, 64, 512) for _ in range(3)]
        n[2] = min(n[2], 400)
        return {"kind": kind, "nx": n[0], "ny": n[1], "nz": n[2], "k": rng.choice([7, 11, 13, 21, 31, 47, 61, 64]),
                "mode": rng.choice(["reference", "linear"]), "times": rng.choice([1, 1, 2, 4, 5, 6]),
                "density": rng.random() < 0.75}
    if kind == "batch":
        return {"kind": kind, "volumes": rng.randint(3, 10), "lo": 96, "hi": rng.choice([160, 224, 300]),
                "sizes": rng.randint(0, 9999), "k": rng.choice([15, 21, 25, 31]),
                "mode": rng.choice(["reference", "linear"]), "times": rng.randint(1, 5),
                "density": rng.random() < 0.75}
    if kind == "correct":
        return {"kind": kind, "nx": rng.randint(48, 176), "ny": rng.randint(48, 176), "nz": rng.randint(40, 176),
                "region": rng.random() < 0.3}
    if kind == "train":
        return {"kind": kind, "nx": rng.randint(24, 128), "ny": rng.randint(24, 128),
                "nz": 32 * rng.randint(1, 4)}
    if kind == "mc":
        nuclide = rng.choice(["Y90", "Lu177"])
        return {"kind": kind, "nx": rng.randint(20, 80), "ny": rng.randint(20, 80), "nz": rng.randint(20, 80),
                "nuclide": nuclide, "voxel_mm": 2.0 if nuclide == "Y90" else 0.98,
                "histories": rng.choice([4, 8, 16, 24, 32])}
    if kind == "tissue":
        return {"kind": kind, "nx": _log_int(rng, 96, 512), "ny": _log_int(rng, 96, 512),
                "nz": _log_int(rng, 64, 400), "implants": rng.choice([0, 1, 2, 3])}
    if kind == "resample":
        up = rng.random() < 0.5
        n = [_log_int(rng, 64, 256 if up else 400) for _ in range(3)]
        a, b = rng.uniform(0.9, 1.5), rng.uniform(1.8, 4.5)
        if up:
            a, b = max(a, b * 0.45), b
        return {"kind": kind, "nx": n[0], "ny": n[1], "nz": n[2], "in_mm": round(b if up else a, 2),
                "out_mm": round(a if up else b, 2), "interp": rng.choice(["linear", "linear", "cubic", "nearest"])}
    return {"kind": kind, "nx": _log_int(rng, 48, 256), "ny": _log_int(rng, 48, 256), "nz": _log_int(rng, 48, 200),
            "times": rng.randint(3, 6), "model": rng.choice(["mono", "f2", "lmfit_mono"])}


# ------------------------------------------------------------------------------ inputs
def _shape(case):
    return case["nx"], case["ny"], case["nz"]


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed & 0x7FFFFFFF)


def _ellipsoid(shape, centre, semi):
    d = 0.0
    for a in range(3):
        view = [1, 1, 1]
        view[a] = shape[a]
        x = torch.arange(shape[a], device="cuda", dtype=torch.float32).view(view)
        d = d + ((x - centre[a] * shape[a]) / max(1.0, semi[a] * shape[a])) ** 2
    return d <= 1.0


def _phantom(shape, seed):
    """(activity, density): a body with lungs and a spine, uptake with 5 % noise, lesions."""
    rng, gen = random.Random(seed), _generator(seed)
    rho = torch.full(shape, 1.04, device="cuda")
    act = torch.full(shape, rng.uniform(0.05, 0.12), device="cuda")
    for side in (0.3, 0.7):
        lung = _ellipsoid(shape, (side, 0.5, 0.65), (0.13, 0.18, 0.28))
        rho[lung] = 0.26
        act[lung] *= 0.3
    spine = _ellipsoid(shape, (0.5, 0.78, 0.5), (0.06, 0.06, 3.0))
    rho[spine] = 1.85
    act[spine] *= 0.1
    for _ in range(rng.randint(3, 6)):
        r = rng.uniform(0.03, 0.08)
        act[_ellipsoid(shape, [rng.uniform(0.15, 0.85) for _ in range(3)], (r, r, r))] = rng.uniform(0.5, 2.0)
    act *= torch.randn(shape, device="cuda", generator=gen).mul_(0.05).add_(1.0).clamp_(0.2, 1.8)
    return act, rho


def _times(n):
    return [4.0, 24.0, 48.0, 72.0, 120.0, 168.0][:n]


def _series(act, seed, n, noise):
    """The activity at the scan times: washout that differs by region, and scan noise."""
    gen = _generator(seed + 77)
    lam = math.log(2.0) / 60.0 * (0.6 + 0.8 * act / act.max())
    out = []
    for t in _times(n):
        m = act * torch.exp(-lam * t)
        if noise:
            m *= torch.randn(m.shape, device="cuda", generator=gen).mul_(noise).add_(1.0).clamp_(0.5, 1.5)
        out.append(m)
    return out


def _point_kernel(k):
    """FP64 k^3 dose-point kernel about k//2: a beta part and a photon tail."""
    i = torch.arange(k, device="cuda", dtype=torch.float64) - k // 2
    r2 = (i * i).view(-1, 1, 1) + (i * i).view(1, -1, 1) + (i * i).view(1, 1, -1)
    r = r2.sqrt()
    return torch.exp(-1.1 * r) + 2e-3 * torch.exp(-0.02 * r) / (r2 + 0.25)


def _batch_shapes(case):
    rng = random.Random(case["sizes"])
    hi_z = max(case["lo"], case["hi"] * 5 // 6)
    return [(rng.randint(case["lo"], case["hi"]), rng.randint(case["lo"], case["hi"]), rng.randint(case["lo"], hi_z))
            for _ in range(case["volumes"])]


def _dose_inputs(shape, case, seed):
    act, rho = _phantom(shape, seed)
    acts = _series(act, seed, case["times"], 0.0) if case["times"] > 1 else [act]
    return acts, (rho if case["density"] else None)


def _weights(times):
    """Trapezoid of hours, in seconds."""
    w = [0.0] * len(times)
    for i in range(len(times) - 1):
        w[i] += (times[i + 1] - times[i]) * 1800.0
        w[i + 1] += (times[i + 1] - times[i]) * 1800.0
    return w


def _ct(case, seed):
    shape = _shape(case)
    rng, gen = random.Random(seed), _generator(seed)
    hu = torch.randn(shape, device="cuda", generator=gen).mul_(25.0).add_(45.0)
    outside = ~_ellipsoid(shape, (0.5, 0.5, 0.5), (0.46, 0.4, 3.0))
    hu[outside] = hu[outside] * 0.2 - 995.0
    for side in (0.3, 0.7):
        lung = _ellipsoid(shape, (side, 0.5, 0.65), (0.13, 0.18, 0.28))
        hu[lung] = hu[lung] - 780.0
    spine = _ellipsoid(shape, (0.5, 0.78, 0.5), (0.06, 0.06, 3.0))
    hu[spine] = hu[spine] * 4.0 + 500.0
    for i in range(case["implants"]):
        c = [rng.uniform(0.35, 0.65) for _ in range(3)]
        semi = (0.012, 0.012, 0.2) if i % 2 else (0.03, 0.025, 0.03)     # a rod, a plate
        hu[_ellipsoid(shape, c, semi)] = 3071.0
    return hu


def _net_state(seed):
    """Weights as a trained network has them (He-scaled, biased, a non-zero last layer), FP32."""
    g = torch.Generator().manual_seed(seed)
    parts = []
    for layer, cin in enumerate(CIN):
        used = 3 if layer == 0 else 32
        scale = (2.0 / (27 * used)) ** 0.5 * (0.5 if 0 < layer < 5 else 0.1 if layer == 5 else 1.0)
        w = torch.randn((27, 32, cin), generator=g) * scale
        w[:, :, used:] = 0.0
        b = torch.randn(32, generator=g) * 0.02
        if layer == 5:
            w[:, 1:] = 0.0
            b[1:] = 0.0
        parts += [w.reshape(-1), b]
    master = torch.cat(parts)
    return {"master": master, "m": torch.zeros_like(master), "v": torch.zeros_like(master), "step": 0}


def _train_inputs(case, seed):
    act, rho = _phantom(_shape(case), seed)
    n = act.numel()
    x = torch.zeros((n, 16), device="cuda", dtype=torch.bfloat16)
    plain = act / rho
    for c, m in enumerate((act / act.max(), rho, plain / plain.max())):
        x[:, c] = m.reshape(-1).to(torch.bfloat16)
    plain = plain.reshape(-1)
    mask = (plain >= 0.05 * plain.max()).float()
    ones = torch.ones_like(plain)
    noise = torch.randn(n, device="cuda", generator=_generator(seed + 5)) * 0.1
    ratio = torch.where(mask > 0, 1.0 + 0.3 * (rho.reshape(-1) - 1.04) + noise, ones)
    return x, ones, ratio, mask


def _tac_params(case):
    from pyvoxeldosimetry_amd import _native as nat
    t = _times(case["times"])
    q = nat.TacParams()
    q.model = {"mono": 0, "f2": 1, "lmfit_mono": 7}[case["model"]]
    q.n_times = len(t)
    for i, x in enumerate(t):
        q.t[i], q.w[i] = x, 1.0
    lam = math.log(2.0) / 161.52                                     # Lu-177, hours
    q.tol = 1.49012e-8
    if case["model"] == "mono":          # the basic fit: start at (A(t0), lambda), tail integral
        q.p0[1], q.p0_from_data, q.fail_params[1], q.max_iter, q.t_int = lam, 1, lam, 200, 100 * 161.52
    else:                                # the advanced fits: fixed start, trapezoid
        q.lambda_phys, q.p0[0], q.auc_mode, q.max_iter = lam, 1.0, 1, 3333
        q.p0[1] = 0.1 if case["model"] == "f2" else 161.52
    return q


# ------------------------------------------------------------------------------ prepare / run
def prepare(case, seed):
    kind = case["kind"]
    if kind == "dose":
        from pyvoxeldosimetry_amd.plan import ConvPlan
        acts, rho = _dose_inputs(_shape(case), case, seed)
        plan = ConvPlan(_shape(case), (case["k"],) * 3, mode=case["mode"])
        plan.set_kernel(_point_kernel(case["k"]))
        return {"kind": kind, "plan": plan, "acts": acts, "rho": rho, "times": _times(case["times"])}
    if kind == "batch":
        from pyvoxeldosimetry_amd.batch import DoseBatch
        shapes = _batch_shapes(case)
        batch = DoseBatch(shapes, [_point_kernel(case["k"])] * len(shapes), mode=case["mode"])
        inputs = [_dose_inputs(s, case, seed + 1000 * i) for i, s in enumerate(shapes)]
        w = _weights(_times(case["times"])) if case["times"] > 1 else [1.0]
        outs = [batch.set_volume(i, acts, w, density=rho) for i, (acts, rho) in enumerate(inputs)]
        return {"kind": kind, "batch": batch, "inputs": inputs, "outs": outs}
    if kind == "correct":
        from pyvoxeldosimetry_amd.learned.pipeline import LearnedCorrector
        act, rho = _phantom(_shape(case), seed)
        return {"kind": kind, "corr": LearnedCorrector.pretrained("Y90", 2.0), "act": act, "rho": rho,
                "region": case["region"]}
    if kind == "train":
        from pyvoxeldosimetry_amd.learned.cnn import ResidualCNN
        net = ResidualCNN()
        net.load_state_dict(_net_state(seed))
        x, dp, dt, mask = _train_inputs(case, seed)
        return {"kind": kind, "net": net, "x": x, "dp": dp, "dt": dt, "mask": mask, "shape": _shape(case)}
    if kind == "mc":
        from pyvoxeldosimetry_amd.learned.mc import MonteCarlo
        act, rho = _phantom(_shape(case), seed)
        return {"kind": kind, "mc": MonteCarlo(case["nuclide"]), "act": act, "rho": rho, "seed": seed,
                "voxel_mm": case["voxel_mm"], "histories": case["histories"]}
    if kind == "tissue":
        from pyvoxeldosimetry_amd.tissue.composition import TissueComposition
        return {"kind": kind, "tissue": TissueComposition(), "ct": _ct(case, seed)}
    if kind == "resample":
        act, _ = _phantom(_shape(case), seed)
        return {"kind": kind, "image": act, "in_mm": (case["in_mm"],) * 3, "out_mm": (case["out_mm"],) * 3,
                "interp": case["interp"]}
    act, _ = _phantom(_shape(case), seed)
    maps = _series(act, seed, case["times"], 0.03)
    return {"kind": kind, "maps": maps, "params": _tac_params(case)}


def run(s):
    kind = s["kind"]
    if kind == "dose":
        if len(s["acts"]) == 1:
            return s["plan"].dose(s["acts"][0], density=s["rho"])
        return s["plan"].dose_timeseries(s["acts"], s["times"], density=s["rho"])
    if kind == "batch":
        return s["batch"].run(graph=True)
    if kind == "correct":
        c = s["corr"].correct(s["act"], s["rho"], region=s["region"])
        # with a region, r is defined on the region only
        return {"dose": c.dose, "plain": c.plain} if s["region"] else {"dose": c.dose, "plain": c.plain, "r": c.r}
    if kind == "train":
        net = s["net"]
        r = net.forward(s["x"], s["shape"])
        sums = net.loss_and_grad(s["dp"], s["dt"], s["mask"], s["shape"])
        net.backward(s["x"], s["shape"])
        return {"r": r, "loss": sums, "grad": net.grad}
    if kind == "mc":
        return s["mc"].edep(s["act"], s["rho"], s["voxel_mm"], s["histories"], seed=s["seed"])
    if kind == "tissue":
        return s["tissue"].map(s["ct"])
    if kind == "resample":
        from pyvoxeldosimetry_amd.resample import resample_device
        return resample_device(s["image"], s["in_mm"], s["out_mm"], s["interp"])
    from pyvoxeldosimetry_amd import _native as nat
    lib, maps = nat.load(), s["maps"]
    n = maps[0].numel()
    params = torch.empty((2, n), device="cuda")
    auc = torch.empty(n, device="cuda")
    status = torch.empty(n, device="cuda", dtype=torch.uint8)
    arr = (ctypes.c_void_p * len(maps))(*[m.data_ptr() for m in maps])
    nat.check(lib.pvd_tac_fit(ctypes.byref(s["params"]), arr, n, ctypes.c_void_p(params.data_ptr()),
                              ctypes.c_void_p(auc.data_ptr()), ctypes.c_void_p(status.data_ptr()),
                              ctypes.c_void_p(nat.current_stream_handle())), "pvd_tac_fit")
    return {"params": params, "auc": auc, "status": status}


# ------------------------------------------------------------------------------ work
def _out_shape(case):
    return tuple(max(1, int(round(n * case["in_mm"] / case["out_mm"]))) for n in _shape(case))


def _dose_work(shape, case):
    n = shape[0] * shape[1] * shape[2]
    maps = case["times"] + (1 if case["density"] else 0) + 1
    return {"bytes": 4.0 * n * maps + 8.0 * case["k"] ** 3,
            "flops": 2 * 2.5 * n * math.log2(n) + 3.0 * n + 2.0 * n * case["times"]}


def work(case):
    kind = case["kind"]
    if kind == "batch":
        each = [_dose_work(s, case) for s in _batch_shapes(case)]
        return {k: sum(w[k] for w in each) for k in ("bytes", "flops")}
    n = case["nx"] * case["ny"] * case["nz"]
    if kind == "dose":
        return _dose_work(_shape(case), case)
    net = 2.0 * 27 * (3 * 32 + 4 * 32 * 32 + 32)                        # flops a voxel of one forward
    if kind == "correct":
        return {"bytes": 4.0 * n * 5, "flops": net * n}                  # two maps in, dose, plain and r out
    if kind == "train":
        return {"bytes": n * (32.0 + 3 * 4 + 4) + 4.0 * 114209, "flops": 3 * net * n}
    if kind == "mc":
        # about 20 steps of 100 operations a history, and the photon packets
        return {"bytes": 16.0 * n, "flops": 2000.0 * n * case["histories"]}
    if kind == "tissue":
        return {"bytes": 13.0 * n, "flops": 20.0 * n}
    if kind == "resample":
        m = math.prod(_out_shape(case))
        per = {"nearest": 1, "linear": 14, "cubic": 128}[case["interp"]]
        return {"bytes": 4.0 * (n + m), "flops": float(per * m + (90 * n if case["interp"] == "cubic" else 0))}
    # four Levenberg-Marquardt iterations of two evaluations, an exponential about 20 operations
    return {"bytes": n * (4.0 * case["times"] + 13.0), "flops": 4 * 2 * 40.0 * case["times"] * n}


# ------------------------------------------------------------------------------ results in 64 bits
def _conv64(a, kernel, mode):
    """Convolution of a (FP64) with the kernel: 'reference' circular of a's extents with the
    kernel's origin at its first element (cropped to a's extents), 'linear' centred."""
    n, k = a.shape, kernel.shape
    if mode == "reference":
        kernel = kernel[:n[0], :n[1], :n[2]]
        size, lo = n, (0, 0, 0)
    else:
        size, lo = tuple(p + q - 1 for p, q in zip(n, k)), tuple(q // 2 for q in k)
    f = torch.fft.rfftn(a, s=size)
    f *= torch.fft.rfftn(kernel, s=size)
    out = torch.fft.irfftn(f, s=size)
    return out[lo[0]:lo[0] + n[0], lo[1]:lo[1] + n[1], lo[2]:lo[2] + n[2]]


def _dose64(shape, case, seed):
    acts, rho = _dose_inputs(shape, case, seed)
    w = _weights(_times(case["times"])) if case["times"] > 1 else [1.0]
    total = sum(x * a.double() for x, a in zip(w, acts))
    del acts
    out = _conv64(total, _point_kernel(case["k"]), case["mode"])
    return out / rho.double() if rho is not None else out


def _layers64(master):
    out, at = [], 0
    for cin in CIN:
        n = 27 * 32 * cin
        out.append((master[at:at + n].view(27, 32, cin), master[at + n:at + n + 32]))
        at += n + 32
    return out


def _conv3(x, w):
    """3^3 convolution of channels-last x by w [27][cout][cin], zero outside."""
    nx, ny, nz = x.shape[:3]
    p = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
    out = 0.0
    for tap in range(27):
        i, j, l = tap // 9, tap // 3 % 3, tap % 3
        out = out + p[i:i + nx, j:j + ny, l:l + nz] @ w[tap].t()
    return out


def _network64(x, layers):
    h = torch.relu(_conv3(x, layers[0][0]) + layers[0][1])
    for w, b in layers[1:5]:
        h = h + torch.relu(_conv3(h, w) + b)
    return _conv3(h, layers[5][0][:, :1])[..., 0] + layers[5][1][0]


def _axis_matrix(n, m, ratio, interp):
    """m x n weights of one axis: output j reads the input at j * ratio, 0 outside
    [-0.5, n - 0.5); cubic: B-spline weights times the inverse of the sampling matrix,
    mirror boundaries."""
    c = torch.arange(m, dtype=torch.float64) * ratio
    inside = (c >= -0.5) & (c < n - 0.5)
    base = torch.floor(c)
    t = c - base
    out = torch.zeros((m, n), dtype=torch.float64)
    rows = torch.arange(m)
    period = max(1, 2 * (n - 1))

    def mirror(i):
        i = torch.remainder(i, period)
        return torch.where(i < n, i, period - i)

    base = base.long()
    if interp == "nearest":
        out[rows, (base + (t >= 0.5).long()).clamp(0, n - 1)] = 1.0
    elif interp == "linear":
        out.index_put_((rows, base.clamp(0, n - 1)), 1.0 - t, accumulate=True)
        out.index_put_((rows, (base + 1).clamp(0, n - 1)), t, accumulate=True)
    else:
        u = 1.0 - t
        w = [u ** 3 / 6, (3 * t ** 3 - 6 * t ** 2 + 4) / 6, (3 * u ** 3 - 6 * u ** 2 + 4) / 6, t ** 3 / 6]
        for q in range(4):
            out.index_put_((rows, mirror(base - 1 + q)), w[q], accumulate=True)
        sample = torch.zeros((n, n), dtype=torch.float64)
        at = torch.arange(n)
        for d, v in ((-1, 1 / 6), (0, 4 / 6), (1, 1 / 6)):
            sample.index_put_((at, mirror(at + d)), torch.full((n,), v, dtype=torch.float64), accumulate=True)
        out = torch.linalg.solve(sample.t(), out.t()).t()
    return (out * inside.unsqueeze(1)).cuda()


def _resample64(case, seed):
    x = _phantom(_shape(case), seed)[0].double()
    ratio = case["out_mm"] / case["in_mm"]
    for a, m in enumerate(_out_shape(case)):
        w = _axis_matrix(x.shape[a], m, ratio, case["interp"])
        x = torch.tensordot(w, x, dims=([1], [a])).movedim(0, a).contiguous()
    return x


def _tissue64(case, seed):
    ct = _ct(case, seed).double()
    metal = ct > 2000.0
    x = torch.where(metal, torch.zeros_like(ct), ct)
    k = torch.arange(-4, 5, dtype=torch.float64)
    w = torch.exp(-0.5 * k * k)
    w = (w / w.sum()).tolist()
    for a in range(3):
        n = x.shape[a]
        i = torch.arange(-4, n + 4)
        i = torch.remainder(i, 2 * n)
        p = x.index_select(a, torch.where(i < n, i, 2 * n - 1 - i).cuda())
        x = sum(v * p.narrow(a, q, n) for q, v in enumerate(w))
    # class bits are whole numbers, densities are entries of a table
    return [torch.where(metal, x, ct), None, None]


def _tac64(case, seed):
    act, _ = _phantom(_shape(case), seed)
    y = torch.stack([m.double().reshape(-1) for m in _series(act, seed, case["times"], 0.03)])
    t = torch.tensor(_times(case["times"]), dtype=torch.float64, device="cuda").unsqueeze(1)
    # least squares of A exp(-lam t): Gauss-Newton with step halving from the log-linear fit
    ly, tm = y.log(), t.mean()
    lam = -((t - tm) * ly).sum(0) / ((t - tm) ** 2).sum()
    a = torch.exp(ly.mean(0) + lam * tm)

    def cost(a, lam):
        return (y - a * torch.exp(-lam * t)).square().sum(0)

    best = cost(a, lam)
    for _ in range(40):
        e = torch.exp(-lam * t)
        r, g = y - a * e, -t * a * e
        ee, eg, gg, er, gr = (e * e).sum(0), (e * g).sum(0), (g * g).sum(0), (e * r).sum(0), (g * r).sum(0)
        det = ee * gg - eg * eg
        da, dl = (gg * er - eg * gr) / det, (ee * gr - eg * er) / det
        step = torch.ones_like(a)
        for _ in range(4):
            c = cost(a + step * da, lam + step * dl)
            step = torch.where(c <= best, step, step * 0.5)
        c = cost(a + step * da, lam + step * dl)
        better = c <= best
        a, lam = torch.where(better, a + step * da, a), torch.where(better, lam + step * dl, lam)
        best = torch.where(better, c, best)
    if case["model"] == "mono":
        return {"params": torch.stack([a, lam]), "auc": a / lam * (1.0 - torch.exp(-lam * 100 * 161.52)),
                "status": None}
    f = a * torch.exp(-lam * t)
    auc = ((f[1:] + f[:-1]) * 0.5 * (t[1:] - t[:-1])).sum(0)
    second = lam - math.log(2.0) / 161.52 if case["model"] == "f2" else math.log(2.0) / lam
    return {"params": torch.stack([a, second]), "auc": auc, "status": None}


def _correct64(case, seed):
    """The plain dose, the correction and the corrected dose from the corrector's point
    kernel (a Monte Carlo tally, taken as it is) and the shipped weights."""
    from pyvoxeldosimetry_amd.learned import pipeline
    act, rho = _phantom(_shape(case), seed)
    corr = pipeline.LearnedCorrector.pretrained("Y90", 2.0)
    kernel, bound, frac = corr.kernel.double(), corr.bound, corr.region_frac
    with open(os.path.join(pipeline.WEIGHTS_DIR, pipeline.PRETRAINED["Y90", 2.0]), "rb") as f:
        head = json.loads(f.read(int.from_bytes(f.read(8), "little")))
        data = f.read()
    lo, hi = head["master"]["data_offsets"]
    master = torch.from_numpy(np.frombuffer(data[lo:hi], np.float32).copy()).cuda().double()
    plain = _conv64(act.double(), kernel, "linear") / rho.double()
    x = torch.zeros((*act.shape, 16), dtype=torch.float64, device="cuda")
    x[..., 0], x[..., 1], x[..., 2] = act / act.max(), rho, plain / plain.max()
    r = _network64(x, _layers64(master))
    use = r.abs() <= bound
    if case["region"]:
        use &= plain >= frac * plain.max()
    exceed = (r.abs() > bound) & (plain >= 0.1 * plain.max())
    if exceed.sum() > corr.max_exceed_frac * (plain >= 0.1 * plain.max()).sum():
        use[:] = False
    out = {"dose": torch.where(use, plain * (1.0 + r), plain), "plain": plain}
    return out if case["region"] else {**out, "r": r}


def _train64(case, seed):
    x, dp, dt, mask = _train_inputs(case, seed)
    # the weights as the network holds them for its products: BF16, biases FP32
    layers = [(w.to(torch.bfloat16).double().requires_grad_(), b.double().requires_grad_())
              for w, b in _layers64(_net_state(seed)["master"].cuda())]
    r = _network64(x.double().view(*_shape(case), 16), layers)
    e = dp.double() * r.reshape(-1) - (dt.double() - dp.double())
    m = mask.double()
    ((m * e * e).sum() / m.sum()).backward()
    with torch.no_grad():
        grads = []
        for layer, (w, b) in enumerate(layers):
            g = w.grad
            if layer == 0:
                g[:, :, 3:] = 0.0
            grads += [g.reshape(-1), b.grad]
        # of the last layer only channel 0 is used
        dr = 2.0 * m * e * dp.double() / m.sum()
        return {"r": r.detach().reshape(-1), "loss": torch.stack([(m * e * e).sum(), m.sum(), dr.sum()]),
                "grad": torch.cat(grads)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "dose":
        return _dose64(_shape(case), case, seed)
    if kind == "batch":
        return [_dose64(s, case, seed + 1000 * i) for i, s in enumerate(_batch_shapes(case))]
    if kind == "correct":
        with torch.no_grad():
            return _correct64(case, seed)
    if kind == "train":
        return _train64(case, seed)
    if kind == "mc":
        return None                       # a random tally: no value of its own
    if kind == "tissue":
        return _tissue64(case, seed)
    if kind == "resample":
        return _resample64(case, seed)
    return _tac64(case, seed)
