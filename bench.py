"""Benchmark of the kernel-convolution dose path on one MI355X.

Default workload (the CT-sized single volume): 256x256x200 FP32 activity at
2.0 mm, liver ellipsoid + 3 lesions, density map with lung and bone, Lu-177
31^3 dose-point kernel, reference (circular) convolution semantics, inputs
resident in HBM.  A step is one full dose-rate map (five HIP passes).

Prints one JSON line with throughput (Gvoxel/s), the roofline of the dominant
kernel (HIP-event timed), the error against the FP64 oracle and the CPU
baseline (the restated reference expression, np.fft complex128, one core).
"""
from __future__ import annotations

import argparse
import json
import os
import re
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "Gvoxel/s dose conv 256x256x200 (FP64 err≤1e-5); CNN-corrected ms/vol @ ≤2% err"
HBM_PEAK_GBS = 8000.0
TRAFFIC_FILE = os.path.join(ROOT, "profiles", "fft_passes_ct_256x256x200.md")
TORSO_TRAFFIC_FILE = os.path.join(ROOT, "profiles", "fft_passes_torso_512x512x400.md")


def pass_bytes(plan, T: int, density: bool):
    """Algorithmic (compulsory) bytes of each FFT pass: its own inputs and outputs.

    FZ reads T FP32 maps, writes the half spectrum Nx*Ny*H complex64; FY reads
    that and writes Nx*Py*H; X reads Nx*Py*H plus the kernel spectrum
    Px*Py*H and writes Nx*Py*H; IY reads Nx*Py*H, writes Nx*Ny*H; IZ reads
    Nx*Ny*H (+ FP32 density) and writes the FP32 dose.  A mirror-symmetric
    kernel has a real, even spectrum: X then reads only its FP32 octant
    (Px/2+1)*(Py/2+1)*H.
    """
    nx, ny, nz = plan.shape
    px, py, pz = plan.fft_n
    h = pz // 2 + 1
    n = nx * ny * nz
    c = 8
    spec = 4 * (px // 2 + 1) * (py // 2 + 1) * h if plan.symmetric_spectrum else c * px * py * h
    return {
        "fft_z_forward": 4 * T * n + c * nx * ny * h,
        "fft_y_forward": c * nx * ny * h + c * nx * py * h,
        "fft_x_spectrum_multiply": c * nx * py * h * 2 + spec,
        "fft_y_inverse": c * nx * py * h + c * nx * ny * h,
        "fft_z_inverse_epilogue": c * nx * ny * h + 4 * n * (2 if density else 1),
    }


def read_traffic(kernel_name: str, summary: str = TRAFFIC_FILE):
    """HBM bytes per launch of `kernel_name` from a committed rocprof summary, if present."""
    try:
        text = open(os.path.join(ROOT, "profiles", summary) if not os.path.isabs(summary) else summary).read()
    except OSError:
        return None
    m = re.search(r"traffic_bytes_per_launch\[" + re.escape(kernel_name) + r"\]\s*=\s*([0-9.eE+]+)", text)
    return float(m.group(1)) if m else None


def cpu_baseline(act64, kernel64, reps: int):
    """The reference expression (kernel_convolution.py:71-74) restated, timed on the host."""
    from oracle import conv
    n = act64.size
    conv.ref_conv(act64, kernel64)                       # warm-up
    ts = []
    d64 = None
    for _ in range(reps):
        t0 = time.perf_counter()
        d64 = conv.ref_conv(act64, kernel64)
        ts.append(time.perf_counter() - t0)
    ts.sort()
    med = ts[len(ts) // 2]
    return {"value": n / med / 1e9, "unit": "Gvoxel/s", "cores": 1, "kind": "port",
            "sample": f"{reps} full 256x256x200 calls of np.fft.ifftn(fftn(A)*fftn(K,s)).real "
                      f"(complex128, numpy unthreaded) after 1 warm-up; median {med:.3f} s"}, d64


def cpu_strong(act64, kernel64, d64, reps: int):
    """A strong multi-threaded CPU path for the same circular convolution: scipy.fft
    rfftn/irfftn in FP32 with one worker per host core this process may use (at most 16,
    the host share of one GPU), timed like the reference path; its error against the
    FP64 result is reported with it."""
    import numpy as np
    import scipy.fft as sfft
    workers = max(1, min(len(os.sched_getaffinity(0)), 16))
    a = act64.astype(np.float32)
    k = kernel64.astype(np.float32)

    def run():
        spec = sfft.rfftn(a, workers=workers) * sfft.rfftn(k, s=a.shape, workers=workers)
        return sfft.irfftn(spec, s=a.shape, workers=workers)

    run()
    ts = []
    d = None
    for _ in range(reps):
        t0 = time.perf_counter()
        d = run()
        ts.append(time.perf_counter() - t0)
    ts.sort()
    med = ts[len(ts) // 2]
    err = float(np.max(np.abs(d - d64)) / np.max(np.abs(d64)))
    model = ""
    try:
        with open("/proc/cpuinfo") as f:
            model = next((ln.split(":", 1)[1].strip() for ln in f if ln.startswith("model name")), "")
    except OSError:
        pass
    return {"value": act64.size / med / 1e9, "unit": "Gvoxel/s", "cores": workers,
            "kind": "scipy.fft rfftn/irfftn f32",
            "sample": f"{reps} full 256x256x200 circular convolutions after 1 warm-up; median {med:.4f} s",
            "max_rel_vs_fp64": err,
            "host": {"cpu_model": model, "cpu_count": os.cpu_count(), "affinity": len(os.sched_getaffinity(0))}}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=500)
    ap.add_argument("--warmup", type=int, default=20)
    ap.add_argument("--cpu-reps", type=int, default=5)
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline and the FP64 error check")
    ap.add_argument("--no-eval", action="store_true", help="cnn and torso configs: skip the Monte Carlo error evaluation")
    ap.add_argument("--no-cnn", action="store_true",
                    help="ct and torso configs: leave the CNN-corrected part out of the line")
    ap.add_argument("--profile-reps", type=int, default=50)
    ap.add_argument("--copy-calibration", action="store_true",
                    help="only run 10 device copies of 256 MiB (reference for rocprof byte counters)")
    ap.add_argument("--config", default="ct",
                    choices=["ct", "batch", "torso", "tissue", "cnn", "tac", "resample", "direct"],
                    help="ct: 256x256x200 single volume (default, the headline metric); batch: 48 uneven "
                         "phantoms x 4 timepoints in one graph; torso: 512x512x400, 61^3, 6 timepoints; "
                         "tissue: HU -> metal fill, class masks and density of a 512x512x400 CT; "
                         "cnn: CNN-corrected Y-90 dose of a 128^3 phantom (time, MFMA use, error vs Monte Carlo); "
                         "tac: voxelwise mono-exponential TAC fit + integral of 256x256x200 voxels x 4 timepoints; "
                         "resample: trilinear 512x512x400 @0.98 mm -> 2 mm grid and back; "
                         "direct: LDS direct convolution of 128^3 with a 13^3 kernel")
    args = ap.parse_args()
    if args.gpus != 1:
        print(json.dumps({"error": "this build measures one GPU only; run with --gpus 1"}))
        sys.exit(2)

    import numpy as np
    import torch

    if args.copy_calibration:
        src = torch.ones(64 * 1024 * 1024, dtype=torch.float32, device="cuda")
        dst = torch.empty_like(src)
        dst.copy_(src)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(10):
            dst.copy_(src)
        torch.cuda.synchronize()
        dt = (time.perf_counter() - t0) / 10
        print(json.dumps({"copy_bytes_read": src.numel() * 4, "copy_bytes_written": dst.numel() * 4, "copies": 11,
                          "copy_GBs": round(2 * src.numel() * 4 / dt / 1e9, 1)}))
        return

    if args.config == "batch":
        return bench_batch(args)
    if args.config == "torso":
        return bench_torso(args)
    if args.config == "tissue":
        return bench_tissue(args)
    if args.config == "cnn":
        return bench_cnn(args)
    if args.config == "tac":
        return bench_tac(args)
    if args.config == "resample":
        return bench_resample(args)
    if args.config == "direct":
        return bench_direct(args)

    from pyvoxeldosimetry_amd import ConvPlan, Lu177KernelGenerator
    from pyvoxeldosimetry_amd.phantoms import ct_phantom

    dev = torch.device("cuda", 0)
    torch.cuda.set_device(dev)
    ph = ct_phantom(seed=2)
    kern = Lu177KernelGenerator("water").generate_kernel_device(ph.voxel_mm, ph.kernel_grid, device=dev)
    act = torch.from_numpy(ph.activity[0]).to(dev)
    # the density map from the phantom's synthetic CT through the HU -> density producer
    from pyvoxeldosimetry_amd.tissue import density_from_hu
    rho = density_from_hu(torch.from_numpy(ph.meta["hu"]).to(dev))
    if not torch.equal(rho.cpu(), torch.from_numpy(ph.density)):
        raise RuntimeError("HU -> density on the device differs from the phantom's table lookup")
    out = torch.empty_like(act)
    plan = ConvPlan(ph.shape, ph.kernel_grid, mode="reference", algo="auto", device=dev)
    plan.set_kernel(kern)
    nvox = act.numel()

    for _ in range(args.warmup):
        plan.dose(act, density=rho, out=out)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        plan.dose(act, density=rho, out=out)
    torch.cuda.synchronize()
    dt = time.perf_counter() - t0
    ms_step = dt * 1e3 / args.steps
    gvox = nvox / (ms_step / 1e3) / 1e9

    # the timed plan's own output is the one checked against the FP64 oracle below
    timed_out = out.clone()

    # cold call: plan + kernel spectrum + one dose, as the reference pays on every call
    # (it recomputes fftn(K, s) each time, kernel_convolution.py:73); the library's
    # one-time set-up is done above
    cold = {}
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    cplan = ConvPlan(ph.shape, ph.kernel_grid, mode="reference", algo=plan.algo, device=dev)
    t1 = time.perf_counter()
    cplan.set_kernel(kern)
    torch.cuda.synchronize()
    t2 = time.perf_counter()
    cplan.dose(act, density=rho, out=out)
    torch.cuda.synchronize()
    t3 = time.perf_counter()
    cplan.close()
    cold = {"total_ms": round((t3 - t0) * 1e3, 3), "plan_ms": round((t1 - t0) * 1e3, 3),
            "spectrum_ms": round((t2 - t1) * 1e3, 3), "dose_ms": round((t3 - t2) * 1e3, 3)}

    # per-kernel durations: HIP events recorded between the passes on the launch stream
    prof = ConvPlan(ph.shape, ph.kernel_grid, mode="reference", algo=plan.algo,
                    fft_n=plan.fft_n if plan.algo == "fft" else None, profile=True, device=dev)
    prof.set_kernel(kern)
    acc = {}
    prof_out = torch.empty_like(act)
    for i in range(args.profile_reps + 3):
        prof.dose(act, density=rho, out=prof_out)
        t = prof.timings()
        if i >= 3:
            for k, v in t.items():
                acc[k] = acc.get(k, 0.0) + v / args.profile_reps
    dom = max(acc, key=acc.get)
    roof = None
    if plan.algo == "fft":
        pb = pass_bytes(plan, 1, True)
        achieved = pb[dom] / (acc[dom] * 1e-3) / 1e9
        roof = {"bound": "hbm", "achieved": round(achieved, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                "frac": round(achieved / HBM_PEAK_GBS, 4), "traffic": read_traffic(dom), "kernel": dom,
                "kernel_ms": round(acc[dom], 5), "algorithmic_bytes": pb[dom]}
    b_alg = nvox * (4 + 4 + 4) + 4 * int(np.prod(ph.kernel_grid))
    operator_roof = {"algorithmic_bytes": b_alg, "achieved_GBs": round(b_alg / (ms_step * 1e-3) / 1e9, 1),
                     "frac": round(b_alg / (ms_step * 1e-3) / 1e9 / HBM_PEAK_GBS, 4)}

    result = {
        "metric": METRIC, "value": round(gvox, 3), "unit": "Gvoxel/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": round(ms_step, 5), "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None, "dtype": "f32", "data": "synthetic (seeded CT phantom, seed 2)",
        "config": {"workload": "ct single volume 256x256x200 f32 @2.0 mm, Lu-177 31^3 kernel, density map from "
                               "a synthetic CT (HU -> density producer), reference (circular) convolution",
                   "algo": plan.algo,
                   "fft_n": list(plan.fft_n), "mode": "reference", "symmetric_spectrum": plan.symmetric_spectrum},
        "roofline": roof, "operator_roofline": operator_roof,
        "per_pass_ms": {k: round(v, 5) for k, v in acc.items()},
        "cold_call_ms": cold,
    }
    if not args.no_cpu:
        cb, d64 = cpu_baseline(ph.activity[0].astype(np.float64), kern.cpu().numpy(), args.cpu_reps)
        result["cpu_baseline"] = cb
        from oracle import conv
        got = timed_out.cpu().numpy()
        m = conv.error_metrics(got, conv.epilogue(d64, ph.density))
        result["error_vs_fp64"] = {"max_rel": m["max_rel"], "rms_rel": m["rms_rel"]}
        result["speedup_vs_cpu_reference"] = round(gvox / cb["value"], 1)
        result["cpu_strong"] = cpu_strong(ph.activity[0].astype(np.float64), kern.cpu().numpy(), d64,
                                          args.cpu_reps)
        result["speedup_vs_cpu_strong"] = round(gvox / result["cpu_strong"]["value"], 1)
    if not args.no_cnn:
        # the metric's second half: CNN-corrected ms/vol and its error against held-out Monte Carlo
        from pyvoxeldosimetry_amd.learned.pipeline import EVAL_SEEDS_TEST
        m = cnn_measure(dev, 50, 5, list(EVAL_SEEDS_TEST), histories=8192)
        ev = m["eval"]
        result["cnn_corrected"] = {
            "ms_per_vol": round(m["ms_corr"], 4), "plain_ms_per_vol": round(m["ms_plain"], 4),
            "ratio_corrected_over_plain": round(m["ms_corr"] / m["ms_plain"], 2),
            "cnn_forward_ms": round(m["ms_net"], 4),
            "mfma_frac": round(m["alg_flops"] / (m["ms_net"] * 1e-3) / 2.5e15, 4),
            "region_mode_ms": round(m["ms_corr_region"], 4),
            "region_mode_block_fraction": round(m["region_block_frac"], 4),
            "workload": "Y-90 128^3 @2 mm (synth_phantom seed 123), plain FFT dose + 6-layer 3^3 residual CNN "
                        "(BF16 MFMA) over the whole volume + bounded correction (region mode: only the blocks "
                        "within the receptive field of plain dose >= 5 % of max)",
            "error_vs_monte_carlo": {k: (round(v, 4) if isinstance(v, float) else v) for k, v in ev.items()},
            "error_sample": "6 held-out phantoms (seeds 20000..20005) at 64^3, Monte Carlo 8192 histories/voxel; "
                            "voxels >= 10 % of max"}
    print(json.dumps(result), flush=True)


def _timed(fn, steps, warmup):
    import torch
    for _ in range(warmup):
        fn()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(steps):
        fn()
    torch.cuda.synchronize()
    return (time.perf_counter() - t0) * 1e3 / steps


def bench_batch(args):
    """48 uneven phantoms (96^3 .. 384x384x320), 4 timepoints each, Y-90 11^3 or Lu-177 31^3,
    trapezoid time-integrated dose, all volumes in one graph of five launches."""
    import numpy as np
    import torch

    from pyvoxeldosimetry_amd import Lu177KernelGenerator, Y90KernelGenerator
    from pyvoxeldosimetry_amd.batch import DoseBatch
    from pyvoxeldosimetry_amd.phantoms import BATCH_TIMEPOINTS_H, batch_phantom, batch_specs

    dev = torch.device("cuda", 0)
    torch.cuda.set_device(dev)
    specs = batch_specs()
    kern = {"Y90": Y90KernelGenerator("water", fix_centre=True).generate_kernel_device(2.0, (11, 11, 11)),
            "Lu177": Lu177KernelGenerator("water").generate_kernel_device(2.0, (31, 31, 31))}
    b = DoseBatch([s.shape for s in specs], [kern[s.nuclide] for s in specs], mode="reference", device=dev)
    host = {}
    t = BATCH_TIMEPOINTS_H
    for i, s in enumerate(specs):
        ph = batch_phantom(s)
        b.set_volume_timeseries(i, [torch.from_numpy(a).to(dev) for a in ph.activity], t)
        if i < 3:
            host[i] = ph
    work = sum(int(np.prod(s.shape)) * len(t) for s in specs)
    ms = _timed(lambda: b.run(graph=True), args.steps, args.warmup)
    res = {"metric": "Gvoxel-timepoint/s batched time-integrated dose (48 uneven phantoms x 4 timepoints)",
           "value": round(work / (ms * 1e-3) / 1e9, 3), "unit": "Gvoxel-timepoint/s", "n_gpus": 1,
           "steps": args.steps, "warmup": args.warmup, "ms_per_step": round(ms, 4), "higher_is_better": True,
           "dtype": "f32", "data": "synthetic (batch_specs seed 3)",
           "config": {"workload": "batch 48 phantoms 96^3..384x384x320, T=4, Y-90 11^3 / Lu-177 31^3, reference "
                                  "(circular) convolution, one hipGraph of five launches",
                      "voxel_timepoints": work}}
    if not args.no_cpu:
        from oracle import conv
        outs = b.run(graph=True)
        torch.cuda.synchronize()
        errs = []
        cpu_t = 0.0
        cpu_work = 0
        for i, ph in host.items():
            k = kern[specs[i].nuclide].cpu().numpy()
            t0 = time.perf_counter()
            exp = conv.ref_absorbed_dose([a.astype(np.float64) for a in ph.activity], t, k)
            cpu_t += time.perf_counter() - t0
            cpu_work += ph.activity[0].size * len(t)
            errs.append(conv.error_metrics(outs[i].cpu().numpy(), exp))
        res["error_vs_fp64"] = {"max_rel": max(e["max_rel"] for e in errs), "rms_rel": max(e["rms_rel"] for e in errs),
                                "volumes_checked": len(errs)}
        cpu_v = cpu_work / cpu_t / 1e9
        res["cpu_baseline"] = {"value": cpu_v, "unit": "Gvoxel-timepoint/s", "cores": 1, "kind": "port",
                               "sample": f"reference calculate_absorbed_dose (4 np.fft convs + trapezoid) on the "
                                         f"first {len(host)} phantoms, {cpu_t:.2f} s"}
        res["speedup_vs_cpu_reference"] = round(res["value"] / cpu_v, 1)
    b.close()
    print(json.dumps(res), flush=True)


def bench_torso(args):
    """512x512x400 at 0.98 mm, Lu-177 61^3, 6 timepoints, density, linear (padded) convolution."""
    import numpy as np
    import torch

    from pyvoxeldosimetry_amd import ConvPlan, Lu177KernelGenerator
    from pyvoxeldosimetry_amd.phantoms import torso_phantom

    dev = torch.device("cuda", 0)
    torch.cuda.set_device(dev)
    ph = torso_phantom()
    kern = Lu177KernelGenerator("water").generate_kernel_device(ph.voxel_mm, ph.kernel_grid, device=dev)
    acts = [torch.from_numpy(a).to(dev) for a in ph.activity]
    rho = torch.from_numpy(ph.density).to(dev)
    plan = ConvPlan(ph.shape, ph.kernel_grid, mode="linear", algo="fft", device=dev)
    plan.set_kernel(kern)
    out = torch.empty_like(acts[0])
    ms = _timed(lambda: plan.dose_timeseries(acts, ph.time_points_h, density=rho, out=out), args.steps, args.warmup)
    timed_out = out.clone()        # the error check reads the timed plan's result
    work = acts[0].numel() * len(acts)
    res = {"metric": "Gvoxel-timepoint/s time-integrated dose 512x512x400, 61^3 kernel, 6 timepoints",
           "value": round(work / (ms * 1e-3) / 1e9, 3), "unit": "Gvoxel-timepoint/s", "n_gpus": 1,
           "steps": args.steps, "warmup": args.warmup, "ms_per_step": round(ms, 4), "higher_is_better": True,
           "dtype": "f32", "data": "synthetic (torso phantom seed 5)",
           "config": {"workload": "torso 512x512x400 @0.98 mm, Lu-177 61^3, T=6, density, linear convolution",
                      "fft_n": list(plan.fft_n)}}
    # per-pass durations (HIP events between the passes) and the dominant pass's roofline
    prof = ConvPlan(ph.shape, ph.kernel_grid, mode="linear", algo="fft", profile=True, device=dev)
    prof.set_kernel(kern)
    acc = {}
    reps = max(3, min(args.profile_reps, 20))
    for i in range(reps + 2):
        prof.dose_timeseries(acts, ph.time_points_h, density=rho, out=out)
        if i >= 2:
            for k, v in prof.timings().items():
                acc[k] = acc.get(k, 0.0) + v / reps
    prof.close()
    dom = max(acc, key=acc.get)
    pb = pass_bytes(plan, len(acts), True)
    achieved = pb[dom] / (acc[dom] * 1e-3) / 1e9
    res["roofline"] = {"bound": "hbm", "achieved": round(achieved, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                       "frac": round(achieved / HBM_PEAK_GBS, 4), "traffic": read_traffic(dom, TORSO_TRAFFIC_FILE),
                       "kernel": dom,
                       "kernel_ms": round(acc[dom], 5), "algorithmic_bytes": pb[dom]}
    res["per_pass_ms"] = {k: round(v, 5) for k, v in acc.items()}
    if not args.no_cpu:
        from oracle import conv
        w = conv.trapezoid_weights_seconds(ph.time_points_h)
        acc = sum(wi * a.astype(np.float64) for wi, a in zip(w, ph.activity))
        exp = conv.epilogue(conv.linear_same(acc, kern.cpu().numpy()), ph.density)
        m = conv.error_metrics(timed_out.cpu().numpy(), exp)
        res["error_vs_fp64"] = {"max_rel": m["max_rel"], "rms_rel": m["rms_rel"]}
        t0 = time.perf_counter()
        conv.ref_conv(ph.activity[0].astype(np.float64), kern.cpu().numpy())
        one = time.perf_counter() - t0
        cpu_v = acts[0].numel() / one / 1e9
        res["cpu_baseline"] = {"value": cpu_v, "unit": "Gvoxel-timepoint/s", "cores": 1, "kind": "port",
                               "sample": f"one reference np.fft conv of the 512x512x400 map ({one:.2f} s); the "
                                         f"reference repeats it per timepoint"}
        res["speedup_vs_cpu_reference"] = round(res["value"] / cpu_v, 1)
    if not args.no_cnn:
        res["cnn_corrected"] = torso_cnn(dev, acts, ph, rho, args)
    print(json.dumps(res), flush=True)


def torso_cnn(dev, acts, ph, rho, args):
    """Learned correction of the torso's time-integrated dose (Lu-177 network at 0.98 mm):
    plain dose with the Monte Carlo point kernel, the network in z slabs of 128 (400 is
    not a multiple of 32), bounded correction; its error against Monte Carlo on 64^3
    sub-regions (activity kept only in the box): around the activity maximum, and across
    the lower boundary of the right lung."""
    import torch

    from pyvoxeldosimetry_amd.core.activity_sampler import trapezoid_weights
    from pyvoxeldosimetry_amd.learned.pipeline import (LearnedCorrector, evaluate_subregion, slab_extent,
                                                       subregion_box)
    corr = LearnedCorrector.pretrained("Lu177", ph.voxel_mm)
    w = [x * 3600.0 for x in trapezoid_weights(ph.time_points_h)]
    cum = torch.zeros_like(acts[0])
    for wi, a in zip(w, acts):
        cum.add_(a, alpha=wi)
    ms_plain = _timed(lambda: corr.plain(cum, rho), 5, 1)
    ms_corr = _timed(lambda: corr.correct(cum, rho), 3, 1)
    c = corr.correct(cum, rho)
    ext = slab_extent(cum.shape[2], cum.shape[0] * cum.shape[1])
    out = {"ms_per_vol": round(ms_corr, 3), "plain_ms_per_vol": round(ms_plain, 3),
           "ratio_corrected_over_plain": round(ms_corr / ms_plain, 2), "fallback": bool(c.fallback),
           "workload": "torso 512x512x400 @0.98 mm, time-integrated activity of the 6 timepoints, Lu-177 "
                       "Monte Carlo point kernel %d^3 (linear), 6-layer 3^3 residual CNN (BF16 MFMA) in z slabs of %d "
                       "(12-voxel overlaps), bounded correction" % (corr.kernel.shape[0], ext)}
    if not args.no_eval:
        sx, sy, sz = cum.shape
        boxes = {"hottest_lesion": subregion_box(cum, 64),
                 "lung_lower_edge": subregion_box(cum, 64, centre=(sx // 2, int(0.32 * sy), int(0.5 * sz)))}
        out["error_vs_monte_carlo_subregion"] = {k: evaluate_subregion(corr, cum, rho, b, histories=4096)
                                                 for k, b in boxes.items()}
    return out




def cnn_measure(dev, steps: int, warmup: int, eval_seeds=None, eval_shape=(64, 64, 64), histories: int = 8192):
    """CNN-corrected Y-90 dose of a 128^3 phantom at 2 mm: plain and corrected ms/vol,
    the network's MFMA throughput, and (eval_seeds) the error against held-out Monte Carlo."""
    import numpy as np
    import torch

    from pyvoxeldosimetry_amd.learned.pipeline import LearnedCorrector, evaluate, synth_phantom

    corr = LearnedCorrector.pretrained("Y90", 2.0)
    shape = (128, 128, 128)
    act, rho = synth_phantom(123, shape, dev)
    ms_plain = _timed(lambda: corr.plain(act, rho), steps, warmup)
    ms_corr = _timed(lambda: corr.correct(act, rho), steps, warmup)
    ms_corr_region = _timed(lambda: corr.correct(act, rho, region=True), steps, warmup)
    dp = corr.plain(act, rho)
    region_blocks = corr.region_blocks(dp, dp.max().reshape(1), corr.region_frac)[1].item()
    all_blocks = int(corr.lib.pvd_cnn_region_block_count(*shape))
    # the network as `correct` runs it: the input layer from the FP32 maps
    amax, dmax = corr.input_maxima(act, dp)
    maps = (act, rho, dp, amax, dmax, shape[2])
    ev0, ev1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    reps = 20
    corr.net.forward(None, shape, keep_activations=False, maps=maps)
    ev0.record()
    for _ in range(reps):
        corr.net.forward(None, shape, keep_activations=False, maps=maps)
    ev1.record()
    torch.cuda.synchronize()
    ms_net = ev0.elapsed_time(ev1) / reps
    n = int(np.prod(shape))
    alg = 2.0 * 27 * (3 * 32 + 4 * 32 * 32 + 32 * 1) * n          # useful MACs x 2 (3 in, 32 hidden, 1 out)
    # as issued on the matrix cores: input layer 7 MFMAs (4 taps x 4 channels each) per 32
    # voxels x 32 channels, residual layers 27 taps x 32 x 32, output layer 11 groups x 2 MFMAs
    # of 32 halo voxels x 32 tap columns per 256 voxels of a plane, in segments of 16 planes
    # with one more at either end
    executed = (2.0 * 7 * 16 * 32 + 4 * 2.0 * 27 * 32 * 32 + 11 * 2 * 32768 / 256 * 18 / 16) * n
    ev = None if eval_seeds is None else evaluate(corr, eval_seeds, eval_shape, histories=histories)
    return {"corr": corr, "ms_plain": ms_plain, "ms_corr": ms_corr, "ms_net": ms_net, "alg_flops": alg,
            "executed_flops": executed, "eval": ev, "act": act, "ms_corr_region": ms_corr_region,
            "region_block_frac": region_blocks / all_blocks}


def bench_cnn(args):
    """Learned heterogeneity correction: plain FFT dose + residual CNN (BF16 MFMA) of a
    128^3 Y-90 phantom at 2 mm; error of the shipped network against held-out Monte Carlo."""
    import numpy as np
    import torch

    from pyvoxeldosimetry_amd.learned.pipeline import EVAL_SEEDS_TEST

    dev = torch.device("cuda", 0)
    torch.cuda.set_device(dev)
    m = cnn_measure(dev, args.steps, args.warmup, None if args.no_eval else EVAL_SEEDS_TEST)
    ms_plain, ms_corr, ms_net, alg, executed = m["ms_plain"], m["ms_corr"], m["ms_net"], m["alg_flops"], \
        m["executed_flops"]
    peak = 2500.0
    res = {"metric": "CNN-corrected ms/vol (Y-90, 128^3 @2 mm) and error vs held-out Monte Carlo",
           "value": round(ms_corr, 4), "unit": "ms/vol", "n_gpus": 1, "steps": max(1, args.steps // 5),
           "warmup": args.warmup, "ms_per_step": round(ms_corr, 4), "higher_is_better": False, "dtype": "bf16",
           "data": "synthetic (synth_phantom seed 123; Monte Carlo targets of held-out seeds 20000..20005)",
           "config": {"workload": "plain FFT dose (linear, 13^3 MC kernel) + 6-layer 3^3 residual CNN "
                                  "(32 ch, BF16 MFMA, FP32 accumulate) + bounded correction, 128^3",
                      "plain_ms": round(ms_plain, 4), "cnn_forward_ms": round(ms_net, 4),
                      "ratio_corrected_over_plain": round(ms_corr / ms_plain, 2),
                      "region_mode_ms": round(m["ms_corr_region"], 4),
                      "region_mode_block_fraction": round(m["region_block_frac"], 4)},
           "roofline": {"bound": "mfma", "achieved": round(alg / (ms_net * 1e-3) / 1e12, 1), "peak": peak,
                        "unit": "TFLOP/s", "frac": round(alg / (ms_net * 1e-3) / 1e12 / peak, 4),
                        "executed_TFLOPs": round(executed / (ms_net * 1e-3) / 1e12, 1),
                        "executed_frac": round(executed / (ms_net * 1e-3) / 1e12 / peak, 4),
                        "traffic": read_traffic("cnn_forward_6_launches", "cnn_forward_128cubed.md"),
                        "kernel": "cnn_conv_in, 4 cnn_conv_march, cnn_conv_out_march", "kernel_ms": round(ms_net, 5),
                        "algorithmic_flops": alg},
           "error_vs_monte_carlo_64cubed": m["eval"]}
    if not args.no_cpu:
        from oracle import conv
        a64 = m["act"].cpu().numpy().astype(np.float64)
        k64 = m["corr"].kernel.cpu().numpy()
        conv.linear_same(a64, k64)
        t0 = time.perf_counter()
        conv.linear_same(a64, k64)
        t_cpu = time.perf_counter() - t0
        res["cpu_baseline"] = {"value": round(t_cpu * 1e3, 2), "unit": "ms/vol", "cores": 1, "kind": "port",
                               "sample": "plain convolution of the same 128^3 map on the host (np.fft complex128, "
                                         "1 core); the reference has no learned correction"}
    print(json.dumps(res), flush=True)


def bench_tac(args):
    """Voxelwise A0 exp(-lam t) fit (FP64 Levenberg-Marquardt per voxel) and the
    A0/lam (1 - exp(-lam 100 T1/2)) integral of a 256x256x200 x 4-timepoint series."""
    import numpy as np
    import torch

    from pyvoxeldosimetry_amd.phantoms import BATCH_TIMEPOINTS_H
    from pyvoxeldosimetry_amd.time_integration import TimeCurveFitting

    dev = torch.device("cuda", 0)
    torch.cuda.set_device(dev)
    rng = np.random.default_rng(12)
    shape = (256, 256, 200)
    n = int(np.prod(shape))
    t = np.array(BATCH_TIMEPOINTS_H, dtype=np.float64)
    a0 = torch.from_numpy(rng.uniform(1e3, 1e5, n).astype(np.float32)).to(dev)
    lam = torch.from_numpy(rng.uniform(0.004, 0.06, n).astype(np.float32)).to(dev)
    maps = [(a0 * torch.exp(-lam * float(ti)) * (1.0 + 0.03 * torch.randn(n, device=dev))).reshape(shape)
            for ti in t]
    tcf = TimeCurveFitting(64.1)
    run = lambda: tcf._fit(t, maps, 0, [0.0, tcf.decay_constant], None, False, 200,  # noqa: E731
                           [0.0, tcf.decay_constant], 0, t_int=100 * 64.1, p0_from_data=True)
    ms = _timed(run, max(1, args.steps // 50), min(args.warmup, 2))
    params, auc, status, _ = run()
    torch.cuda.synchronize()
    res = {"metric": "Gvoxel/s voxelwise mono-exponential TAC fit + integral, 256x256x200 x 4 timepoints",
           "value": round(n / (ms * 1e-3) / 1e9, 4), "unit": "Gvoxel/s", "n_gpus": 1,
           "steps": max(1, args.steps // 50), "warmup": min(args.warmup, 2), "ms_per_step": round(ms, 4),
           "higher_is_better": True, "dtype": "f64", "data": "synthetic (A0 U[1e3,1e5], lam U[0.004,0.06]/h, 3% noise)",
           "config": {"workload": "TimeCurveFitting.fit_time_activity_curve, 13.1 M voxels, T=4 at 4/24/72/144 h",
                      "converged_fraction": float(status.float().mean().item())},
           "roofline": {"bound": "hbm", "achieved": round(n * (16 + 12) / (ms * 1e-3) / 1e9, 1), "peak": HBM_PEAK_GBS,
                        "unit": "GB/s", "frac": round(n * 28 / (ms * 1e-3) / 1e9 / HBM_PEAK_GBS, 4), "traffic": None,
                        "kernel": "tac_fit_kernel", "note": "FP64 VALU-bound (exp and 2x2 solves per iteration); "
                                                           "28 B/voxel moved"}}
    if not args.no_cpu:
        from oracle import tac
        m = 3000
        y = np.stack([mp.reshape(-1)[:m].cpu().numpy().astype(np.float64) for mp in maps], axis=1)
        t0 = time.perf_counter()
        pe, acce = tac.fit_basic(t, y, 64.1)
        t_cpu = time.perf_counter() - t0
        res["cpu_baseline"] = {"value": m / t_cpu / 1e9, "unit": "Gvoxel/s", "cores": 1, "kind": "port",
                               "sample": f"reference loop (scipy curve_fit per voxel) on the first {m} voxels, "
                                         f"{t_cpu:.2f} s"}
        res["speedup_vs_cpu_reference"] = round(res["value"] / res["cpu_baseline"]["value"], 1)
        pg = params[:, :m].cpu().numpy().astype(np.float64)
        res["max_rel_param_err_vs_curve_fit"] = float(np.max(np.abs(pg - pe) / np.abs(pe)))
    print(json.dumps(res), flush=True)


def bench_direct(args):
    """The LDS-tiled direct convolution: 128^3 FP32 at 2 mm, Y-90 13^3 kernel (fixed centre),
    reference semantics, density map; FP32 VALU roofline (2 FLOP per tap and voxel)."""
    import numpy as np
    import torch

    from pyvoxeldosimetry_amd import ConvPlan, Y90KernelGenerator
    from pyvoxeldosimetry_amd.learned.pipeline import synth_phantom

    dev = torch.device("cuda", 0)
    torch.cuda.set_device(dev)
    shape, grid = (128, 128, 128), (13, 13, 13)
    act, rho = synth_phantom(31, shape, dev)
    kern = Y90KernelGenerator("water", fix_centre=True).generate_kernel_device(2.0, grid, device=dev)
    plan = ConvPlan(shape, grid, mode="reference", algo="direct", device=dev)
    plan.set_kernel(kern)
    out = torch.empty_like(act)
    ms = _timed(lambda: plan.dose(act, density=rho, out=out), args.steps, args.warmup)
    n = act.numel()
    flops = 2.0 * float(np.prod(grid)) * n
    # FP32 VALU peak without packed FP32 instructions (all HIP code here is built without them)
    peak = 157.3e12 / 2
    res = {"metric": "Gvoxel/s direct convolution 128^3, 13^3 kernel", "value": round(n / (ms * 1e-3) / 1e9, 3),
           "unit": "Gvoxel/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup, "ms_per_step": round(ms, 4),
           "higher_is_better": True, "dtype": "f32", "data": "synthetic (synth_phantom seed 31)",
           "config": {"workload": "direct conv 128^3 f32 @2 mm, Y-90 13^3 kernel, density, reference semantics",
                      "algo": plan.algo},
           "roofline": {"bound": "valu", "achieved": round(flops / (ms * 1e-3) / 1e12, 2),
                        "peak": round(peak / 1e12, 2), "unit": "TFLOP/s",
                        "frac": round(flops / (ms * 1e-3) / peak, 4), "traffic": None,
                        "kernel": "pvd_direct_kernel", "flop_per_step": flops}}
    if not args.no_cpu:
        from oracle import conv
        got = out.cpu().numpy()
        exp = conv.epilogue(conv.ref_conv(act.cpu().numpy().astype(np.float64), kern.cpu().numpy()),
                            rho.cpu().numpy())
        m = conv.error_metrics(got, exp)
        res["error_vs_fp64"] = {"max_rel": m["max_rel"], "rms_rel": m["rms_rel"]}
    print(json.dumps(res), flush=True)


def bench_resample(args):
    """Trilinear resampling of a 512x512x400 map at 0.98 mm onto the 2 mm kernel grid
    (251x251x196) and of that grid back to 0.98 mm: the voxel-size round trip of the dose path."""
    import numpy as np
    import torch

    from pyvoxeldosimetry_amd.phantoms import torso_phantom
    from pyvoxeldosimetry_amd.resample import output_shape_for, resample_device

    dev = torch.device("cuda", 0)
    torch.cuda.set_device(dev)
    ph = torso_phantom()
    a = torch.from_numpy(ph.activity[0]).to(dev)
    fine, coarse = (0.98,) * 3, (2.0,) * 3
    cshape = output_shape_for(a.shape, fine, coarse)
    down = torch.empty(cshape, dtype=torch.float32, device=dev)
    up = torch.empty_like(a)
    step = lambda: (resample_device(a, fine, coarse, "linear", cshape, out=down),  # noqa: E731
                    resample_device(down, coarse, fine, "linear", a.shape, out=up))
    ms = _timed(step, args.steps, args.warmup)
    n_out = down.numel() + up.numel()
    ev0, ev1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    ev0.record()
    for _ in range(20):
        resample_device(down, coarse, fine, "linear", a.shape, out=up)
    ev1.record()
    torch.cuda.synchronize()
    k_ms = ev0.elapsed_time(ev1) / 20
    alg = 4 * (down.numel() + up.numel())      # read the coarse grid once, write the fine one
    res = {"metric": "Gvoxel/s trilinear resampling 512x512x400 @0.98 mm <-> 2 mm (output voxels)",
           "value": round(n_out / (ms * 1e-3) / 1e9, 3), "unit": "Gvoxel/s", "n_gpus": 1, "steps": args.steps,
           "warmup": args.warmup, "ms_per_step": round(ms, 4), "higher_is_better": True, "dtype": "f32",
           "data": "synthetic (torso phantom seed 5, first timepoint)",
           "config": {"workload": "resample down to %s and back up to %s" % (list(cshape), list(a.shape))},
           "roofline": {"bound": "hbm", "achieved": round(alg / (k_ms * 1e-3) / 1e9, 1), "peak": HBM_PEAK_GBS,
                        "unit": "GB/s", "frac": round(alg / (k_ms * 1e-3) / 1e9 / HBM_PEAK_GBS, 4),
                        "traffic": read_traffic("resample_kernel_coarse_to_fine", "resample_512x512x400.md"),
                        "kernel": "resample_linear (coarse -> fine)", "kernel_ms": round(k_ms, 5),
                        "algorithmic_bytes": alg}}
    if not args.no_cpu:
        from oracle import resample as ors
        sub = ph.activity[0][:, :, :100]
        t0 = time.perf_counter()
        ors.resample(sub, fine, coarse, "linear")
        t_cpu = time.perf_counter() - t0
        n_cpu = int(np.prod(output_shape_for(sub.shape, fine, coarse)))
        res["cpu_baseline"] = {"value": n_cpu / t_cpu / 1e9, "unit": "Gvoxel/s", "cores": 1, "kind": "port",
                               "sample": f"scipy map_coordinates order 1 (the oracle) on a 512x512x100 slab, "
                                         f"{t_cpu:.2f} s"}
        got = down.cpu().numpy()
        exp = ors.resample(ph.activity[0][:64, :64, :64], fine, coarse, "linear")
        gsub = resample_device(torch.from_numpy(np.ascontiguousarray(ph.activity[0][:64, :64, :64])).to(dev),
                               fine, coarse, "linear").cpu().numpy()
        res["max_abs_err_vs_oracle"] = float(np.abs(gsub - exp).max())
        del got
    print(json.dumps(res), flush=True)


def bench_tissue(args):
    """HU -> (metal fill, 5 class masks as bits, density) of a 512x512x400 torso CT in one pass."""
    import numpy as np
    import torch

    from pyvoxeldosimetry_amd.phantoms import ct_hu_phantom
    from pyvoxeldosimetry_amd.tissue import HU_MATERIALS, TissueComposition

    dev = torch.device("cuda", 0)
    torch.cuda.set_device(dev)
    ct_np = ct_hu_phantom(seed=6)
    ct = torch.from_numpy(ct_np).to(dev)
    tc = TissueComposition()
    ms = _timed(lambda: tc.map(ct), args.steps, args.warmup)
    ev0, ev1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    ev0.record()
    reps = 20
    for _ in range(reps):
        corr, bits, dens = tc.map(ct)
    ev1.record()
    torch.cuda.synchronize()
    k_ms = ev0.elapsed_time(ev1) / reps
    n = ct.numel()
    alg = 13 * n                 # 4 B HU read; 4 B corrected HU, 1 B class bits, 4 B density written
    achieved = alg / (k_ms * 1e-3) / 1e9
    res = {"metric": "Gvoxel/s HU -> metal fill + tissue classes + density, 512x512x400 CT",
           "value": round(n / (ms * 1e-3) / 1e9, 3), "unit": "Gvoxel/s", "n_gpus": 1, "steps": args.steps,
           "warmup": args.warmup, "ms_per_step": round(ms, 4), "higher_is_better": True, "dtype": "f32",
           "data": "synthetic (ct_hu_phantom seed 6, two 3000 HU implants)",
           "config": {"workload": "tissue map 512x512x400 f32 HU, metal fill sigma 1 (r=4), 5 classes, "
                                  "16-material density", "metal_voxels": int((ct_np > 2000).sum())},
           "roofline": {"bound": "hbm", "achieved": round(achieved, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                        "frac": round(achieved / HBM_PEAK_GBS, 4),
                        "traffic": read_traffic("tissue_map4", "tissue_map_512x512x400.md"), "kernel": "tissue_map4",
                        "kernel_ms": round(k_ms, 5), "algorithmic_bytes": alg}}
    if not args.no_cpu:
        from oracle import tissue as ot
        slab = ct_np[:, :, :100]
        t0 = time.perf_counter()
        comp = ot.calculate_composition(slab)
        t_cpu = time.perf_counter() - t0
        res["cpu_baseline"] = {"value": slab.size / t_cpu / 1e9, "unit": "Gvoxel/s", "cores": 1, "kind": "port",
                               "sample": f"reference calculate_composition (scipy gaussian_filter + 5 masks, "
                                         f"float64) on a 512x512x100 slab, {t_cpu:.2f} s"}
        res["speedup_vs_cpu_reference"] = round(res["value"] / res["cpu_baseline"]["value"], 1)
        exp = ot.handle_artifacts(ct_np)
        got = corr.cpu().numpy()
        res["max_abs_err_hu"] = float(np.nanmax(np.abs(got.astype(np.float64) - exp)))
        dexp = ot.density_from_hu(exp, HU_MATERIALS).astype(np.float32)
        res["density_mismatches"] = int((dens.cpu().numpy() != dexp).sum())
        del comp
    print(json.dumps(res), flush=True)


if __name__ == "__main__":
    main()
