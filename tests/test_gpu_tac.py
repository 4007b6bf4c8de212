"""GPU tests of the voxelwise TAC fits (include/pvd_tac.h) against oracle/tac.py
(scipy.optimize.curve_fit per voxel, as the reference).

Tolerances: both solvers converge to the weighted least-squares minimum with
MINPACK's default relative tolerance 1.49e-8; the GPU stores float32, so
well-conditioned parameters agree to ~1e-5 relative.
For models whose minimum is not unique on the sampled times (f3, bi-exponential),
the test checks that the GPU reaches a cost no higher than scipy's on at least
95 % of the voxels (a different descent path may end in another local minimum)."""
import sys

import numpy as np
import pytest

from oracle import tac

pytestmark = pytest.mark.gpu
T4 = [4.0, 24.0, 72.0, 144.0]
T6 = [1.0, 4.0, 24.0, 48.0, 96.0, 168.0]


def _say(*a):
    print("[gpu-case]", *a, file=sys.stderr, flush=True)


def _maps(y, shape):
    return [np.ascontiguousarray(y[:, i].reshape(shape), dtype=np.float32) for i in range(y.shape[1])]


def test_basic_fit_matches_curve_fit():
    from pyvoxeldosimetry_amd.time_integration import TimeCurveFitting
    _say("tac basic")
    rng = np.random.default_rng(0)
    shape = (8, 9, 10)
    n = int(np.prod(shape))
    A0 = rng.uniform(1e3, 1e5, n)
    lam = rng.uniform(0.004, 0.06, n)
    y = A0[:, None] * np.exp(-lam[:, None] * np.array(T4)) * rng.normal(1.0, 0.03, (n, 4))
    y[0] = 0.0                                   # all-zero voxel: p0 = (0, lambda), accumulated 0
    y[1] = [5.0, 10.0, 20.0, 40.0]               # growing curve: negative rate
    y = y.astype(np.float32).astype(np.float64)  # the GPU reads float32 maps
    w = [1.0, 2.0, 1.0, 0.5]
    tcf = TimeCurveFitting(64.1)
    p, acc = tcf.fit_time_activity_curve(T4, _maps(y, shape), weight_factors=w)
    assert p.shape == (2,) + shape and acc.shape == shape and p.dtype == np.float64
    pe, acce = tac.fit_basic(T4, y, 64.1, weights=w)
    np.testing.assert_allclose(p.reshape(2, -1), pe, rtol=2e-5, atol=1e-9)
    np.testing.assert_allclose(acc.reshape(-1), acce, rtol=5e-5)
    assert p.reshape(2, -1)[1, 0] == pytest.approx(np.log(2) / 64.1, rel=1e-6) and acc.reshape(-1)[0] == 0.0


@pytest.mark.parametrize("model,name", [("nukfit", "f2"), ("nukfit", "f3a"), ("lmfit", "mono-exponential"),
                                        ("nukfit", "f4a"), ("lmfit", "bi-exponential")])
def test_advanced_fit_reaches_the_least_squares_minimum(model, name):
    from pyvoxeldosimetry_amd.time_integration import TimeCurveFitting
    _say("tac advanced", model, name)
    rng = np.random.default_rng(hash(name) % 1000)
    hl = 64.1
    lp = np.log(2) / hl
    nuk, lmf = tac.models(hl, lp)
    f, p0 = (nuk if model == "nukfit" else lmf)[name]
    n = 120
    truth = {"f2": lambda: [rng.uniform(1, 5), rng.uniform(0.005, 0.05)],
             "f3a": lambda: [rng.uniform(1, 5), rng.uniform(0.2, 0.8), rng.uniform(0.02, 0.2)],
             "mono-exponential": lambda: [rng.uniform(1, 5), rng.uniform(20, 120)],
             "f4a": lambda: [rng.uniform(1, 3), rng.uniform(0.05, 0.2), rng.uniform(0.5, 1.5), rng.uniform(0.0, 0.01)],
             "bi-exponential": lambda: [rng.uniform(1, 5), rng.uniform(60, 120), rng.uniform(2, 10)]}[name]
    y = np.array([f(np.array(T6), *truth()) for _ in range(n)]) * rng.normal(1.0, 0.02, (n, len(T6)))
    y = y.astype(np.float32).astype(np.float64)
    shape = (4, 5, 6)
    tcf = TimeCurveFitting(hl)
    p, auc, info = tcf.fit_time_activity_curve_advanced(T6, _maps(y, shape), model=model, model_name=name,
                                                         return_fit_params=True)
    pe, auce, oke = tac.fit_advanced(T6, y, hl, model, name)
    pg = p.reshape(len(p0), -1)
    okg = np.array(info["success"])
    assert info["model_name"] == name and len(info["params"]) == n
    both = okg & oke
    assert okg.mean() >= 0.95 and both.mean() >= 0.9
    cg = np.array([tac.weighted_cost(f, T6, y[i], pg[:, i]) for i in range(n)])
    ce = np.array([tac.weighted_cost(f, T6, y[i], pe[:, i]) for i in range(n)])
    scale = np.array([np.sum(yy ** 2) for yy in y])
    as_good = cg[both] <= ce[both] * (1 + 1e-4) + 1e-9 * scale[both]
    if name in ("f2", "mono-exponential"):       # a unique minimum: the same parameters
        assert as_good.all()
        np.testing.assert_allclose(pg[:, both], pe[:, both], rtol=1e-4, atol=1e-7)
        np.testing.assert_allclose(auc.reshape(-1)[both], auce[both], rtol=1e-4)
    else:                                         # several local minima: a minimum at least as good, nearly always
        _say(f"{name}: GPU cost <= scipy cost on {as_good.mean():.3f} of {both.sum()} voxels")
        assert as_good.mean() >= 0.95
    # the integral is the trapezoid of the returned fit
    for i in np.nonzero(okg)[0][:20]:
        assert auc.reshape(-1)[i] == pytest.approx(tac.trapezoid(f(np.array(T6), *pg[:, i]), T6), rel=1e-5)


def test_more_parameters_than_samples_fail_like_the_reference():
    from pyvoxeldosimetry_amd.time_integration import TimeCurveFitting
    _say("tac underdetermined")
    y = np.array([[10.0, 8.0, 5.0, 3.0]] * 64)
    p, auc, info = TimeCurveFitting(64.1).fit_time_activity_curve_advanced(
        T4, _maps(y, (4, 4, 4)), "nukfit", "f4b", return_fit_params=True)
    assert not p.any() and not auc.any() and not any(info["success"])
    with pytest.raises(ValueError):
        TimeCurveFitting(64.1).fit_time_activity_curve_advanced(T4, _maps(y, (4, 4, 4)), model="other")


@pytest.mark.parametrize("T", [2, 4, 5, 8, 9, 16])
def test_sample_counts_of_the_compiled_forms(T):
    """Every compiled sample count at its edges (up to 4, 8, 16 samples): the basic fit against
    curve_fit, tolerances as above."""
    from pyvoxeldosimetry_amd.time_integration import TimeCurveFitting
    _say("tac sample counts", T)
    rng = np.random.default_rng(T)
    shape = (4, 5, 13)                              # 260 voxels: one past a block
    n = int(np.prod(shape))
    times = list(np.linspace(2.0, 150.0, T))
    A0 = rng.uniform(1e3, 1e5, n)
    lam = rng.uniform(0.004, 0.06, n)
    y = A0[:, None] * np.exp(-lam[:, None] * np.array(times)) * rng.normal(1.0, 0.02, (n, T))
    y = y.astype(np.float32).astype(np.float64)
    tcf = TimeCurveFitting(64.1)
    p, acc = tcf.fit_time_activity_curve(times, _maps(y, shape))
    pe, acce = tac.fit_basic(times, y, 64.1)
    np.testing.assert_allclose(p.reshape(2, -1), pe, rtol=2e-5, atol=1e-9)
    np.testing.assert_allclose(acc.reshape(-1), acce, rtol=5e-5)


@pytest.mark.parametrize("T", [4, 6, 8, 9, 16])
@pytest.mark.parametrize("model,name,centre", [("nukfit", "f3", [3.0, 0.02, 0.3]), ("nukfit", "f3a", [3.0, 0.6, 0.1]),
                                               ("nukfit", "f4a", [3.0, 0.15, 1.0, 0.01]),
                                               ("nukfit", "f4b", [4.0, 0.02, 2.0, 0.15, 0.8]),
                                               ("nukfit", "f4c", [3.0, 0.02, 1.0, 0.1, 0.8]),
                                               ("lmfit", "bi-exponential", [3.0, 80.0, 6.0]),
                                               ("lmfit", "tri-exponential", [4.0, 90.0, 2.0, 15.0, 2.0])])
def test_models_of_three_to_five_parameters_at_each_sample_count(T, model, name, centre):
    """Every compiled form of the larger models, through the C ABI: noise-free curves whose
    parameters lie within 10 % of the start are fitted and recovered.  The same iteration in
    FP64 numpy recovers them within 8e-6 (FP32 samples) and the curve within 7e-8 of its
    largest value; five FP32 parameters of a few units add 6e-7: tolerances 2e-5 and 2e-6.
    Fewer samples than parameters: fail_params and status 0."""
    import ctypes
    import torch
    from pyvoxeldosimetry_amd import _native as nat
    _say("tac larger models", name, T)
    lib = nat.load()
    rng = np.random.default_rng(T)
    n, k = 260, len(centre)                         # one past a block
    hl = 64.1
    f = tac.models(hl, np.log(2) / hl)[model == "lmfit"][name][0]
    t = np.geomspace(0.5, 160.0, T)
    truth = np.array(centre) * rng.uniform(0.9, 1.1, (n, k))
    y = np.array([f(t, *p) for p in truth]).astype(np.float32)
    q = nat.TacParams()
    q.model = {"f3": 2, "f3a": 3, "f4a": 4, "f4b": 5, "f4c": 6, "bi-exponential": 8, "tri-exponential": 9}[name]
    q.n_times, q.lambda_phys, q.max_iter, q.tol, q.auc_mode = T, np.log(2) / hl, 3333, 1.49012e-8, 1
    for i in range(T):
        q.t[i], q.w[i] = t[i], 1.0
    for i in range(k):
        q.p0[i], q.fail_params[i] = centre[i], 0.25 * centre[i]
    maps = [torch.from_numpy(np.ascontiguousarray(y[:, i])).cuda() for i in range(T)]
    params, auc = torch.empty((k, n), device="cuda"), torch.empty(n, device="cuda")
    status = torch.full((n,), 7, dtype=torch.uint8, device="cuda")
    ptr = lambda x: ctypes.c_void_p(x.data_ptr())  # noqa: E731
    torch.cuda.synchronize()
    nat.check(lib.pvd_tac_fit(ctypes.byref(q), (ctypes.c_void_p * T)(*[m.data_ptr() for m in maps]), n, ptr(params),
                              ptr(auc), ptr(status), None), "pvd_tac_fit")
    torch.cuda.synchronize()
    p, s, a = params.cpu().double().numpy(), status.cpu().numpy(), auc.cpu().numpy()
    if T < k:
        assert not s.any()
        np.testing.assert_allclose(p, np.tile(0.25 * np.array(centre)[:, None], n), rtol=1e-6)
    else:
        assert (s == 1).all()
        np.testing.assert_allclose(p.T, truth, rtol=2e-5)
    got = np.array([f(t, *p[:, i]) for i in range(n)])
    if T >= k:
        assert (np.abs(got - y).max(1) <= 2e-6 * np.abs(y).max(1)).all()
    scale = np.array([tac.trapezoid(np.abs(g), t) for g in got])
    np.testing.assert_array_less(np.abs(a - np.array([tac.trapezoid(g, t) for g in got])), 1e-5 * scale + 1e-30)
