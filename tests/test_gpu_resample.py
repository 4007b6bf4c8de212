"""GPU tests of the grid resampler (include/pvd_resample.h) against oracle/resample.py,
and of the dose path with a voxel size other than the kernel resolution.

Tolerances: FP64 coordinates on both sides, FP32 interpolation on the GPU:
|diff| <= 1e-6 x max|image|.  Nearest is exact."""
import sys

import numpy as np
import pytest

from oracle import conv, dpk
from oracle import resample as ors

pytestmark = pytest.mark.gpu


def _say(*a):
    print("[gpu-case]", *a, file=sys.stderr, flush=True)


@pytest.mark.parametrize("sin,sout", [((2.0, 2.0, 2.0), (1.0, 1.0, 1.0)), ((1.0, 1.0, 1.0), (2.2, 2.2, 2.2)),
                                      ((0.98, 0.98, 2.5), (2.0, 1.3, 1.7)), ((3.0, 3.0, 3.0), (3.0, 3.0, 3.0))])
def test_resample_matches_oracle(sin, sout):
    from pyvoxeldosimetry_amd.resample import resample
    _say("resample", sin, sout)
    rng = np.random.default_rng(3)
    img = rng.normal(size=(33, 27, 41)).astype(np.float32)
    for mode in ("linear", "nearest"):
        got = resample(img, sin, sout, mode)
        exp = ors.resample(img, sin, sout, mode)
        assert got.shape == exp.shape
        if mode == "nearest":
            np.testing.assert_array_equal(got, exp.astype(np.float32))
        else:
            np.testing.assert_allclose(got, exp, rtol=0, atol=1e-6 * np.abs(img).max())


def test_activity_resampling_keeps_total():
    from pyvoxeldosimetry_amd.phantoms import create_spherical_activity
    from pyvoxeldosimetry_amd.resample import resample_activity
    _say("resample activity total")
    act = create_spherical_activity((64, 64, 64), (32, 32, 32), 12, 1000.0)
    from scipy.ndimage import gaussian_filter
    act = gaussian_filter(act, 2.0).astype(np.float32)            # smooth: interpolation keeps the integral
    down = resample_activity(act, (1.0,) * 3, (2.0,) * 3)
    up = resample_activity(act, (1.0,) * 3, (0.5,) * 3)
    assert down.sum() == pytest.approx(act.sum(), rel=2e-3)
    assert up.sum() == pytest.approx(act.sum(), rel=2e-3)


def test_dose_at_other_voxel_size_goes_through_the_kernel_grid():
    """2 mm activity, 1 mm Y-90 kernel: activity and density onto the 1 mm grid,
    convolution there, dose back onto the 2 mm grid (the reference's intended path)."""
    from pyvoxeldosimetry_amd import KernelConvolutionCalculator
    _say("dose with resampling")
    rng = np.random.default_rng(5)
    act = np.zeros((24, 20, 22), np.float32)
    act[8:14, 6:13, 9:15] = rng.uniform(1e4, 2e4, size=(6, 7, 6))
    rho = rng.uniform(0.8, 1.2, size=act.shape).astype(np.float32)
    calc = KernelConvolutionCalculator("Y90", "water", 1.0, {"kernel_grid": (15, 15, 15), "fix_kernel_centre": True,
                                                             "conv_mode": "linear"})
    got = calc.calculate_dose_rate(act, (2.0, 2.0, 2.0), density_map=rho)
    ak = ors.resample(act, (2.0,) * 3, (1.0,) * 3, "linear", scale=1.0 / 8.0)
    rk = ors.resample(rho, (2.0,) * 3, (1.0,) * 3, "linear", shape=ak.shape)
    dk = conv.epilogue(conv.linear_same(ak, dpk.y90_kernel(1.0, (15, 15, 15), fix_centre=True)), rk)
    exp = ors.resample(dk, (1.0,) * 3, (2.0,) * 3, "linear", shape=act.shape)
    assert got.shape == act.shape
    assert conv.error_metrics(got, exp)["max_rel"] < 1e-5


@pytest.mark.parametrize("sin,sout,shape", [((2.0, 2.0, 2.0), (0.98, 0.98, 0.98), (19, 23, 17)),
                                            ((0.98, 1.2, 2.5), (2.0, 1.0, 1.7), (41, 30, 22)),
                                            ((1.0, 1.0, 1.0), (1.0, 1.0, 1.0), (5, 1, 9)),
                                            ((1.0, 1.0, 1.0), (0.3, 0.4, 0.35), (2, 3, 4))])
def test_cubic_bspline_matches_oracle(sin, sout, shape):
    """interpolation='cubic' (sitkBSpline): mirror-boundary interpolating cubic B-spline;
    FP32 prefilter and evaluation against the FP64 oracle within 2e-6 of max|image|."""
    from pyvoxeldosimetry_amd.resample import resample
    _say("cubic", sin, sout, shape)
    rng = np.random.default_rng(sum(shape))
    img = rng.normal(size=shape).astype(np.float32)
    got = resample(img, sin, sout, "cubic")
    exp = ors.resample(img, sin, sout, "cubic")
    assert got.shape == exp.shape
    np.testing.assert_allclose(got, exp, rtol=0, atol=2e-6 * np.abs(img).max())


def test_resample_dose_map_shape_affine_and_values():
    from pyvoxeldosimetry_amd.core import resample_dose_map
    _say("resample_dose_map")
    rng = np.random.default_rng(9)
    dose = rng.random((30, 26, 21)).astype(np.float32)
    out, aff = resample_dose_map(dose, (2.0, 2.0, 2.5), (0.98, 1.5, 2.0))
    shape = tuple(int(np.ceil(n * i / o)) for n, i, o in zip(dose.shape, (2.0, 2.0, 2.5), (0.98, 1.5, 2.0)))
    assert out.shape == shape
    np.testing.assert_array_equal(aff, np.diag([0.98, 1.5, 2.0, 1.0]))
    exp = ors.resample(dose, (2.0, 2.0, 2.5), (0.98, 1.5, 2.0), "cubic", shape=shape)
    np.testing.assert_allclose(out, exp, rtol=0, atol=2e-6)


@pytest.mark.parametrize("shape,ratio", [
    ((3, 9, 300), (1.0, 1.0, 1.0)),          # more input columns than one tile
    ((5, 17, 64), (0.7, 0.31, 0.11)),        # many outputs per input row
    ((9, 40, 33), (1.3, 2.5, 2.5)),          # the coarsest linear ratio of the staged form
    ((9, 40, 70), (1.3, 2.51, 2.51)),        # just past it
    ((6, 64, 90), (1.0, 8.0, 8.0)),          # the coarsest cubic ratio of the staged form
    ((6, 64, 90), (1.0, 8.01, 8.01)),
    ((2, 49, 477), (0.9, 1.1, 0.8)),         # prefilter: y tile of 24 + 1, two z tiles
    ((49, 3, 14), (1.2, 0.5, 1.0)),          # prefilter: x chunk of 48 + 1, one z unit
    ((97, 25, 15), (0.6, 0.9, 0.77)),
    ((1, 1, 1), (0.4, 1.0, 3.0)),
])
def test_staged_interpolation_edges(shape, ratio):
    """Tile edges of the staged linear / cubic interpolation and of the B-spline prefilter,
    and both sides of the rules that choose it.  FP32 sums of at most 29 + 4 terms per axis
    with FP64 coordinates: linear 1e-6, cubic 2e-6 of max|image|."""
    from pyvoxeldosimetry_amd.resample import resample
    _say("staged", shape, ratio)
    rng = np.random.default_rng(sum(shape))
    img = rng.normal(size=shape).astype(np.float32)
    out_shape = tuple(max(1, int(np.ceil(n / r)) + 1) for n, r in zip(shape, ratio))     # past the far edge: zeros
    for mode, tol in (("linear", 1e-6), ("cubic", 2e-6)):
        got = resample(img, (1.0, 1.0, 1.0), ratio, mode, output_shape=out_shape, scale=1.0)
        exp = ors.resample(img, (1.0, 1.0, 1.0), ratio, mode, shape=out_shape)
        np.testing.assert_allclose(got, exp, rtol=0, atol=tol * np.abs(img).max())


@pytest.mark.parametrize("shape", [(40, 33, 29), (33, 25, 55), (70, 49, 81)])
def test_prefilter_windows_and_what_a_non_finite_sample_reaches(shape):
    """The prefilter at the edges of its windows (32 along x, 24 along y, 27 along z) against
    the FP64 FIR, 2e-6 of max|image| (rounding of three FP32 recursions), and one infinite
    sample: the outputs more than 14 + 2 samples from it along an axis stay as they were."""
    from pyvoxeldosimetry_amd.resample import resample
    _say("prefilter", shape)
    rng = np.random.default_rng(sum(shape))
    img = rng.normal(size=shape).astype(np.float32)
    got = resample(img, (1.0, 1.0, 1.0), (1.0, 1.0, 1.0), "cubic", output_shape=shape, scale=1.0)
    exp = ors.resample(img, (1.0, 1.0, 1.0), (1.0, 1.0, 1.0), "cubic", shape=shape)
    np.testing.assert_allclose(got, exp, rtol=0, atol=2e-6 * np.abs(img).max())
    at = (3, 2, 5)
    bad = img.copy()
    bad[at] = np.inf
    out = resample(bad, (1.0, 1.0, 1.0), (1.0, 1.0, 1.0), "cubic", output_shape=shape, scale=1.0)
    assert not np.isfinite(out[at])
    far = np.zeros(shape, bool)
    for a, p in enumerate(at):
        i = np.arange(shape[a]).reshape([-1 if b == a else 1 for b in range(3)])
        far |= np.abs(i - p) > 14 + 2
    np.testing.assert_allclose(out[far], got[far], rtol=0, atol=2e-6 * np.abs(img).max())


@pytest.mark.parametrize("shape,ratio", [
    ((9, 70, 40), (0.13, 0.07, 0.5)),        # four planes a workgroup, two left over, zeros past the end
    ((3, 9, 260), (0.5, 1.0, 0.5)),          # 513 + outputs along z: two tiles of a row's lanes
    ((2, 11, 330), (1.0, 0.9, 1.0)),         # more input columns than one tile
    ((5, 6, 700), (1.5, 1.2, 2.4)),
])
def test_linear_tiles_of_several_planes(shape, ratio):
    """The linear kernel's tiles (eight rows, 512 outputs or 320 input columns, up to four
    planes) and their remainders: FP32 products with FP64 coordinates, 1e-6 of max|image|."""
    from pyvoxeldosimetry_amd.resample import resample
    _say("linear tiles", shape, ratio)
    rng = np.random.default_rng(sum(shape))
    img = rng.normal(size=shape).astype(np.float32)
    out_shape = tuple(max(1, int(np.ceil(n / r)) + 1) for n, r in zip(shape, ratio))
    got = resample(img, (1.0, 1.0, 1.0), ratio, "linear", output_shape=out_shape, scale=1.0)
    exp = ors.resample(img, (1.0, 1.0, 1.0), ratio, "linear", shape=out_shape)
    np.testing.assert_allclose(got, exp, rtol=0, atol=1e-6 * np.abs(img).max())


@pytest.mark.parametrize("mode,size,out_size", [("linear", 1500, (24000, 24001)), ("cubic", 1500, (12000, 12001))])
def test_outputs_of_more_workgroups_than_one_launch_takes(mode, size, out_size):
    """A flat output whose tiles have 2^32 threads or more (17e6 and more workgroups of 256): the
    image is an outer product, so every output is the product of two one-dimensional results.
    FP32 interpolation along three axes on either side: 4e-6 of the largest product."""
    import torch
    from pyvoxeldosimetry_amd.resample import resample_device
    _say("resample beyond a launch", mode, out_size)
    gen = torch.Generator(device="cuda").manual_seed(3)
    g, h = (torch.randn(size, device="cuda", generator=gen) for _ in range(2))
    ratio = (size / out_size[0], size / out_size[1], 1.0)
    image = (g[:, None] * h[None, :]).reshape(size, size, 1).contiguous()
    out = torch.full((*out_size, 1), float("nan"), device="cuda")
    resample_device(image, (1.0,) * 3, ratio, mode, (*out_size, 1), out=out)
    G = resample_device(g.reshape(size, 1, 1), (1.0,) * 3, ratio, mode, (out_size[0], 1, 1)).reshape(-1)
    H = resample_device(h.reshape(1, size, 1), (1.0,) * 3, ratio, mode, (1, out_size[1], 1)).reshape(-1)
    tol = 4e-6 * float(G.abs().max() * H.abs().max())
    for i in range(0, out_size[0], 1000):
        d = (out[i:i + 1000, :, 0] - G[i:i + 1000, None] * H[None, :]).abs().max()
        assert float(d) <= tol, (i, float(d))              # (a NaN that was left fails)


def test_prefilter_of_more_workgroups_than_one_launch_takes():
    """A line of 540e6 voxels (either launch beyond 2^32 threads): every coefficient is written
    and those at both ends and around the launches' seam are a short line's (15 samples and
    more from its cuts; three FP32 recursions over other windows: 4e-6)."""
    import ctypes
    import torch
    from pyvoxeldosimetry_amd import _native as nat
    _say("prefilter beyond a launch")
    lib = nat.load()
    n = 540_000_001
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731

    def prefilter(x):
        coef, tmp = torch.full_like(x, float("nan")), torch.empty_like(x)
        torch.cuda.synchronize()
        nat.check(lib.pvd_bspline_prefilter(p(x), x.numel(), 1, 1, p(coef), p(tmp), None), "pvd_bspline_prefilter")
        torch.cuda.synchronize()
        return coef

    x = torch.rand(n, device="cuda", generator=torch.Generator(device="cuda").manual_seed(4))
    coef = prefilter(x)
    assert not bool(torch.isnan(coef).any())
    seam = (1 << 21) * 32
    for a in (0, seam - 2048, 8 * seam - 2048, n - 4096):
        part = prefilter(x[a:a + 4096].clone())
        lo, hi = (0 if a == 0 else 64), (4096 if a + 4096 == n else 4032)
        assert float((part[lo:hi] - coef[a + lo:a + hi]).abs().max()) <= 4e-6


@pytest.mark.parametrize("mode", ["nearest", "linear", "cubic"])
@pytest.mark.parametrize("m", [(410, 411, 409), (405, 406, 407)])
def test_outputs_on_either_side_of_the_streaming_threshold(mode, m):
    """Outputs above and below 256 MB (stored past the last-level cache, and through it): the
    image is an outer product, so every output is the product of three one-dimensional
    results.  FP32 interpolation along three axes on either side: 6e-6 of the largest
    product (nearest: two roundings)."""
    import torch
    from pyvoxeldosimetry_amd.resample import resample_device
    _say("streamed resample", mode, m)
    gen = torch.Generator(device="cuda").manual_seed(6)
    n = (61, 70, 83)
    f = [torch.randn(k, device="cuda", generator=gen) for k in n]
    ratio = tuple(a / b for a, b in zip(n, m))
    image = (f[0][:, None, None] * f[1][None, :, None] * f[2][None, None, :]).contiguous()
    out = torch.full(m, float("nan"), device="cuda")
    resample_device(image, (1.0,) * 3, ratio, mode, m, out=out)
    one = []
    for a in range(3):
        shape, size, r = [1, 1, 1], [1, 1, 1], [1.0, 1.0, 1.0]
        shape[a], size[a], r[a] = n[a], m[a], ratio[a]
        one.append(resample_device(f[a].reshape(shape), (1.0,) * 3, r, mode, tuple(size)).reshape(-1))
    want = one[0][:, None, None] * one[1][None, :, None] * one[2][None, None, :]
    top = float(want.abs().max())
    assert float((out - want).abs().max()) <= (2.0 ** -22 if mode == "nearest" else 6e-6) * top
