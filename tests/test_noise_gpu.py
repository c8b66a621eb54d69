"""The noise estimator's modes end to end on the GPU (inlm_denoise): the
semimanual mode (Noise/noiselevel.cpp:56-79) and the circular sampling mask
(:204-224), against the oracle's FP64 estimator on the same sample list and
the oracle's FP32 filter on the sigma lists the library used."""
import time

import numpy as np
import pytest

from microtomodenoise_amd import DenoiseParameters, IterativeNLM_GPU
from microtomodenoise_amd import _capi
from microtomodenoise_amd import phantom as ph
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def run_schedule(raw, p):
    nz, ny, nx = raw.shape
    g = IterativeNLM_GPU()
    assert g.configure_device([nx, ny, nz], p) == nz
    out, log = g.denoise(raw)
    g.free_device()
    return out, log


@pytest.mark.parametrize("mode,mask", [("semimanual", 0), ("z-adaptive", 70), ("global", 60), ("semimanual", 64)])
def test_noise_modes_schedule_vs_oracle(gpu_available, mode, mask):
    spec = ph.PhantomSpec((80, 72, 12), seed=61, radii=(3, 10), noise_sigma=1800.0, blur_sigma=0.8)
    raw = ph.make(spec)
    nz, ny, nx = raw.shape
    p = DenoiseParameters(radius_searchspace=[3, 3, 2], radius_patchspace=[1, 1, 1], maxiterations=3)
    p.noiselevel.mode = mode
    p.noiselevel.n_samples = 30000
    p.noiselevel.zwindow = 5
    p.noiselevel.sigma = [900.0, 0.0]
    p.noiselevel.circular_mask_diameter = mask
    print(f"[gpu] noise mode {mode} mask {mask}", flush=True)
    out, log = run_schedule(raw, p)

    samples = O.draw_samples((nx, ny, nz), 30000, 15, seed=0, mask_diameter=mask)
    assert np.array_equal(samples, _capi.draw_samples((nx, ny, nz), 30000, 15, 0, mask))
    op = O.Params(radius_searchspace=(3, 3, 2), radius_patchspace=(1, 1, 1), maxiterations=3, noise_mode=mode,
                  zwindow=5, sigma=(900.0, 0.0), blockwise=True)
    st = {}
    s0 = O.noiselevel(raw, samples, op, "f64", which=0, state=st).astype(np.float32)
    assert np.allclose(log[0], s0, rtol=2e-7, atol=0)
    out1 = O.filter_iteration(raw, raw, log[0], op)
    s1 = O.noiselevel(out1, samples, op, "f64", which=1, state=st)
    want1 = O.blend_sigma(log[0], s1.astype(np.float32), op.alpha)
    assert np.allclose(log[1], want1, rtol=2e-7, atol=0)
    if mode == "semimanual":
        assert np.all(log[0] == np.float32(900.0)) and np.unique(log[1]).size == 1
    want = O.iternlm(raw, op, sigma0=log[0], sigma1=log[1])
    assert np.array_equal(bits(out), bits(want))


def _noise_volume(kind):
    rng = np.random.default_rng(7)
    v = rng.normal(size=(9, 40, 70)).astype(np.float32) * 50 + 1000
    if kind == "flat":  # no sample varies: every patch std is zero
        v[:] = 3.0
    elif kind == "half-flat":  # zeros are left out; windows without a valid sample are filled from their neighbours
        v[:5] = 1.0
    elif kind == "two-level":
        v[:, :, 35:] *= 40
    elif kind == "outlier":  # a few samples so far off that both densities underflow
        v[4, 3, 3] = 1e12
    elif kind == "tiny":  # densities outside the range the logarithms decide
        v = (v - 1000) * np.float32(1e-30)
    return np.ascontiguousarray(v)


@pytest.mark.parametrize("n", [1, 2, 1023, 1024, 1025, 4097, 16384, 20479, 20480, 20737])
@pytest.mark.parametrize("kind", ["plain", "flat", "half-flat", "two-level", "outlier", "tiny"])
def test_clustering_on_the_gpu_equals_the_host(gpu_available, kind, n):
    """Both run the same steps in FP64 and differ by the order of at most
    2e4-term sums (about 1e-12 relative), so the float results agree to one
    unit in the last place (1.2e-7)."""
    raw = _noise_volume(kind)
    nz, ny, nx = raw.shape
    samples = _capi.draw_samples([nx, ny, nz], n, 15, 5)
    for mode, window in (("global", 0), ("z-adaptive", 4), ("z-adaptive", 100)):
        p = DenoiseParameters(radius_searchspace=[2, 2, 2], radius_patchspace=[1, 1, 1])
        p.noiselevel.mode = mode
        p.noiselevel.zwindow = window
        p.noiselevel.n_samples = n
        print(f"[gpu] clustering {kind} {mode} {window} n={n}", flush=True)
        g = IterativeNLM_GPU()
        assert g.configure_device([nx, ny, nz], p) == nz
        g.load_raw(raw)
        stds = g.patchstd(samples)
        got = g.estimate_noise(samples)
        g.free_device()
        want = _capi.sigma_from_patchstd(p.to_c(), [nx, ny, nz], samples, stds)
        assert np.allclose(got, want, rtol=2e-7, atol=0), (got, want)


def test_clustering_beyond_the_bits_in_lds(gpu_available):
    """More samples than the 2^20 whose assignments LDS keeps; the sums of
    1.1e6 terms differ by 1e-10 relative at most."""
    raw = _noise_volume("two-level")
    nz, ny, nx = raw.shape
    n = 1_100_003
    samples = _capi.draw_samples([nx, ny, nz], n, 15, 5)
    p = DenoiseParameters(radius_searchspace=[2, 2, 2], radius_patchspace=[1, 1, 1])
    p.noiselevel.mode = "global"
    p.noiselevel.n_samples = n
    print(f"[gpu] clustering n={n}", flush=True)
    g = IterativeNLM_GPU()
    assert g.configure_device([nx, ny, nz], p) == nz
    g.load_raw(raw)
    stds = g.patchstd(samples)
    got = g.estimate_noise(samples)
    g.free_device()
    want = _capi.sigma_from_patchstd(p.to_c(), [nx, ny, nz], samples, stds)
    assert np.allclose(got, want, rtol=2e-7, atol=0), (got, want)


@pytest.mark.parametrize("mode,window,n", [("global", 0, 20), ("global", 0, 200), ("z-adaptive", 4, 50), ("z-adaptive", 1, 300)])
def test_few_samples_cost_no_more_than_the_host_clustering(gpu_available, mode, window, n):
    """An estimate of a few samples takes the time of their patch statistics
    and the host's clustering (1.3 to 1.8 times that when clustered on the
    GPU), and gives its very result."""
    raw = _noise_volume("plain")
    nz, ny, nx = raw.shape
    samples = _capi.draw_samples([nx, ny, nz], n, 15, 5)
    p = DenoiseParameters(radius_searchspace=[2, 2, 2], radius_patchspace=[1, 1, 1])
    p.noiselevel.mode = mode
    p.noiselevel.zwindow = window
    p.noiselevel.n_samples = n
    g = IterativeNLM_GPU()
    assert g.configure_device([nx, ny, nz], p) == nz
    g.load_raw(raw)
    c = p.to_c()

    def whole():
        return g.estimate_noise(samples)

    def parts():
        return _capi.sigma_from_patchstd(c, [nx, ny, nz], samples, g.patchstd(samples))

    best = {whole: 1e9, parts: 1e9}
    assert np.array_equal(whole(), parts())
    for _ in range(300):
        for f in best:
            t = time.perf_counter()
            f()
            best[f] = min(best[f], time.perf_counter() - t)
    g.free_device()
    print(f"[gpu] {mode} n={n}: estimate {best[whole] * 1e6:.1f} us, parts {best[parts] * 1e6:.1f} us", flush=True)
    assert best[whole] < 1.15 * best[parts], best


@pytest.mark.parametrize("shape,n", [((70, 40, 9), 700_001), ((70, 40, 9), 1_100_003), ((70, 40, 64), 1_100_003)])
def test_large_windows_on_the_gpu_equal_the_host(gpu_available, shape, n):
    """z windows of one list: 7e5 samples, whose bits take more than 64 KB of
    LDS, and 1.1e6, for which the kernel derives the last assignment again
    instead of keeping bits; the sums of a window's 6e5 terms differ by 1e-10
    relative at most."""
    nx, ny, nz = shape
    rng = np.random.default_rng(7)
    raw = rng.normal(size=(nz, ny, nx)).astype(np.float32) * 50 + 1000
    raw[:, :, 35:] *= 40
    samples = _capi.draw_samples([nx, ny, nz], n, 15, 5)
    p = DenoiseParameters(radius_searchspace=[2, 2, 2], radius_patchspace=[1, 1, 1])
    p.noiselevel.mode = "z-adaptive"
    p.noiselevel.zwindow = 4
    p.noiselevel.n_samples = n
    print(f"[gpu] clustering {shape} n={n}", flush=True)
    g = IterativeNLM_GPU()
    assert g.configure_device([nx, ny, nz], p) == nz
    g.load_raw(raw)
    stds = g.patchstd(samples)
    got = g.estimate_noise(samples)
    g.free_device()
    want = _capi.sigma_from_patchstd(p.to_c(), [nx, ny, nz], samples, stds)
    assert np.unique(want).size > 1
    assert np.allclose(got, want, rtol=2e-7, atol=0), (got, want)
