"""GPU tests of extended jobs: border quality 0 and 1 at deconwolf's exact
work size (method_shb.c:137-153), a circular convolution whose period the
fused passes cannot transform, computed at a longer length with the data
continued periodically.  Sizes where the continuation can go wrong: a PSF as
long as the period, one whose maximum sits at an end (the continuation is
then all on one side), even PSF lengths, one axis extended and the others
not, one-value axes, rows that end within a tile.  Against the float32
oracle, with the bars of the any-size tests (relative L2 1e-5, error trace
1e-4); and the calls that stay on the any-size path: a depth no padded plan
covers, and a job whose padded spectra exceed the static block."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import deconwolf_amd as dw
from deconwolf_amd import synth
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rel_l2(a, b):
    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def _psf(shape, at):
    """Asymmetric PSF with its maximum at `at`, sum 1."""
    d = [np.arange(n) - a for n, a in zip(shape, at)]
    g = [np.exp(-0.5 * np.where(v < 0, v / 0.9, v / 1.7) ** 2) for v in d]
    k = g[0][:, None, None] * g[1][None, :, None] * g[2][None, None, :]
    return (k / k.sum()).astype(np.float32)


def _image(shape, seed=3):
    rng = np.random.default_rng(seed)
    V = synth.point_sources(shape, 20, rng=rng)
    V = synth.blur(V, synth.gaussian_psf(5, 5, 5 if shape[0] > 4 else 1, 1.2, 1.2, 1.2))
    return synth.noisy_image(V, 60.0, rng=rng) + np.float32(5.0)


# image (P, N, M), psf (pP, pN, pM), maximum at, bq
CASES = [
    ((11, 23, 37), (11, 23, 37), (5, 11, 18), 0),   # PSF as long as the period
    ((11, 23, 37), (7, 9, 9), (0, 0, 0), 0),        # maximum at the first value
    ((11, 23, 37), (7, 9, 9), (6, 8, 8), 0),        # and at the last
    ((13, 22, 33), (6, 8, 10), (2, 3, 6), 1),       # even lengths
    ((16, 24, 37), (5, 7, 7), (2, 3, 3), 0),        # x alone
    ((16, 29, 36), (5, 7, 7), (2, 3, 3), 0),        # y alone
    ((17, 24, 36), (5, 7, 7), (2, 1, 3), 0),        # z alone
    ((1, 37, 41), (1, 7, 7), (0, 3, 3), 0),         # one plane
    ((19, 1, 41), (5, 1, 7), (2, 0, 3), 0),         # one row per plane
    ((9, 131, 211), (5, 31, 41), (2, 15, 20), 1),   # several x tiles per plane, the last one short
]


@pytest.mark.parametrize("shape,psf_shape,at,bq", CASES)
@pytest.mark.parametrize("method", [dw.METHOD_SHB, dw.METHOD_RL])
def test_extended_matches_oracle(shape, psf_shape, at, bq, method):
    print("extended:", shape, psf_shape, at, "bq", bq, "method", method, flush=True)
    im, k = _image(shape), _psf(psf_shape, at)
    w, r, rc = dw.work_size(im.shape, k.shape, bq)
    assert rc == 0 and w == r
    s = dw.DwOpts(nIter=4, iter_type=dw.ITER_FIXED, borderQuality=bq, method=method)
    run = dw.deconvolve_rl_hip if method == dw.METHOD_RL else dw.deconvolve_shb_hip
    out = run(im, k, s)
    assert tuple(s.stats["work"]) == tuple(r)
    orun = po.rl if method == dw.METHOD_RL else po.shb
    o32, e32, bg, n = orun(im, k, niter=4, border_quality=bq)
    assert n == 4 and s.bg == np.float32(bg)
    assert rel_l2(out, o32) <= 1e-5
    np.testing.assert_allclose(s.err_trace, e32, rtol=1e-4)


def test_full_result_of_odd_rows():
    """The full-size hook hands out the period's volume (odd rows, no padding)."""
    print("extended: full-size hook", flush=True)
    im, k = _image((12, 26, 37)), _psf((7, 9, 9), (3, 4, 4))
    got = {}
    s = dw.DwOpts(nIter=3, iter_type=dw.ITER_FIXED, borderQuality=0, fulldump=1,
                  iter_hook=lambda i, e, x: got.__setitem__(i, x))
    out = dw.deconvolve_shb_hip(im, k, s)
    assert got[-1].shape == (12, 26, 37)
    np.testing.assert_array_equal(got[-1], out)


def test_depth_beyond_padded_plans():
    """A prime depth above the longest z transform stays on the any-size path."""
    print("extended: depth 2503", flush=True)
    im, k = _image((2503, 5, 8)), _psf((5, 3, 3), (2, 1, 1))
    s = dw.DwOpts(nIter=3, iter_type=dw.ITER_FIXED, borderQuality=0)
    out = dw.deconvolve_shb_hip(im, k, s)
    o32, _, _, _ = po.shb(im, k, niter=3, border_quality=0)
    assert rel_l2(out, o32) <= 1e-5


def test_static_block_takes_what_it_took():
    """A job whose padded spectra exceed the static block runs there on the
    any-size path, as before, and agrees with the extended run (two float32
    transforms of one volume: 1e-5, as against the oracle)."""
    print("extended: static block", flush=True)
    im = torch.from_numpy(_image((151, 211, 257))).to(DEV)
    k = torch.from_numpy(synth.gaussian_psf(111, 111, 111, 3.0, 3.0, 3.0)).to(DEV)
    s1 = dw.DwOpts(nIter=2, iter_type=dw.ITER_FIXED, borderQuality=0)
    s2 = dw.DwOpts(nIter=2, iter_type=dw.ITER_FIXED, borderQuality=0)
    a = dw.deconvolve_shb_hip_device(im, k, s1)
    b = dw.deconvolve_shb_hip_device_noalloc(im, k, s2, torch.empty_like(im))
    assert rel_l2(b.cpu(), a.cpu()) <= 1e-5
    np.testing.assert_allclose(s2.err_trace, s1.err_trace, rtol=1e-4)
