"""A NaN in the image reaches every voxel of the volume (its transform is NaN),
those without a weight included."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import deconwolf_amd as dw
from test_gpu_extended import _image, _psf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("method", [dw.METHOD_RL, dw.METHOD_SHB])
@pytest.mark.parametrize("shape,bq", [((12, 20, 24), 2), ((13, 23, 31), 1)])
def test_nan_reaches_the_whole_volume(method, shape, bq):
    print("NaN image:", method, shape, bq, flush=True)
    im, k = _image(shape), _psf((9, 15, 17), (4, 7, 8))
    im[3, 4, 5] = np.nan
    got = {}
    s = dw.DwOpts(nIter=4, iter_type=dw.ITER_FIXED, borderQuality=bq, fulldump=1, method=method,
                  iter_hook=lambda i, e, x: got.__setitem__(i, x))
    out = (dw.deconvolve_rl_hip if method == dw.METHOD_RL else dw.deconvolve_shb_hip)(im, k, s)
    assert np.isnan(out).all()
    assert np.isnan(got[-1]).all()


@pytest.mark.parametrize("method", [dw.METHOD_RL, dw.METHOD_SHB])
@pytest.mark.parametrize("where", ["image", "psf"])
def test_infinite_start_has_no_forward_model(method, where):
    """With an infinite value in the image (the flat start is infinite) or in the
    PSF, iteration 0's forward model is NaN, which the I-divergence does not count
    and the squared error hands on (getError, dw.c:1436-1524)."""
    print("infinite", where, method, flush=True)
    im, k = _image((12, 20, 24)), _psf((5, 7, 9), (2, 3, 4))
    if where == "image":
        im[3, 4, 5] = np.inf
    else:
        k[1, 2, 3] = np.inf
    run = dw.deconvolve_rl_hip if method == dw.METHOD_RL else dw.deconvolve_shb_hip
    for metric in (dw.METRIC_IDIV, dw.METRIC_MSE):
        s = dw.DwOpts(nIter=2, iter_type=dw.ITER_FIXED, method=method, metric=metric)
        run(im, k, s)
        if metric == dw.METRIC_IDIV:
            assert s.err_trace[0] == 0
        else:
            assert np.isnan(s.err_trace[0])


@pytest.mark.parametrize("scale", [1.0, 1e-3, 1e-6, 1e6])
@pytest.mark.parametrize("method", [dw.METHOD_RL, dw.METHOD_SHB])
def test_flat_model_scales_with_the_image(scale, method):
    """Iteration 0's forward model of a flat start, the start times the PSF's sum,
    to float32's rounding (2^-23 of it, twice) at every scale of the image."""
    print("flat model at scale", scale, method, flush=True)
    im = np.full((12, 3, 40), 3.0 * scale, np.float32)
    im[::2] *= 0.5
    k = np.ones((3, 2, 3), np.float32)
    k[1, 1, 1] = 5
    k /= k.sum()
    s = dw.DwOpts(nIter=1, iter_type=dw.ITER_FIXED, borderQuality=1, metric=dw.METRIC_MSE, method=method,
                  bg_auto=0, bg=0.0)
    (dw.deconvolve_rl_hip if method == dw.METHOD_RL else dw.deconvolve_shb_hip)(im, k, s)
    n = np.prod([float(v) for v in s.stats["ref_work"]])
    y = im.astype(np.float64).sum() / n * k.astype(np.float64).sum()
    d = im.astype(np.float64) - y
    # the start, the sum and their product are rounded to float32, the error too
    tol = 2 * np.abs(d).mean() * y * 4 * 2.0 ** -24 + (d ** 2).mean() * 2.0 ** -24
    assert abs(float(s.err_trace[0]) - (d ** 2).mean()) <= tol
