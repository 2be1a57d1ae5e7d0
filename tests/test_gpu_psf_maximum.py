"""A PSF without a maximum (NaN in all of it, or no value above -inf) takes its
first value for it, on each path: the result is NaN, as its transform is, and
no value outside the PSF is read."""
import pytest

torch = pytest.importorskip("torch")

import deconwolf_amd as dw

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# image (P, N, M), psf (pP, pN, pM), bq: the plain passes, an extended job, and
# a depth that only the any-size path transforms
CASES = [((6, 20, 24), (5, 7, 7), 2), ((11, 23, 37), (7, 9, 9), 0), ((2503, 5, 8), (5, 3, 3), 0)]


@pytest.mark.parametrize("shape,psf_shape,bq", CASES)
@pytest.mark.parametrize("value", [float("nan"), -float("inf")])
def test_psf_without_a_maximum(shape, psf_shape, bq, value):
    print("no PSF maximum:", shape, bq, value, flush=True)
    im = torch.full(shape, 20.0, device=DEV)
    k = torch.full(psf_shape, value, device=DEV)
    s = dw.DwOpts(nIter=3, iter_type=dw.ITER_FIXED, borderQuality=bq)
    out = dw.deconvolve_shb_hip_device(im, k, s)
    assert bool(torch.isnan(out).all())
    assert (s.err_trace == 0).all()  # the I-divergence counts voxels with y > 0 (dw.c:1436-1524)
