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
