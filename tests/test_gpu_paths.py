"""Sizes on both sides of the rule between extended jobs and the any-size path,
and one voxel wide or deep, against the float32 oracle (relative L2 1e-5, error
trace 1e-4, the any-size tests' bars)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import deconwolf_amd as dw
from oracle import pyoracle as po
from test_gpu_extended import _image, _psf, rel_l2

pytestmark = pytest.mark.gpu

# image (P, N, M), psf (pP, pN, pM), maximum at, bq
CASES = [
    ((1200, 25, 25), (5, 9, 9), (2, 4, 4), 0),          # extended, four z columns
    ((1344, 25, 25), (5, 9, 9), (2, 4, 4), 0),          # any-size, no Bluestein axis
    ((701, 23, 25), (701, 23, 25), (350, 11, 12), 0),   # any-size, PSF as long as the period
    ((1341, 20, 20), (5, 9, 9), (0, 8, 0), 1),          # any-size with weights
    ((2503, 5, 1), (5, 3, 1), (2, 1, 0), 0),            # one column, any-size
    ((31, 37, 1), (5, 3, 1), (2, 1, 0), 0),             # one column, extended
]


@pytest.mark.parametrize("shape,psf_shape,at,bq", CASES)
@pytest.mark.parametrize("method", [dw.METHOD_SHB, dw.METHOD_RL])
def test_both_sides_of_the_rule(shape, psf_shape, at, bq, method):
    print("paths:", shape, psf_shape, at, "bq", bq, "method", method, flush=True)
    im, k = _image(shape), _psf(psf_shape, at)
    s = dw.DwOpts(nIter=4, iter_type=dw.ITER_FIXED, borderQuality=bq, method=method)
    out = (dw.deconvolve_rl_hip if method == dw.METHOD_RL else dw.deconvolve_shb_hip)(im, k, s)
    o32, e32, _, _ = (po.rl if method == dw.METHOD_RL else po.shb)(im, k, niter=4, border_quality=bq)
    assert rel_l2(out, o32) <= 1e-5
    np.testing.assert_allclose(s.err_trace, e32, rtol=1e-4)


def test_extended_job_takes_a_cached_plan(tmp_path):
    """A plan cached for the transform length of an extended job (37 x 23 x 11 with
    a 9 x 9 x 7 PSF: 48 x 32 x 18) is the one it runs."""
    print("paths: cached plan of an extended job", flush=True)
    f = tmp_path / "plans.txt"
    f.write_text("gfx950 48 32 18 x=4,6 xrows=7 y=4,8 ycols=8 z=3,6 zcols=4\n")
    im, k = _image((11, 23, 37)), _psf((7, 9, 9), (3, 4, 4))
    o32, e32, _, _ = po.shb(im, k, niter=4, border_quality=0)
    outs = []
    try:
        for path in ("", str(f)):
            dw.plan_cache_path(path)
            assert dw.plan_get((48, 32, 18))[0] == bool(path)
            s = dw.DwOpts(nIter=4, iter_type=dw.ITER_FIXED, borderQuality=0)
            outs.append(dw.deconvolve_shb_hip(im, k, s))
            assert rel_l2(outs[-1], o32) <= 1e-5
            np.testing.assert_allclose(s.err_trace, e32, rtol=1e-4)
    finally:
        dw.plan_cache_path("")
    assert not np.array_equal(*outs)    # other radices round differently
