"""y passes with enough tiles for the small workgroups (as many as there are
CUs): their longest pencil, plain and extended, SHB and RL, against the float32
oracle (relative L2 1e-5, error trace 1e-4); and a batch whose jobs reach that
number only together, equal to the jobs alone bit for bit."""
import copy

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import deconwolf_amd as dw
from deconwolf_amd.serve import Engine
from oracle import pyoracle as po
from test_gpu_shb import DEV, case, rel_l2

pytestmark = pytest.mark.gpu

# image (P, N, M), psf (pP, pN, pM), bq: one tile of 16 columns per plane and
# rows of 640 values; 260 and more planes
CASES = [((260, 632, 21), (5, 9, 7), 2), ((263, 631, 23), (3, 9, 7), 0)]


@pytest.mark.parametrize("shape,psf_shape,bq", CASES)
@pytest.mark.parametrize("method", [dw.METHOD_SHB, dw.METHOD_RL])
def test_small_workgroups_match_oracle(shape, psf_shape, bq, method):
    print("small y workgroups:", shape, bq, method, flush=True)
    im, k = case(shape, psf_shape, seed=43)
    s = dw.DwOpts(nIter=3, iter_type=dw.ITER_FIXED, borderQuality=bq, method=method)
    out = (dw.deconvolve_rl_hip if method == dw.METHOD_RL else dw.deconvolve_shb_hip)(im, k, s)
    o32, e32, _, _ = (po.rl if method == dw.METHOD_RL else po.shb)(im, k, niter=3, border_quality=bq,
                                                                   work=s.stats["work"])
    assert rel_l2(out, o32) <= 1e-5
    np.testing.assert_allclose(s.err_trace, e32, rtol=1e-4)


def test_batch_reaches_the_small_workgroups():
    print("small y workgroups: batch", flush=True)
    jobs = []
    for i in range(12):
        im, k = case((24, 40 + i, 36), (7, 9, 9), seed=60 + i)
        jobs.append((torch.from_numpy(im).to(DEV), torch.from_numpy(k).to(DEV),
                     dw.DwOpts(nIter=4 + i % 3, iter_type=dw.ITER_FIXED)))
    eng = Engine(hbm_budget_gb=1.0, max_active=16)
    try:
        for t, (im, k, s) in enumerate(jobs):
            eng.submit(t, im, k, s)
        done = 0
        while done < len(jobs):
            done += len(eng.step())
        for t, (im, k, s) in enumerate(jobs):
            ref = dw.deconvolve_shb_hip_device(im, k, copy.copy(s))
            out, _ = eng.result(t)
            assert torch.equal(out, ref), t
    finally:
        eng.close()
