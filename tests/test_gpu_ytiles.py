"""The y passes' two workgroup sizes: the longest pencil whose 16-column tile
fits the small workgroup (640 values) and the next one (648) against the
float32 oracle (relative L2 1e-5), SHB and RL, plain and extended; and a batch
that holds both kinds (its table runs the large workgroups) equal to the jobs
alone bit for bit."""
import copy

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import deconwolf_amd as dw
from deconwolf_amd.serve import Engine
from oracle import pyoracle as po
from test_gpu_shb import DEV, case, rel_l2

pytestmark = pytest.mark.gpu

# image (P, N, M), psf (pP, pN, pM), bq; transform rows 640, 648, and an
# extended y axis of 1 + 631 -> 640 and 641 + 8 -> 675 at most
CASES = [((6, 632, 21), (5, 9, 7), 2), ((6, 640, 21), (5, 9, 7), 2), ((7, 631, 24), (3, 9, 7), 0),
         ((7, 641, 24), (3, 9, 7), 0)]


@pytest.mark.parametrize("shape,psf_shape,bq", CASES)
@pytest.mark.parametrize("method", [dw.METHOD_SHB, dw.METHOD_RL])
def test_long_rows_match_oracle(shape, psf_shape, bq, method):
    print("y tiles:", shape, bq, method, flush=True)
    im, k = case(shape, psf_shape, seed=41)
    s = dw.DwOpts(nIter=4, iter_type=dw.ITER_FIXED, borderQuality=bq, method=method)
    out = (dw.deconvolve_rl_hip if method == dw.METHOD_RL else dw.deconvolve_shb_hip)(im, k, s)
    o32, e32, _, _ = (po.rl if method == dw.METHOD_RL else po.shb)(im, k, niter=4, border_quality=bq,
                                                                   work=s.stats["work"])
    assert rel_l2(out, o32) <= 1e-5
    np.testing.assert_allclose(s.err_trace, e32, rtol=1e-4)


def test_batch_of_both_sizes():
    print("y tiles: batch of both", flush=True)
    jobs = []
    for i, (shape, psf_shape, bq) in enumerate(CASES):
        im, k = case(shape, psf_shape, seed=50 + i)
        jobs.append((torch.from_numpy(im).to(DEV), torch.from_numpy(k).to(DEV),
                     dw.DwOpts(nIter=3 + i, iter_type=dw.ITER_FIXED, borderQuality=bq)))
    eng = Engine(hbm_budget_gb=1.0, max_active=8)
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
