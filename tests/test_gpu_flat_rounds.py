"""Iteration 0 of a flat start in the engine: its forward passes have no tiles
for the job (nothing is launched where no other job has any), and batches whose
jobs start flat, from an image or by the other method, some later than others,
give each job's own result bit for bit."""
import copy

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import deconwolf_amd as dw
from deconwolf_amd import _lib
from deconwolf_amd.serve import Engine
from test_gpu_engine import make_job, solo

pytestmark = pytest.mark.gpu

FLAT = [(1, (16, 36, 40), (7, 9, 9), 4, {}), (2, (10, 24, 30), (5, 7, 7), 4, {})]
START = {"start_condition": dw.START_IDENTITY}


def test_first_round_launches_no_forward_pass():
    print("flat rounds: launches", flush=True)
    for extra, per_pass in ((None, 3), ((3, (12, 40, 28), (7, 7, 5), 4, START), 4)):
        jobs = [make_job(sd, sh, ps, n, **o) for sd, sh, ps, n, o in FLAT + ([extra] if extra else [])]
        eng = Engine(hbm_budget_gb=1.0, max_active=8)
        try:
            for t, (im, k, s) in enumerate(jobs):
                eng.submit(t, im, k, s)
            _lib.profile_enable(True)
            done = []
            while len(done) < len(jobs):
                done += eng.step()
            p = _lib.profile_read()
        finally:
            _lib.profile_enable(False)
            eng.close()
        for k in ("x_update", "y_fwd", "z_conv", "y_inv_img"):
            assert p[k][0] == per_pass, (k, p[k])
        assert p["x_ratio"][0] == 4


JOBS = [(1, (16, 36, 40), (7, 9, 9), 12, {}), (2, (10, 24, 30), (5, 7, 7), 11, START),
        (3, (12, 40, 28), (7, 7, 5), 9, {"method": dw.METHOD_RL}), (4, (8, 20, 24), (5, 5, 5), 14, {}),
        (5, (11, 26, 43), (7, 7, 9), 10, {"iter_type": dw.ITER_REL, "err_rel": 0.02, "maxiter": 20})]


@pytest.mark.parametrize("groups", [1, 2])
@pytest.mark.parametrize("first", [5, 2])
def test_late_and_mixed_starts_equal_alone(groups, first):
    """`first` jobs at once, the others after one step of several rounds."""
    print("flat rounds: groups", groups, "first", first, flush=True)
    jobs = [make_job(sd, sh, ps, n, **o) for sd, sh, ps, n, o in JOBS]
    eng = Engine(hbm_budget_gb=1.0, max_active=8, groups=groups, rounds_per_step=5)
    try:
        for t in range(first):
            eng.submit(t, *jobs[t])
        done = list(eng.step())
        for t in range(first, len(jobs)):
            eng.submit(t, *jobs[t])
        while len(done) < len(jobs):
            done += eng.step()
        for t, (im, k, s) in enumerate(jobs):
            out, st = eng.result(t)
            if s.method == dw.METHOD_RL:
                s2 = copy.copy(s)
                ref = dw.deconvolve_rl_hip_device(im, k, s2).cpu().numpy()
            else:
                ref, s2 = solo(im, k, s)
            assert st["iterations"] == s2.stats["iterations"], t
            assert np.array_equal(out.cpu().numpy(), ref), t
            np.testing.assert_array_equal(st["err_trace"], s2.err_trace)
    finally:
        eng.close()
