"""Algorithmic bytes of profiled passes: a job's totals are the same in an
engine as alone, and what the transform size gives, iteration 0 of a flat start
(no forward passes, no spectrum for the ratio pass) included."""
import pytest

torch = pytest.importorskip("torch")

import deconwolf_amd as dw
from deconwolf_amd import _lib
from deconwolf_amd.serve import Engine
from test_gpu_engine import make_job

pytestmark = pytest.mark.gpu
START = {"start_condition": dw.START_IDENTITY}


def profiled(f):
    _lib.profile_enable(True)
    try:
        f()
        torch.cuda.synchronize()
        return {k: (n, b) for k, (n, _, b) in _lib.profile_read().items()}
    finally:
        _lib.profile_enable(False)


@pytest.mark.parametrize("method", [dw.METHOD_SHB, dw.METHOD_RL])
@pytest.mark.parametrize("opt", [{}, START])
def test_bytes_alone_and_in_an_engine(method, opt):
    print("profiled bytes:", method, opt, flush=True)
    shape, n = (16, 36, 40), 5
    im, k, s = make_job(1, shape, (7, 9, 9), n, method=method, **opt)
    rl = method == dw.METHOD_RL
    solo = dw.deconvolve_rl_hip_device if rl else dw.deconvolve_shb_hip_device
    solo(im, k, s)  # measures the size's plans, whose trials would count
    alone = profiled(lambda: solo(im, k, s))
    eng = Engine(hbm_budget_gb=1.0, max_active=4)

    def run():
        eng.submit(0, im, k, s)
        while not eng.step():
            pass

    try:
        batch = profiled(run)
    finally:
        eng.close()
    assert batch == alone
    P, N, M = shape
    nx, ny, nz = s.stats["work"]
    row = 8 * (nx // 2 + 1)
    X, V, img, rows = row * ny * nz, 4 * nx * ny * nz, 4 * M * N * P, row * N * P
    flat = not opt
    assert alone["x_ratio"] == (n, n * (2 * rows + img) - (rows if flat else 0))
    first = 0 if flat else (1 if rl else 2) * V + X
    later = n - 1 + (1 if rl else 0)    # RL ends in one more update
    assert alone["x_update"] == (later + (0 if flat else 1), first + later * (2 * X + ((2 if rl else 3) + 1) * V))
    assert alone["y_fwd"][0] == (n - 1 if flat else n)
