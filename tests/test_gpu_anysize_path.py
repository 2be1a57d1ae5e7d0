"""The any-size path itself: jobs whose extended layout does not fit (an engine
whose budget is what dwhip_job_bytes names, a device without room) or does not
exist (a depth no padded plan covers), SHB and RL, with and without weights, MSE
and REL, beside fused jobs, the full-size hook.  Against the float32 oracle
(relative L2 1e-5, error trace 1e-4).  Each test asserts the path: fused and
extended jobs launch the update pass, any-size jobs none of the profiled ones."""
import copy
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import deconwolf_amd as dw
from deconwolf_amd import _lib
from deconwolf_amd.serve import Engine
from oracle import pyoracle as po
from test_gpu_extended import _image, _psf, rel_l2

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def job_bytes(shape, psf_shape, bq, niter):
    w, _, rc = dw.work_size(shape, psf_shape, bq)
    assert rc == 0
    n = _lib.lib().dwhip_job_bytes((ctypes.c_int64 * 3)(*w), *shape[::-1], *psf_shape[::-1], bq, niter)
    return (n + 4095) // 4096 * 4096


def updates(f):
    """Update passes launched while f runs."""
    _lib.profile_enable(True)
    try:
        f()
        torch.cuda.synchronize()
        return _lib.profile_read().get("x_update", (0,))[0]
    finally:
        _lib.profile_enable(False)


def drive(jobs, budget):
    """[(out, stats)] of (im, psf, opts) jobs through an engine of `budget` bytes."""
    eng = Engine(hbm_budget_gb=budget / 2 ** 30, max_active=8)
    try:
        for t, (im, k, s) in enumerate(jobs):
            eng.submit(t, torch.from_numpy(im).to(DEV), torch.from_numpy(k).to(DEV), s)
        n = 0
        while n < len(jobs):
            n += len(eng.step())
        return [(o.cpu().numpy(), st) for o, st in (eng.result(t) for t in range(len(jobs)))]
    finally:
        eng.close()


# image (P, N, M), psf (pP, pN, pM), maximum at, bq
CASES = [
    ((31, 53, 74), (7, 9, 9), (3, 4, 4), 0),        # 74 x 53 x 31: primes 37, 53, 31
    ((20, 61, 101), (7, 9, 9), (3, 4, 4), 1),       # 106 x 66 x 24 with weights: 53, 11
    ((27, 81, 105), (7, 9, 31), (0, 8, 0), 0),      # odd x, no Bluestein, 2187 rows: an odd number
    ((29, 59, 97), (29, 59, 97), (14, 29, 48), 0),  # primes, PSF as long as the period, 1711 rows
    ((17, 64, 92), (6, 8, 10), (2, 3, 6), 1),       # 97 x 68 x 20 with weights
]


@pytest.mark.parametrize("shape,psf_shape,at,bq", CASES)
@pytest.mark.parametrize("method", [dw.METHOD_SHB, dw.METHOD_RL])
def test_engine_of_the_least_budget(shape, psf_shape, at, bq, method):
    print("any-size in an engine:", shape, psf_shape, "bq", bq, "method", method, flush=True)
    im, k = _image(shape), _psf(psf_shape, at)
    s = dw.DwOpts(nIter=6, iter_type=dw.ITER_FIXED, borderQuality=bq, method=method)
    got = []
    assert updates(lambda: got.extend(drive([(im, k, s)], job_bytes(shape, psf_shape, bq, 6)))) == 0
    o32, e32, bg, _ = (po.rl if method == dw.METHOD_RL else po.shb)(im, k, niter=6, border_quality=bq)
    out, st = got[0]
    assert st["iterations"] == 6 and st["bg"] == np.float32(bg)
    assert rel_l2(out, o32) <= 1e-5
    np.testing.assert_allclose(st["err_trace"], e32, rtol=1e-4)
    # with room for it the same job runs extended
    assert updates(lambda: drive([(im, k, s)], 1 << 30)) > 0


@pytest.mark.parametrize("metric", [dw.METRIC_MSE, dw.METRIC_IDIV])
def test_rel_rule(metric):
    print("any-size in an engine: REL, metric", metric, flush=True)
    shape, ps = (20, 61, 101), (7, 9, 9)
    im, k = _image(shape), _psf(ps, (3, 4, 4))
    s = dw.DwOpts(iter_type=dw.ITER_REL, err_rel=0.02, maxiter=40, borderQuality=1, metric=metric)
    got = []
    assert updates(lambda: got.extend(drive([(im, k, s)], job_bytes(shape, ps, 1, 40)))) == 0
    o32, e32, _, n = po.shb(im, k, iter_type=po.ITER_REL, err_rel=0.02, maxiter=40, border_quality=1, metric=metric)
    out, st = got[0]
    assert st["iterations"] == n > 1
    assert rel_l2(out, o32) <= 1e-5
    np.testing.assert_allclose(st["err_trace"], e32, rtol=1e-4)


def test_beside_fused_jobs():
    """An any-size job and fused jobs in one engine, FIXED and REL: each result
    bit-identical to the same job's alone (the any-size one in an engine of its own)."""
    print("any-size beside fused jobs", flush=True)
    big, bps = (29, 59, 97), (29, 59, 97)
    jobs = [(_image(big), _psf(bps, (14, 29, 48)), dw.DwOpts(nIter=7, iter_type=dw.ITER_FIXED, borderQuality=0)),
            (_image((10, 24, 30)), _psf((5, 7, 7), (2, 3, 3)), dw.DwOpts(nIter=5, iter_type=dw.ITER_FIXED)),
            (_image((8, 20, 24)), _psf((5, 5, 5), (2, 2, 2)),
             dw.DwOpts(iter_type=dw.ITER_REL, err_rel=0.01, maxiter=20))]
    need = job_bytes(big, bps, 0, 7)
    got = drive(jobs, need + job_bytes((10, 24, 30), (5, 7, 7), 2, 5) + job_bytes((8, 20, 24), (5, 5, 5), 2, 20))
    alone = []
    assert updates(lambda: alone.extend(drive(jobs[:1], need))) == 0
    assert np.array_equal(got[0][0], alone[0][0])
    np.testing.assert_array_equal(got[0][1]["err_trace"], alone[0][1]["err_trace"])
    for (im, k, s), (out, st) in list(zip(jobs, got))[1:]:
        s2 = copy.copy(s)
        ref = dw.deconvolve_shb_hip(im, k, s2)
        assert st["iterations"] == s2.stats["iterations"]
        assert np.array_equal(out, ref)


def test_full_size_hook():
    print("any-size: full-size hook", flush=True)
    im, k = _image((2503, 3, 7)), _psf((5, 3, 3), (2, 1, 1))
    for method, run in ((dw.METHOD_SHB, dw.deconvolve_shb_hip), (dw.METHOD_RL, dw.deconvolve_rl_hip)):
        got = {}
        s = dw.DwOpts(nIter=3, iter_type=dw.ITER_FIXED, borderQuality=0, fulldump=1, method=method,
                      iter_hook=lambda i, e, x: got.__setitem__(i, x))
        out = []
        assert updates(lambda: out.append(run(im, k, s))) == 0
        np.testing.assert_array_equal(got[-1], out[0])
        assert np.unravel_index(np.argmax(got[-2]), got[-2].shape) == (0, 0, 0)
        o32, _, _, _ = (po.rl if method == dw.METHOD_RL else po.shb)(im, k, niter=3, border_quality=0)
        assert rel_l2(out[0], o32) <= 1e-5


CHILD = """
import sys
import numpy as np, torch
sys.path[:0] = [%r, %r]
import deconwolf_amd as dw
from test_gpu_anysize_path import job_bytes, updates
from test_gpu_extended import _image, _psf, rel_l2
shape = (127, 251, 251)
im = torch.from_numpy(_image(shape)).cuda()
k = torch.from_numpy(_psf(shape, (63, 125, 125))).cuda()
s = lambda: dw.DwOpts(nIter=2, iter_type=dw.ITER_FIXED, borderQuality=0)
need = job_bytes(shape, shape, 0, 2)
out = [torch.empty_like(im), torch.empty_like(im)]
held = []
for piece in (8 << 30, 1 << 30, 64 << 20):
    while torch.cuda.mem_get_info()[0] > need + (128 << 20) + piece:
        held.append(torch.empty(piece, dtype=torch.uint8, device="cuda"))
print("free MiB", torch.cuda.mem_get_info()[0] >> 20, "any-size MiB", need >> 20, flush=True)
n = updates(lambda: dw.deconvolve_shb_hip_device(im, k, s(), out=out[0]))
held.clear()
torch.cuda.empty_cache()
m = updates(lambda: dw.deconvolve_shb_hip_device(im, k, s(), out=out[1]))
print("updates", n, m, "rel", rel_l2(out[0].cpu(), out[1].cpu()), flush=True)
assert n == 0 and m > 0 and rel_l2(out[0].cpu(), out[1].cpu()) <= 1e-5
"""


def test_device_without_room_for_the_extension():
    """With device memory for the any-size layout alone a per-image job runs on
    it (in a process of its own: the library keeps the largest block it had)."""
    print("any-size: device without room", flush=True)
    r = subprocess.run([sys.executable, "-c", CHILD % (ROOT, os.path.join(ROOT, "tests"))], cwd=ROOT,
                       capture_output=True, text=True, timeout=100)
    print(r.stdout, r.stderr[-2000:], flush=True)
    assert r.returncode == 0
