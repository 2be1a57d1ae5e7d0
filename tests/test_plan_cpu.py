"""Host-side plans without a GPU: what dwhip_job_plan lays out, read through a
small program compiled against the library's internal header."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "deconwolf_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc" if os.path.exists("/opt/rocm/bin/hipcc") else shutil.which("hipcc")


@pytest.fixture(scope="session")
def probe(tmp_path_factory):
    """run(body, rows): a C++ program that reads rows of integers into v[] and
    runs `body` for each; its output lines as lists of integers."""
    if not HIPCC:
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("plan")

    def run(body, rows):
        n = len(rows[0])
        src = d / ("p%d.cpp" % (abs(hash(body)) % 10 ** 9))
        exe = str(src)[:-4]
        src.write_text("""
#include <hip/hip_runtime.h>
#include <stdio.h>
#include "dwhip.h"
#include "dwhip_internal.h"
int main() {
    dwhip_plan_cache_path("");
    long long v[%d];
    for (;;) {
        for (int i = 0; i < %d; ++i) if (scanf("%%lld", &v[i]) != 1) return 0;
        %s
    }
}""" % (n, n, body))
        lib = os.path.join(ROOT, "deconwolf_amd", "libdwhip.so")
        subprocess.run([HIPCC, "--cuda-host-only", "-O0", "-w", "-x", "hip", "-I" + os.path.join(ROOT, "include"),
                        "-I" + CSRC, str(src), "-x", "none", lib, "-Wl,-rpath," + os.path.dirname(lib), "-o", exe],
                       check=True)
        out = subprocess.run([exe], input="\n".join(" ".join(map(str, r)) for r in rows), text=True,
                             capture_output=True, check=True).stdout
        return [[int(x) for x in line.split()] for line in out.splitlines()]
    return run


# smallest, odd-rowed, ordinary and large transform sizes of the fused passes
FAST = [(2, 1, 1), (4, 3, 5), (64, 45, 21), (256, 256, 96), (810, 640, 90), (1250, 1215, 140), (4096, 27, 8)]


def test_trial_image_lies_outside_the_job(probe):
    """The planner's trial runs the ratio pass, which reads the job's image and
    overwrites its spectrum: the image has memory of its own, behind the block
    of every candidate (the layout of the smallest tiles is the largest)."""
    body = """
        int64_t w[3] = {v[0], v[1], v[2]};
        size_t job = 0, image = 0;
        const int64_t whole[3] = {v[0], v[1], v[2]};
        dwhip_plan_trial_block(w, v[3] ? whole : nullptr, &job, &image);
        int64_t m[3] = {w[0] / 2, w[1] > 1 ? w[1] / 2 : 1, w[2] > 1 ? w[2] / 2 : 1};
        if (v[3]) m[0] = w[0], m[1] = w[1], m[2] = w[2];
        size_t most = 0;
        for (int x = 0; x <= 1; ++x) {
            DwhipPlanChoice c;
            if (x) c.xrows = c.ycols = c.zcols = 1;
            DwhipJob j;
            j.force_plan = &c;
            dwhip_params p;
            dwhip_params_default(&p, 2);
            for (int d = 0; d < 3; ++d) p.work[d] = w[d];
            const float* im = (const float*)(uintptr_t)256;
            if (dwhip_job_plan(&j, im, m[0], m[1], m[2], im, 1, 1, 1, &p, nullptr) != DWHIP_OK) return 1;
            if (j.bytes > most) most = j.bytes;
        }
        printf("%zu %zu %zu %lld\\n", job, image, most, (long long)(m[0] * m[1] * m[2] * 4));
    """
    # half the transform, or the job's image (here as large as the transform)
    for job, image, most, need in probe(body, [w + (whole,) for w in FAST for whole in (0, 1)]):
        assert job % 256 == 0 and most <= job
        assert image >= need


# image and PSF: either larger, both small, a PSF longer than the period (bq 1)
STATS = [(1, 1, 1, 1, 1, 1, 2), (40, 36, 1, 181, 181, 79, 2), (8, 8, 8, 63, 63, 63, 1), (64, 64, 8, 181, 181, 31, 1),
         (1024, 1024, 60, 181, 181, 79, 2), (37, 23, 11, 9, 9, 7, 0), (5, 8, 2503, 3, 3, 5, 0)]


def test_statistics_cover_the_psf_and_fit_the_spectrum(probe):
    """The set-up statistics' grid follows the larger of image and PSF (both are
    walked), and its partials, which lie in C, fit there."""
    body = """
        DwhipJob j;
        dwhip_params p;
        dwhip_params_default(&p, 2);
        p.border_quality = v[6];
        const float* im = (const float*)(uintptr_t)256;
        if (dwhip_job_plan(&j, im, v[0], v[1], v[2], im, v[3], v[4], v[5], &p, nullptr) != DWHIP_OK) return 1;
        printf("%d %zu\\n", dwhip_stat_blocks(&j.d), j.lay.K - j.lay.C);
    """
    for (M, N, P, pM, pN, pP, _), (blocks, room) in zip(STATS, probe(body, STATS)):
        assert 1 <= blocks <= 1024 and 32 * blocks <= room
        n = max(M * N * P, pM * pN * pP)
        assert blocks in (1024, room // 32, max(1, n // 2048))


# image, PSF, bq 0: sizes timed on both paths (us per iteration, extended and
# any-size) and the one that runs them; near ties in between are left out
PATHS = [
    ((61, 61, 31), (61, 61, 31), "ext"),             # 128, 170
    ((251, 249, 131), (31, 31, 131), "ext"),         # 427, 1697
    ((375, 375, 75), (375, 375, 75), "ext"),         # 546, 663
    ((1021, 1021, 31), (1021, 1021, 31), "ext"),     # 2941, 4767
    ((25, 25, 250), (9, 9, 5), "ext"),               # 83, 102
    ((61, 61, 1008), (9, 9, 5), "ext"),              # 334, 468
    ((125, 125, 1500), (125, 125, 5), "any"),        # 3200, 1299
    ((125, 125, 640), (125, 125, 5), "any"),         # 938, 601
    ((63, 61, 701), (63, 61, 701), "any"),           # 1027, 419
    ((63, 61, 1009), (31, 31, 1009), "any"),         # 913, 569
    ((25, 25, 1800), (9, 9, 5), "any"),              # 235, 204
    # no choice: a depth no padded plan covers
    ((5, 5, 2503), (3, 3, 5), "any"),
]


def test_extended_or_any_size_by_time(probe):
    body = """
        DwhipJob j;
        dwhip_params p;
        dwhip_params_default(&p, 2);
        p.border_quality = 0;
        const float* im = (const float*)(uintptr_t)256;
        if (dwhip_job_plan(&j, im, v[0], v[1], v[2], im, v[3], v[4], v[5], &p, nullptr) != DWHIP_OK) return 1;
        printf("%d %d\\n", j.ext, j.generic);
    """
    got = probe(body, [a + b for a, b, _ in PATHS])
    for (shape, psf, want), (ext, gen) in zip(PATHS, got):
        assert (ext, gen) == ((1, 0) if want == "ext" else (0, 1)), (shape, psf)


def test_any_size_plan_of_one_column(probe):
    """A job one voxel wide has a plan on the any-size path too."""
    body = """
        DwhipJob j;
        j.allow_ext = false;
        dwhip_params p;
        dwhip_params_default(&p, 2);
        p.border_quality = 0;
        const float* im = (const float*)(uintptr_t)256;
        if (dwhip_job_plan(&j, im, v[0], v[1], v[2], im, 1, 1, 1, &p, nullptr) != DWHIP_OK) return 1;
        printf("%d\\n", j.generic);
    """
    assert probe(body, [(1, 1021, 31), (1, 1, 2503)]) == [[1], [1]]


# work sizes: image, x rows per tile, values of the pad (forward, inverse plan)
PADS = [
    ((672, 784, 18), 19, 0, 0),      # 743 tiles without the pad, 830 with it
    ((672, 672, 80), 17, 42, 0),     # several turns either way
    ((672, 784, 17), 19, 0, 0),      # 702 and 784
    ((672, 784, 16), 17, 42, 0),     # one turn either way
    ((256, 256, 96), 46, 8, 16),     # 16 * 8
    ((1250, 1215, 140), 10, 0, 0),   # 25 * 25: odd
]


def test_x_pad_keeps_tiles_at_once(probe):
    """The padded exchange of the x rows is given up where its rows would take
    the tiles from one turn (three workgroups per CU) to two; plan and tiles agree."""
    body = """
        DwhipJob j;
        dwhip_params p;
        dwhip_params_default(&p, 2);
        for (int d = 0; d < 3; ++d) p.work[d] = v[d];
        const float* im = (const float*)(uintptr_t)256;
        if (dwhip_job_plan(&j, im, v[0] / 2, v[1] / 2, v[2] / 2, im, 1, 1, 1, &p, nullptr) != DWHIP_OK) return 1;
        printf("%d %d %d %zu\\n", j.tiles.xrows, j.d.pxf.pad, j.d.pxi.pad, j.tiles.lds[KIND_X]);
    """
    for (w, rows, fwd, inv), got in zip(PADS, probe(body, [w for w, *_ in PADS])):
        assert got[:3] == [rows, fwd, inv], w
        h = w[0] // 2
        assert got[3] >= rows * 8 * max(h + 1, h + fwd, h + inv)


# image, PSF, bq, iterations: plain, extended and any-size jobs
BYTES = [(1024, 1024, 60, 181, 181, 79, 2, 50), (128, 128, 32, 127, 127, 63, 2, 1), (701, 512, 211, 31, 9, 1, 2, 10),
         (40, 36, 16, 9, 9, 7, 2, 250), (1, 1, 1, 1, 1, 1, 2, 1), (2048, 2048, 1, 63, 63, 1, 2, 5),
         (64, 64, 60, 9, 9, 7, 0, 5), (257, 211, 151, 111, 111, 111, 0, 2), (1024, 1024, 60, 181, 181, 79, 1, 10),
         (37, 23, 11, 37, 23, 11, 0, 4), (1, 1021, 31, 1, 1, 5, 0, 1), (5, 8, 2503, 3, 3, 5, 0, 3),
         (2011, 11, 7, 101, 11, 7, 1, 100), (125, 125, 1500, 125, 125, 5, 0, 3)]


def test_job_bytes_is_what_a_job_needs(probe):
    """dwhip_job_bytes covers what a job lays out and asks for little more; a job
    that also has a larger, extended layout runs in it (the static block, an
    engine's budget and a failed allocation plan it without the extension)."""
    body = """
        dwhip_params p;
        dwhip_params_default(&p, (int)v[7]);
        p.border_quality = v[6];
        int64_t w[3], r[3];
        if (dwhip_work_size(v[0], v[1], v[2], v[3], v[4], v[5], v[6], w, r) != DWHIP_OK) return 1;
        size_t most = 0, ext = 0;
        for (int k = 0; k < 4; ++k) {
            p.method = k & 1 ? DWHIP_METHOD_RL : DWHIP_METHOD_SHB;
            DwhipJob j;
            j.allow_ext = k >= 2;
            const float* im = (const float*)(uintptr_t)256;
            if (dwhip_job_plan(&j, im, v[0], v[1], v[2], im, v[3], v[4], v[5], &p, nullptr) != DWHIP_OK) return 1;
            size_t& n = j.ext ? ext : most;
            if (j.bytes > n) n = j.bytes;
        }
        printf("%zu %zu %zu\\n", dwhip_job_bytes(w, v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7]), most, ext);
    """
    for job, (est, need, ext) in zip(BYTES, probe(body, BYTES)):
        assert need <= est <= need + 24 * 1024, job
        assert not ext or ext > need, job
    # runs in the static block by its any-size layout
    est, _, ext = probe(body, [(257, 211, 151, 111, 111, 111, 0, 2)])[0]
    assert est <= 256 << 20 < ext


def test_paths_of_the_gpu_tests(probe):
    """The sizes that test_gpu_anysize and test_gpu_extended compare with the
    oracle run extended, those of test_gpu_paths on both paths (the any-size path's
    own tests take the extension's room away)."""
    pytest.importorskip("torch")
    import test_gpu_anysize
    import test_gpu_extended
    import test_gpu_paths
    body = """
        DwhipJob j;
        dwhip_params p;
        dwhip_params_default(&p, 2);
        p.border_quality = v[6];
        const float* im = (const float*)(uintptr_t)256;
        if (dwhip_job_plan(&j, im, v[2], v[1], v[0], im, v[5], v[4], v[3], &p, nullptr) != DWHIP_OK) return 1;
        printf("%d\\n", j.ext);
    """
    cases = [c[0] + c[1] + (c[2],) for c in test_gpu_anysize.CASES]
    cases += [c[0] + c[1] + (c[3],) for c in test_gpu_extended.CASES]
    assert probe(body, cases) == [[1]] * len(cases)
    cases = [c[0] + c[1] + (c[3],) for c in test_gpu_paths.CASES]
    assert probe(body, cases) == [[1], [0], [0], [0], [0], [1]]
