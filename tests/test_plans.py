"""The kernels' plans and grids (plain C++ headers under bus-fill_amd/csrc)
checked on the CPU: tests/plan_check.cpp compiled with g++."""
import os
import shutil
import subprocess

import pytest

import busfill as bf

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def planner(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path_factory.mktemp("plans") / "plan_check")
    subprocess.run([gxx, "-O2", "-std=c++17", "-Wall", "-Wextra", "-Werror",
                    "-I", os.path.join(ROOT, "bus-fill_amd", "csrc"),
                    os.path.join(ROOT, "tests", "plan_check.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("part", ["dequant", "block_grid", "block_choice", "tile_grid", "tile_choice"])
def test_plans(planner, part):
    r = subprocess.run([planner, part], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


def plan(planner, kind, *shape):
    r = subprocess.run([planner, kind, *map(str, shape)], capture_output=True, text=True, check=True, timeout=60)
    return tuple(map(int, r.stdout.split()))


def test_tile_shapes_reach_every_form(planner):
    """The GPU tests' shapes run the form each stands for, and together every tile
    shape uncut and cut, with and without whole rounds before the cut ones."""
    from test_gpu_tile import FORMS
    for shape, (ta, nb, rounds, s) in FORMS.items():
        TA, NB, F, R, S, slices = plan(planner, "tile", *shape)
        assert (TA, NB, F // 256, S, slices) == (ta, nb, rounds, s, 0) and R, shape
    forms = {(ta, nb, rounds > 0, s > 1) for ta, nb, rounds, s in FORMS.values()}
    for tile in ((2, 1), (3, 1), (4, 1), (4, 2)):
        assert {f[3] for f in forms if f[:2] == tile} == {True, False}, tile
    assert {(3, 1, True, True), (4, 1, True, True), (4, 2, True, True), (3, 1, False, True), (4, 1, False, True)} <= forms


def test_block_shapes_reach_every_form(planner):
    from test_gpu_block import FORMS
    for shape, form in FORMS.items():
        assert plan(planner, "block", *shape) == form, shape
    every = {(mt, nt, 8) for mt in (1, 2, 3, 4) for nt in (1, 2)} | {(mt, 0, nw) for mt in (3, 4) for nw in (4, 8)}
    assert set(FORMS.values()) == every


def test_fp32_rows_inside_the_gemm():
    """ggml hook: up to eight fp32 rows go to the LDS kernel itself (no
    workspace) wherever its plan keeps all of A; nine rows, and plans with an
    activation ring, are staged."""
    fmts = {"q4_0": (bf.GGML_Q4_0, 32, 18), "q4_k": (bf.GGML_Q4_K, 256, 144)}
    most = {(3000, 8192, "q4_0"): 7, (300, 8192, "q4_k"): 7, (3000, 8192, "q4_k"): 6}
    for fmt, (gt, blk, bb) in fmts.items():
        for N, K in ((1, 1024), (77, 2048), (5120, 5120), (17408, 1024), (17408, 5120), (27648, 5120), (300, 8192),
                     (3000, 8192)):
            for M in range(1, 10):
                views = (bf.ggml_tensor(gt, 1 << 20, (K, N), (bb, K // blk * bb)),
                         bf.ggml_tensor(bf.GGML_F32, 1 << 24, (K, M), (4, 4 * K)),
                         bf.ggml_tensor(bf.GGML_F32, 1 << 28, (N, M), (4, 4 * N)))
                inside = bf.ggml_mul_mat_workspace_bytes(*views) == 0
                assert inside == (M <= most.get((N, K, fmt), 8)), (fmt, N, K, M)
