"""The grids of test_gpu_march2d.py take the strip shapes that they are there for (march2d_shape,
kernels.hpp, at 256 CUs): strips of 64 and of 32 columns, one and several rows, a ragged last
strip, two strips of a wave on different rows, and a wave whose second strip does not exist."""
import os
import subprocess

import pytest

from test_gpu_march2d import LONG, SMALL

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def shapes(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("shape") / "march_shape")
    r = subprocess.run(["/opt/rocm/bin/hipcc", "--offload-host-only", "-std=c++17", "-O1",
                        "-DPPK_NS=strict", "-I", os.path.join(ROOT, "include"),
                        "-I", os.path.join(ROOT, "ppkmhd_amd", "csrc"),
                        os.path.join(ROOT, "tests", "cxx", "march_shape.cpp"), "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    grids = SMALL + LONG
    out = subprocess.run([exe, *(str(n) for g in grids for n in g)], capture_output=True, text=True)
    return {g: tuple(map(int, line.split())) for g, line in zip(grids, out.stdout.splitlines())}


def test_small_grids_have_one_row_per_strip(shapes):
    assert all(shapes[g][:2] == (64, 1) for g in SMALL)


def test_long_grids_cover_the_strip_shapes(shapes):
    several = [(g, shapes[g]) for g in LONG if shapes[g][1] > 1]
    for lw in (32, 64):
        mine = [(g, s) for g, s in several if s[0] == lw]
        assert any(g[1] % s[1] for g, s in mine), f"no ragged last strip of {lw} columns"
        assert any(s[2] > 1 for g, s in mine), f"no row of several strips of {lw} columns"
    halves = [s for _, s in several if s[0] == 32]
    assert any(s[2] % 2 for s in halves), "no wave with strips of different rows"
    assert any(s[2] * s[3] % 2 for s in halves), "no wave with a strip that does not exist"
    assert any(shapes[g][:2] == (32, 1) for g in LONG)
