"""The default build's solver forms against the reference's expressions (both from mhd_device.hpp,
built for the host) where a field component vanishes: 0, or so small that its square is subnormal
or 0, as ahead of a front in a component that starts at 0; and where wave speeds coincide because
the sound speed is lost in the velocity, so that a denominator of one side or direction is 0."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "tests", "cxx", "edge_emf.cpp")


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    d = tmp_path_factory.mktemp("edge")
    out = {}
    for name, flags in (("lean", []), ("ref", ["-DPPK_KEEP_ROUNDING"])):
        exe = str(d / name)
        cmd = ["/opt/rocm/bin/hipcc", "--offload-host-only", "-std=c++17", "-O1", *flags,
               "-ffp-contract=off", "-I", os.path.join(ROOT, "include"),
               "-I", os.path.join(ROOT, "ppkmhd_amd", "csrc"), SRC, "-o", exe]
        r = subprocess.run(cmd, capture_output=True, text=True)
        assert r.returncode == 0, r.stderr[-4000:]
        out[name] = exe

    def both(*args):
        res = []
        for name in ("lean", "ref"):
            r = subprocess.run([out[name], *map(str, args)], capture_output=True, text=True)
            assert r.returncode == 0, r.stderr[-4000:]
            res.append(np.array([l.split() for l in r.stdout.splitlines()], dtype=np.float64))
        return res
    return both


def test_vanishing_fields(run):
    lean, ref = run("vanishing", 20000)
    assert np.isfinite(ref).all() and np.isfinite(lean).all()
    # EMFs are u B of values up to 1; the forms differ by roundings of some tens of operations
    for col, eps in ((0, 2.0 ** -53), (1, 2.0 ** -24)):
        assert np.abs(lean[:, col] - ref[:, col]).max() < 200 * eps


@pytest.mark.parametrize("mode", ["cold", "stream"])
def test_coinciding_waves(run, mode):
    """A side or direction whose denominator is 0 leaves the others as they are: what is finite with
    the reference's expressions is finite, and equal to the roundings of some tens of operations."""
    lean, ref = run(mode, 2000)
    ok = np.isfinite(ref)
    assert ok.any() and np.isfinite(lean[ok]).all()
    scale = np.abs(np.where(ok, ref, 0.0)).max(0)
    assert (np.abs(lean - ref)[ok] <= (200 * 2.0 ** -53 * scale * np.ones_like(ref))[ok]).all()
