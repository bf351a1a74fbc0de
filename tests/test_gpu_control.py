"""Time-loop control: t, dt and the iteration as the host reads them (a pinned copy that the
step's last kernel writes) equal the oracle's through every call that changes them, on every
kernel form; and a step whose CFL partials are too many for the prologue's one block."""
import numpy as np
import pytest

from ppkmhd_amd import _abi as A
from ppkmhd_amd import default_problem, make_params
from ppkmhd_amd.params import make_hydro_params

pytestmark = pytest.mark.gpu


def pair(kind, path, tEnd):
    kw = dict(gamma0=5 / 3, cfl=0.8, tEnd=tEnd, precision=A.FP64_STRICT, kernel_path=path,
              float_round=False)
    if kind == "hydro":
        if path == A.PATH_FUSED_RECORDS:
            kw["kernel_path"] = A.PATH_FUSED  # the Euler solvers have no form with records
        from oracle import pyhydro as O
        from ppkmhd_amd.solver import SolverHydroMuscl as S
        p = make_hydro_params(2, 40, 24, riemann=A.RIEMANN_HLLC, bc=A.BC_DIRICHLET, **kw)
        pr = default_problem(A.PROBLEM_IMPLODE, p)
    else:
        from oracle import pyoracle as O
        from ppkmhd_amd.solver import SolverMHDMuscl as S
        dims = (40, 24) if kind == "mhd2" else (12, 10, 9)
        p = make_params(len(dims), *dims, **kw)
        pr = default_problem(A.PROBLEM_ORSZAG_TANG if kind == "mhd2" else A.PROBLEM_BLAST, p)
    o = O.Solver(p)
    o.init_problem(pr)
    return o, S(p, pr)


@pytest.mark.parametrize("kind", ["mhd2", "mhd3", "hydro"])
@pytest.mark.parametrize("path", [A.PATH_AUTO, A.PATH_FUSED, A.PATH_FUSED_RECORDS,
                                  A.PATH_STAGED])
def test_time_follows_every_call(oracle, gpu, kind, path):
    o, g = pair(kind, path, 1.0)
    with g:
        for k in range(2):
            o.step(0.0, A.DT_CFL)
            g.step(0.0, A.DT_CFL)
            assert g.time() == o.time()
        dt = g.compute_dt_local()
        t, _, it = g.time()
        assert (t, it) == (o.time()[0], o.time()[2])
        o.step(0.0, A.DT_CFL)
        g.step(0.0, A.DT_CFL)
        assert g.time() == o.time() and g.time()[1] == dt
        for mode, value in ((A.DT_FIXED, 1e-4), (A.DT_CFL, 0.0)):
            o.step(value, mode)
            g.step(value, mode)
            assert g.time() == o.time()
        o.set_time(0.25, 7)
        g.set_time(0.25, 7)
        assert g.time()[0] == 0.25 and g.m_iteration == 7
        o.step(0.0, A.DT_CFL)
        g.run(1)
        assert g.time() == o.time()
        g.set_time(1.0 - 1e-3, 9)
        assert not g.finished()
        g.run(50)  # reaches tEnd; the steps after it do nothing
        t, _, it = g.time()
        assert t == 1.0 and 9 < it < 59 and g.finished()
        U = g.download()
        g.run(3)
        assert g.time()[2] == it and np.array_equal(g.download(), U)


def test_more_partials_than_the_prologue_reduces(gpu):
    """128^3 in the three-kernel form leaves 9398 CFL partials; the single-pass form leaves one
    per block: the same dt, strict bit for bit."""
    from ppkmhd_amd.solver import SolverMHDMuscl
    p = make_params(3, 128, 128, 128, gamma0=5 / 3, cfl=0.8, tEnd=1.0, precision=A.FP64_STRICT)
    pr = default_problem(A.PROBLEM_BLAST, p)
    out = []
    for path in (A.PATH_FUSED, A.PATH_FUSED_RECORDS):
        p.kernel_path = path
        with SolverMHDMuscl(p, pr) as s:
            s.run(4)
            out.append((s.time(), s.download()))
    assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])
