"""The single-pass 2D step where its strips end: widths around multiples of the 60 and 28 output
columns of a strip, on grids whose strips are 64 columns of one row (SMALL) and on grids with strips
of 32 columns, of several rows, with a ragged last strip (LONG; test_march2d_shape_cpu.py holds the
shapes), with every boundary type and solver.  The strict build is bit-identical to the oracle
(ghosts, t and dt included) and, where strips hold many rows, to the three-kernel form."""
import numpy as np
import pytest

from ppkmhd_amd import _abi as A
from ppkmhd_amd import default_problem, make_params

pytestmark = pytest.mark.gpu

P, N, D = A.BC_PERIODIC, A.BC_NEUMANN, A.BC_DIRICHLET


def case(nx, ny, bc, **kw):
    p = make_params(2, nx, ny, gamma0=5 / 3, cfl=0.8, tEnd=10.0, bc=bc,
                    precision=A.FP64_STRICT, **kw)
    return p, default_problem(A.PROBLEM_ORSZAG_TANG, p)


SMALL = [(3, 3), (28, 5), (29, 7), (57, 4), (60, 3), (61, 16), (120, 9), (121, 33), (5, 131)]
LONG = [(3, 1273), (67, 1272), (3, 5003), (61, 2001), (61, 2503), (85, 1272), (29, 2503),
        (121, 1272), (29, 5003)]


def solver(p, pr, path):
    from ppkmhd_amd.solver import SolverMHDMuscl
    q = A.Params.from_buffer_copy(p)
    q.kernel_path = path
    return SolverMHDMuscl(q, pr)


@pytest.mark.parametrize("nx,ny", SMALL + LONG)
@pytest.mark.parametrize("bc,kw", [
    (P, {}),
    ([P, P, N, N, P, P], dict(slope_type=2.0, riemann=A.RIEMANN_HLL)),
    ([N, N, D, N, P, P], dict(riemann=A.RIEMANN_LLF)),
    ([D, N, N, D, P, P], dict(slope_type=2.0)),
])
def test_strict_equals_oracle(oracle, gpu, nx, ny, bc, kw):
    p, pr = case(nx, ny, bc, **kw)
    o = oracle.Solver(p)
    o.init_problem(pr)
    with solver(p, pr, A.PATH_FUSED) as g:
        for _ in range(4):
            o.step(0.0, A.DT_CFL)
            g.step(0.0, A.DT_CFL)
        assert np.array_equal(g.download(), o.get_state())
        assert g.time() == o.time()


@pytest.mark.parametrize("nx,ny", [(640, 480), (1021, 517), (1500, 1301)])
def test_strict_equals_three_kernel_form(gpu, nx, ny):
    p, pr = case(nx, ny, [P, P, N, N, P, P], slope_type=2.0)
    with solver(p, pr, A.PATH_FUSED) as a, solver(p, pr, A.PATH_FUSED_RECORDS) as b:
        for s in (a, b):
            s.run(3)
            s.step(1e-5, A.DT_FIXED)
            s.run(2)
        assert np.array_equal(a.download(), b.download())
        assert a.time() == b.time()


@pytest.mark.parametrize("nx,ny", [(64, 64), (16, 4096), (5, 20000), (400, 400)])
def test_auto_gives_the_bits_of_either_form(gpu, nx, ny):
    """AUTO takes the faster form by size (march2d_pays): here both forms occur."""
    p, pr = case(nx, ny, [N, N, P, P, P, P])
    out = []
    for path in (A.PATH_AUTO, A.PATH_FUSED, A.PATH_FUSED_RECORDS):
        with solver(p, pr, path) as s:
            s.run(4)
            out.append((s.time(), s.download()))
    for t, U in out[1:]:
        assert t == out[0][0] and np.array_equal(U, out[0][1])
