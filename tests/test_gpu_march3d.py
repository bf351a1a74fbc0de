"""The single-pass 3D step on boxes of few tile-planes, where every block marches one or two
planes and ranges cut tiles (strict build, bit-identical to the oracle), and the choice between
it and the three-kernel form: PPK_PATH_AUTO gives the same bits as either."""
import numpy as np
import pytest

from ppkmhd_amd import _abi as A
from ppkmhd_amd import default_problem, make_params

pytestmark = pytest.mark.gpu

P, N, D = A.BC_PERIODIC, A.BC_NEUMANN, A.BC_DIRICHLET


def case(dims, path, bc=P, **kw):
    p = make_params(3, *dims, gamma0=5 / 3, cfl=0.8, tEnd=10.0, bc=bc, kernel_path=path,
                    precision=A.FP64_STRICT, **kw)
    pr = default_problem(A.PROBLEM_BLAST, p)
    pr.blast_radius = 0.25
    return p, pr


@pytest.mark.parametrize("dims", [(3, 3, 3), (16, 12, 5), (17, 13, 4), (37, 29, 11), (5, 40, 31)])
@pytest.mark.parametrize("bc,kw", [(P, {}), ([P, P, N, N, N, D],
                                             dict(slope_type=2.0, riemann=A.RIEMANN_HLL))])
def test_strict_equals_oracle_on_small_boxes(oracle, gpu, dims, bc, kw):
    from ppkmhd_amd.solver import SolverMHDMuscl
    p, pr = case(dims, A.PATH_FUSED, bc, **kw)
    o = oracle.Solver(p)
    o.init_problem(pr)
    with SolverMHDMuscl(p, pr) as g:
        for _ in range(3):
            o.step(0.0, A.DT_CFL)
            g.step(0.0, A.DT_CFL)
        assert np.array_equal(g.download(), o.get_state())
        assert g.time() == o.time()


@pytest.mark.parametrize("dims", [(20, 20, 20), (48, 48, 48), (64, 64, 64), (75, 70, 81)])
def test_either_form_gives_the_same_bits(gpu, dims):
    from ppkmhd_amd.solver import SolverMHDMuscl
    out = []
    for path in (A.PATH_AUTO, A.PATH_FUSED, A.PATH_FUSED_RECORDS):
        with SolverMHDMuscl(*case(dims, path)) as s:
            s.run(3)
            out.append((s.time(), s.download()))
    for t, U in out[1:]:
        assert t == out[0][0] and np.array_equal(U, out[0][1])
