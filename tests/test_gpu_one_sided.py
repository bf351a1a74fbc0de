"""Directions that are periodic on one face only.  The time step after a step depends on the face
field behind the last cell of a direction: where its upper face is periodic, the next ghost fill
puts the first cell's new field there.  Its EMFs come from the lower ghost cells, which are the
image of the upper end only if the lower face is periodic too.  Each grid has a strong field
component at the face in question, so that the last cells decide dt; strict build, every kernel
form, bit-identical to the oracle (states, t and dt)."""
import numpy as np
import pytest

from ppkmhd_amd import _abi as A
from ppkmhd_amd import make_params

pytestmark = pytest.mark.gpu

P, N, D = A.BC_PERIODIC, A.BC_NEUMANN, A.BC_DIRICHLET


def layered(p, d):
    """A rough state whose field component d (face-centred along d) is strong in the first and
    the last cell of direction d.  Not divergence-free, which strict equality does not need."""
    rng = np.random.default_rng(7)
    U = np.empty((8, p.ksize, p.jsize, p.isize))
    r = rng.uniform(-1.0, 1.0, U.shape)
    U[A.ID] = 1.0 + 0.2 * r[A.ID]
    for v in (A.IU, A.IV, A.IW):
        U[v] = U[A.ID] * 0.3 * r[v]
    for v in (A.IA, A.IB, A.IC):
        U[v] = 0.2 * r[v]
    n, axis = (p.nx, p.ny, p.nz)[d], 2 - d
    for c in (0, n - 1):
        at = [slice(None)] * 3
        at[axis] = p.ghost_width + c
        U[A.IA + d][tuple(at)] += 3.0
    U[A.IP] = 2.0 / (p.gamma0 - 1.0) + 0.5 * (U[A.IU:A.IA] ** 2).sum(0) / U[A.ID]
    U[A.IP] += 0.5 * np.maximum(U[A.IA:] ** 2, np.roll(U[A.IA:], -1, 3 - d) ** 2).sum(0)
    return U


CASES = [((70, 37), [N, P, P, P, P, P], 0), ((70, 37), [D, P, N, N, P, P], 0),
         ((37, 70), [P, P, N, P, P, P], 1), ((37, 70), [N, P, D, P, P, P], 1),
         ((70, 37), [P, N, P, D, P, P], 0),
         ((21, 17, 9), [N, P, P, P, P, P], 0), ((21, 17, 9), [P, P, D, P, N, N], 1),
         ((21, 17, 9), [P, P, N, D, N, P], 2), ((21, 17, 9), [D, P, N, P, D, P], 2)]


@pytest.mark.parametrize("path", [A.PATH_FUSED, A.PATH_FUSED_RECORDS, A.PATH_STAGED])
@pytest.mark.parametrize("dims,bc,d", CASES)
def test_strict_equals_oracle(oracle, gpu, dims, bc, d, path):
    from ppkmhd_amd.solver import SolverMHDMuscl
    p = make_params(len(dims), *dims, gamma0=5 / 3, cfl=0.4, tEnd=10.0, bc=bc, kernel_path=path,
                    precision=A.FP64_STRICT)
    U = layered(p, d)
    o = oracle.Solver(p)
    o.set_state(U)
    with SolverMHDMuscl(p) as g:
        g.upload(U)
        for k in range(6):
            o.step(0.0, A.DT_CFL)
            g.step(0.0, A.DT_CFL)
            assert g.time() == o.time(), f"step {k}"
        assert np.isfinite(o.get_state()).all() and np.array_equal(g.download(), o.get_state())
