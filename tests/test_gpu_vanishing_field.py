"""One step of the default build where field components vanish beside ordinary ones: 0, and values
from 1e-100 to 1e-320, whose squares are subnormal or 0.  The result is finite and equal to the
oracle's within the default build's bar for a step at fixed dt (a relative L-inf of 1e-12)."""
import numpy as np
import pytest

from parity import rel_linf
from ppkmhd_amd import _abi as A
from ppkmhd_amd import make_params

pytestmark = pytest.mark.gpu


def state(p, moving):
    rng = np.random.default_rng(11)
    shape = (p.ksize, p.jsize, p.isize)
    U = np.empty((8,) + shape)
    U[A.ID] = rng.uniform(0.5, 2.0, shape)
    for v in (A.IU, A.IV, A.IW):
        U[v] = U[A.ID] * rng.uniform(-0.5, 0.5, shape) * (moving if v == A.IU else moving > 0.5)
    for v in (A.IA, A.IB, A.IC):
        kind = rng.uniform(0.0, 1.0, shape)
        U[v] = 10.0 ** -rng.uniform(100.0, 320.0, shape) * np.sign(rng.uniform(-1.0, 1.0, shape))
        U[v] = np.where(kind < 0.2, 0.0, np.where(kind < 0.3, rng.uniform(0.1, 0.5, shape), U[v]))
    U[A.IP] = rng.uniform(1.0, 2.0, shape) + 0.5 * (U[A.IU:A.IA] ** 2).sum(0) / U[A.ID] + 0.4
    return U


@pytest.mark.parametrize("path", [A.PATH_FUSED, A.PATH_FUSED_RECORDS, A.PATH_STAGED])
@pytest.mark.parametrize("dims", [(75, 41), (33, 14, 10)])
@pytest.mark.parametrize("moving", [0.0, 0.5, 1.0])
def test_default_build_equals_oracle(oracle, gpu, dims, path, moving):
    from ppkmhd_amd.solver import SolverMHDMuscl
    p = make_params(len(dims), *dims, gamma0=5 / 3, cfl=0.8, tEnd=10.0, kernel_path=path)
    U = state(p, moving)
    o = oracle.Solver(p)
    o.set_state(U)
    with SolverMHDMuscl(p) as g:
        g.upload(U)
        o.step(1e-3, A.DT_FIXED)
        g.step(1e-3, A.DT_FIXED)
        got, ref = g.download(), o.get_state()
        assert np.isfinite(ref).all() and np.isfinite(got).all()
        assert rel_linf(got, ref, p) < 1e-12
