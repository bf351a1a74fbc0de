"""Performance cases: what a program that uses this library has it do, through the public
Python entry points, over the range of sizes and options that are met in use.

    listed()           the fixed cases
    draw(rng)          one more case of the same ranges
    prepare(case, s)   inputs (from the seed alone) and the solver / batch / network handle
    run(state)         one pass: time steps (or training steps, ...) and the whole result
    work(case)         bytes and operations a pass cannot do without
    tolerance(case)    how far two correct implementations at this precision may differ
    exact(case, s)     the same result in plain torch in 64 bits, written from the scheme's
                       equations (MUSCL-Hancock, HLLD / HLL / LLF / HLLC / two-shock fluxes,
                       2D HLLD edge EMFs, constrained transport; MLP with Adam)

A time-stepping pass is one output interval of a program that keeps its state on the GPU: run
`steps` steps, take the device state (ghosts included) and the time.  The main-loop cases call
next_iteration() and finished() for every step, as the reference's driver does.
"""
import math

import numpy as np
import torch

from ppkmhd_amd import _abi as A
from ppkmhd_amd import surrogate as S
from ppkmhd_amd.params import make_hydro_params, make_params
from ppkmhd_amd.solver import BatchSolver, SolverHydroMuscl, SolverMHDMuscl

RIEMANN = {"approx": A.RIEMANN_APPROX, "llf": A.RIEMANN_LLF, "hll": A.RIEMANN_HLL,
           "hllc": A.RIEMANN_HLLC, "hlld": A.RIEMANN_HLLD}
PRECISION = {"fp64": A.FP64, "strict": A.FP64_STRICT, "fp32": A.FP32_BULK}
# boundary types of the faces x-, x+, y-, y+, z-, z+
BOUNDARY = {"periodic": [A.BC_PERIODIC] * 6, "walls": [A.BC_DIRICHLET] * 6,
            "open": [A.BC_NEUMANN] * 6,
            "mixed": [A.BC_PERIODIC] * 2 + [A.BC_DIRICHLET, A.BC_NEUMANN] +
                     [A.BC_NEUMANN, A.BC_DIRICHLET]}
BATCH_SIDES = (64, 128, 192, 256, 384, 512)  # the ensemble workload's side lengths


# ---- cases -----------------------------------------------------------------------------------
def _steps(name, kind, nx, ny, nz, steps, **kw):
    c = {"kind": kind, "problem": "ot", "nx": nx, "ny": ny, "nz": nz, "steps": steps,
         "riemann": "hlld", "slope": 1.0, "boundary": "periodic", "precision": "fp64",
         "gamma": 5.0 / 3.0}
    c.update(kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest grid in use, driven step by step: launches and synchronizations
        _steps("mhd2d_64_main_loop", "loop", 64, 64, 1, 10),
        # Orszag-Tang at the resolution it is usually shown at
        _steps("mhd2d_256", "mhd", 256, 256, 1, 50),
        # a ragged grid between walls and open faces, MC slopes
        _steps("mhd2d_1021x517_mixed_mc", "mhd", 1021, 517, 1, 20, problem="kh", slope=2.0,
               boundary="mixed", gamma=1.4),
        # a large 2D run
        _steps("mhd2d_2048", "mhd", 2048, 2048, 1, 10),
        # a small ragged 3D box, the size of a convergence study or a test
        _steps("mhd3d_37x29x45_mixed", "mhd", 37, 29, 45, 20, problem="kh",
               boundary="mixed"),
        # the 3D blast of the headline benchmark
        _steps("mhd3d_blast_256", "mhd", 256, 256, 256, 5, problem="blast"),
        # Kelvin-Helmholtz in the FP32-bulk form
        _steps("mhd3d_kh_fp32", "mhd", 160, 144, 128, 5, problem="kh", precision="fp32"),
        # Euler solvers: the implosion and the blast of the settings files at higher resolution
        _steps("hydro2d_implode", "hydro", 4096, 2048, 1, 20, problem="implode",
               riemann="hllc", boundary="walls", slope=2.0, gamma=1.666),
        _steps("hydro3d_blast", "hydro", 256, 192, 128, 10, problem="blast", riemann="hllc",
               boundary="walls", slope=2.0, gamma=1.666),
        # the ensemble: 64 Orszag-Tang runs of uneven sides, autotuned, downloaded at the end
        {"name": "ensemble2d_64", "kind": "batch", "dim": 2, "members": 64, "max_side": 512,
         "steps": 200, "riemann": "hlld", "slope": 1.0, "boundary": "periodic",
         "precision": "fp64", "autotune": True},
        # the learned face fluxes in the 2D step
        _steps("surrogate2d_1024", "surrogate", 1024, 1024, 1, 10),
        # training the network at the batch size of the surrogate workloads
        {"name": "mlp_train_4096", "kind": "train", "samples": 200000, "batch": 4096,
         "steps": 100},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mhd2", "mhd2", "mhd2", "mhd3", "mhd3", "mhd3", "loop", "hydro2",
                       "hydro2", "hydro3", "hydro3", "batch", "batch3", "surrogate", "train",
                       "gradient", "infer"])
    slope = rng.choice([1.0, 1.0, 2.0])
    boundary = rng.choice(["periodic", "periodic", "walls", "open", "mixed"])
    gamma = rng.choice([5.0 / 3.0, 1.4])
    precision = rng.choice(["fp64", "fp64", "fp64", "fp32", "strict"])
    riemann = rng.choice(["hlld", "hlld", "hlld", "hll", "llf"])
    # the MHD problems between walls: the shear layers along the periodic direction (walls
    # reverse the normal field, so the other problems would meet them as current sheets)
    problem2, problem3 = rng.choice(["ot", "kh", "blast"]), rng.choice(["kh", "blast"])
    if kind[:5] != "hydro" and boundary in ("walls", "mixed"):
        boundary, problem2, problem3 = "mixed", "kh", "kh"
    common = {"slope": slope, "boundary": boundary, "gamma": gamma}
    if kind == "mhd2":
        return _steps(None, "mhd", _log_int(rng, 24, 1400), _log_int(rng, 24, 1400), 1,
                      rng.randint(5, 20), problem=problem2, precision=precision,
                      riemann=riemann, **common)
    if kind == "mhd3":
        return _steps(None, "mhd", _log_int(rng, 12, 160), _log_int(rng, 12, 160),
                      _log_int(rng, 12, 160), rng.randint(3, 8), problem=problem3,
                      precision=precision, riemann=riemann, **common)
    if kind == "loop":
        return _steps(None, "loop", _log_int(rng, 24, 256), _log_int(rng, 24, 256), 1,
                      rng.randint(5, 20), problem=problem2, precision=precision, **common)
    if kind == "hydro2":
        return _steps(None, "hydro", _log_int(rng, 24, 3000), _log_int(rng, 24, 3000), 1,
                      rng.randint(5, 20), problem=rng.choice(["implode", "blast", "kh"]),
                      riemann=rng.choice(["hllc", "approx", "hll", "llf"]),
                      precision=rng.choice(["fp64", "fp64", "strict"]), **common)
    if kind == "hydro3":
        return _steps(None, "hydro", _log_int(rng, 12, 200), _log_int(rng, 12, 200),
                      _log_int(rng, 12, 200), rng.randint(3, 8),
                      problem=rng.choice(["implode", "blast", "kh"]),
                      riemann=rng.choice(["hllc", "approx", "llf"]),
                      precision=rng.choice(["fp64", "fp64", "strict"]), **common)
    if kind in ("batch", "batch3"):
        dim = 2 if kind == "batch" else 3
        return {"kind": "batch", "dim": dim, "members": rng.randint(2, 32 if dim == 2 else 8),
                "max_side": rng.choice([64, 128, 256, 384] if dim == 2 else [24, 32, 48]),
                "steps": rng.randint(20, 60), "riemann": riemann, "slope": slope,
                "boundary": rng.choice(["periodic", "open"]),
                "precision": rng.choice(["fp64", "fp64", "fp32", "strict"]),
                "autotune": rng.random() < 0.5}
    if kind == "surrogate":
        three = rng.random() < 0.5
        n = [_log_int(rng, 24, 96) if three else _log_int(rng, 64, 900) for _ in range(3)]
        return _steps(None, "surrogate", n[0], n[1], n[2] if three else 1, rng.randint(3, 8),
                      problem="kh" if three else problem2,
                      precision=rng.choice(["fp64", "fp32"]), **common)
    if kind == "train":
        return {"kind": "train", "samples": _log_int(rng, 5000, 200000),
                "batch": 256 * _log_int(rng, 1, 32), "steps": rng.randint(10, 60)}
    if kind == "gradient":
        return {"kind": "gradient", "samples": 256 * _log_int(rng, 1, 64)}
    return {"kind": "infer", "samples": _log_int(rng, 1, 400000)}


# ---- parameters and initial states ------------------------------------------------------------
def _is3(case):
    return case.get("nz", 1) > 1


def _box(case):
    """Physical extent: unit cells along the longest side, so that dx = dy = dz nearly."""
    n = max(case["nx"], case["ny"], case["nz"])
    return case["nx"] / n, case["ny"] / n, case["nz"] / n


def _params(case):
    lx, ly, lz = _box(case)
    make = make_hydro_params if case["kind"] == "hydro" else make_params
    return make(3 if _is3(case) else 2, case["nx"], case["ny"], case["nz"], xmax=lx, ymax=ly,
                zmax=lz if _is3(case) else 1.0, gamma0=case["gamma"], cfl=0.8,
                slope_type=case["slope"], riemann=RIEMANN[case["riemann"]],
                bc=BOUNDARY[case["boundary"]], tEnd=1e9, n_step_max=1 << 30,
                precision=PRECISION[case["precision"]], float_round=False)


def _coords(p, dev):
    """Cell-centre coordinates of the padded box, broadcastable to (k, j, i)."""
    gw = p.ghost_width
    x = p.xmin + (torch.arange(p.isize, dtype=torch.float64, device=dev) - gw + 0.5) * p.dx
    y = p.ymin + (torch.arange(p.jsize, dtype=torch.float64, device=dev) - gw + 0.5) * p.dy
    z = torch.zeros(1, dtype=torch.float64, device=dev)
    if p.dim == 3:
        z = p.zmin + (torch.arange(p.ksize, dtype=torch.float64, device=dev) - gw + 0.5) * p.dz
    return x.view(1, 1, -1), y.view(1, -1, 1), z.view(-1, 1, 1)


def _initial(p, problem, seed, dev):
    """Initial state (variables, k, j, i) of a problem, its free parameters from the seed."""
    rng = np.random.RandomState(seed % (1 << 31))
    x, y, z = _coords(p, dev)
    shape = (p.ksize, p.jsize, p.isize)
    lx, ly, lz = p.xmax - p.xmin, p.ymax - p.ymin, p.zmax - p.zmin
    one = torch.ones(shape, dtype=torch.float64, device=dev)
    zero = torch.zeros_like(one)
    two_pi = 2 * math.pi
    sx, sy, sz = x / lx, y / ly, (z / lz if p.dim == 3 else z)
    # a few per cent of smooth density structure, so that no region is exactly uniform
    ph = rng.rand(3) * two_pi
    ripple = 0.02 * torch.sin(two_pi * sx + ph[0]) * torch.cos(two_pi * sy + ph[1]) * \
        torch.cos(two_pi * sz + ph[2])
    vel = [zero, zero, zero]
    bfield = [zero, zero, zero]
    if problem == "ot":  # Orszag-Tang vortex, field amplitude and phases from the seed
        b0 = rng.uniform(0.5, 2.0) / math.sqrt(4 * math.pi)
        rho = 25 / (36 * math.pi) * (one + ripple)
        pre = 5 / (12 * math.pi) * one
        a, b = rng.rand(2) * two_pi
        vel = [-torch.sin(two_pi * sy + a) * one, torch.sin(two_pi * sx + b) * one, zero]
        bfield = [-b0 * torch.sin(two_pi * sy + a) * one, b0 * torch.sin(2 * two_pi * sx + b) * one,
                  zero]
    elif problem == "blast":  # over-pressured sphere in a uniform oblique field
        c = rng.uniform(0.4, 0.6, 3)
        r2 = (x - c[0] * lx) ** 2 + (y - c[1] * ly) ** 2
        if p.dim == 3:
            r2 = r2 + (z - c[2] * lz) ** 2
        radius = rng.uniform(0.08, 0.15) * min(lx, ly, lz if p.dim == 3 else ly)
        rho = one + ripple
        pre = torch.where(r2 < radius * radius, 10.0, 0.1) * one
        n = rng.randn(3)
        n = n / np.linalg.norm(n)
        bfield = [float(v) * one for v in n]
    elif problem == "kh":  # shear layers with a random velocity perturbation
        gen = torch.Generator(device="cpu").manual_seed(seed % (1 << 31))
        inner = ((sy - 0.5).abs() < 0.25) & (one > 0)
        rho = torch.where(inner, 2.0, 1.0) * (one + ripple)
        pre = 2.5 * one
        noise = [0.02 * (torch.rand(shape, dtype=torch.float32, generator=gen).to(dev).double()
                         - 0.5) for _ in range(p.dim)]
        vel = [torch.where(inner, -0.5, 0.5) + noise[0], noise[1],
               noise[2] if p.dim == 3 else zero]
        bfield = [0.1 * rng.uniform(0.5, 1.5) * one, zero, zero]
    else:  # "implode": light corner below a diagonal
        cut = rng.uniform(0.4, 0.6)
        s = sx + sy + sz
        outer = (s > cut * (2.0 if p.dim == 2 else 3.0)) & (one > 0)
        rho = torch.where(outer, 1.0, 0.125) * (one + ripple)
        pre = torch.where(outer, 1.0, 0.14) * one
    nv = 8 if p.ghost_width == 3 else p.dim + 2
    ke = 0.5 * rho * sum(v * v for v in vel)
    U = torch.zeros((nv,) + shape, dtype=torch.float64, device=dev)
    U[0], U[2], U[3] = rho, rho * vel[0], rho * vel[1]
    U[1] = pre / (p.gamma0 - 1) + ke
    if nv != 4:
        U[4] = rho * vel[2]
    if nv == 8:
        # these fields do not vary along their own direction: the centred values are the face
        # values, and the discrete divergence is zero
        U[1] += 0.5 * sum(b * b for b in bfield)
        for d in range(3):
            U[5 + d] = bfield[d]
    return U


def _batch_members(case, seed):
    """(params, problem name, seed) of the members: sides, gamma and field from the seed."""
    rng = np.random.RandomState((seed + 7919) % (1 << 31))
    # the sides do not depend on the seed (other inputs, the same work)
    sides = np.random.RandomState(case["members"])
    out = []
    for m in range(case["members"]):
        if case["dim"] == 2:
            side = int(sides.choice([s for s in BATCH_SIDES if s <= case["max_side"]]))
            n = (side, side, 1)
        else:
            n = tuple(int(v) for v in sides.randint(12, case["max_side"] + 1, 3))
        p = make_params(case["dim"], *n, gamma0=float(rng.uniform(1.4, 2.0)), cfl=0.8,
                        slope_type=case["slope"], riemann=RIEMANN[case["riemann"]],
                        bc=BOUNDARY[case["boundary"]], tEnd=1e9, n_step_max=1 << 30,
                        precision=PRECISION[case["precision"]], float_round=False)
        out.append((p, "ot" if case["dim"] == 2 else "kh", seed * 131 + m))
    return out


def _net_params(seed, trained):
    """A network's parameter vector: hidden weights as a fresh network has them; `trained`
    standardises inputs and outputs by the typical spreads of face samples, with corrections
    that are a small part of them."""
    rng = np.random.RandomState((seed + 104729) % (1 << 31))
    P = np.zeros(S.N_PARAMS, dtype=np.float32)
    for off, n, fan in ((S.W1, 128 * 16, 16), (S.W2, 128 * 128, 128), (S.W3, 8 * 128, 128)):
        P[off:off + n] = rng.uniform(-1, 1, n) * math.sqrt(6.0 / fan)
    P[S.W3:S.B3] *= 0.1
    P[S.ISIG_IN:S.MU_OUT] = 1.0
    P[S.SIG_OUT:S.N_PARAMS] = 1.0
    if trained:
        P[S.ISIG_IN:S.MU_OUT] = [50] + [3] * 3 + [5] * 3 + [5, 10] + [50] * 6 + [1]
        P[S.MU_IN + 7] = 0.3
        P[S.SIG_OUT:S.N_PARAMS] = 1e-4
    return P


def _samples(n, seed):
    """Features and targets with a smooth nonlinear relation and a little noise."""
    g = torch.Generator(device="cpu").manual_seed((seed + 15485863) % (1 << 31))
    X = torch.randn((n, 16), generator=g)
    M = torch.randn((16, 8), generator=g) / 4
    T = torch.tanh(X @ M) + 0.3 * (X[:, :8] * X[:, 8:]) + 0.02 * torch.randn((n, 8), generator=g)
    return X.numpy(), T.numpy()


# ---- prepare / run ----------------------------------------------------------------------------
class _DeviceArray:
    """A solver's device state, seen by torch.  The tensor made from it holds this object, so
    the solver and its buffers live as long as the tensor."""

    def __init__(self, solver, ptr):
        self.solver = solver
        self.__cuda_array_interface__ = {"shape": tuple(solver.params.shape), "typestr": "<f8",
                                         "data": (ptr, False), "version": 3}


def _view(solver, ptr):
    return torch.as_tensor(_DeviceArray(solver, ptr), device="cuda")


def _state_of(st):
    """The solver's device state as a tensor (its two buffers are wrapped once each)."""
    ptr = st["solver"].device_state_ptr()
    if ptr not in st["views"]:
        st["views"][ptr] = _view(st["solver"], ptr)
    return st["views"][ptr]


def _start(st):
    """Put the solver's or the members' initial states in place."""
    if "batch" in st:
        for m, U in enumerate(st["initial"]):
            st["batch"].upload(m, U)
    else:
        _state_of(st).copy_(st["initial"])
        torch.cuda.current_stream().synchronize()  # the solver's stream reads it
    st["done"] = 0


def _advance(st):
    """Count the steps of a pass.  A program that is called again and again starts its problem
    afresh after a run's length (about 600 steps): the problems are not made to run for ever."""
    st["done"] += st["case"]["steps"]
    if st["done"] > max(600, st["case"]["steps"]):
        _start(st)
        st["done"] = st["case"]["steps"]


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind in ("mhd", "loop", "hydro", "surrogate"):
        p = _params(case)
        st["solver"] = (SolverHydroMuscl if kind == "hydro" else SolverMHDMuscl)(p)
        st["views"] = {}
        st["initial"] = _initial(p, case["problem"], seed, "cuda")
        _start(st)
    if kind == "surrogate":
        st["net"] = S.MLP(0)
        st["net"].set_params(_net_params(seed, True))
        S.attach(st["solver"], st["net"], 0.005, 0.005)
    if kind == "batch":
        members = _batch_members(case, seed)
        st["batch"] = BatchSolver([p for p, _, _ in members])
        st["initial"] = [_initial(*m, "cuda").cpu().numpy() for m in members]
        _start(st)
        if case["autotune"]:
            st["batch"].autotune(3)
    if kind in ("train", "gradient", "infer"):
        st["net"] = S.MLP(0)
        st["net"].set_params(_net_params(seed, False))
        X, T = _samples(case["samples"], seed)
        st["X"], st["T"] = X, T
        if kind == "train":
            st["set"] = S.FaceSet(case["samples"])
            st["set"].append(X, T)
            st["seed"] = seed & 0xFFFF
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind not in ("train", "gradient", "infer"):
        _advance(st)
    if kind in ("mhd", "hydro", "surrogate"):
        s = st["solver"]
        s.run(case["steps"])
        return {"t": s.m_t, "U": _state_of(st)}
    if kind == "loop":
        s = st["solver"]
        for _ in range(case["steps"]):
            if s.finished():
                break
            s.next_iteration()
        return {"t": s.m_t, "U": _state_of(st)}
    if kind == "batch":
        b = st["batch"]
        b.run(case["steps"])
        return [b.download(m) for m in range(len(b))]
    if kind == "train":
        st["net"].train(st["set"], case["steps"], batch=case["batch"], lr=1e-3, seed=st["seed"])
        return st["net"].get_params()
    if kind == "gradient":
        return st["net"].gradient(st["X"], st["T"])
    return st["net"].infer(st["X"])


# ---- work and tolerance ------------------------------------------------------------------------
# operations per cell and step: adds, multiplies, divisions and square roots of the scheme
FLOPS = {("mhd", 2): 1682.0, ("mhd", 3): 3367.0, ("hydro", 2): 386.0, ("hydro", 3): 667.0}
NET = 2.0 * (16 * 128 + 128 * 128 + 128 * 8)  # multiply-adds of one network evaluation


def work(case):
    kind = case["kind"]
    if kind in ("mhd", "loop", "hydro", "surrogate"):
        dim = 3 if _is3(case) else 2
        cells = float(case["nx"] * case["ny"] * case["nz"]) * case["steps"]
        nv = (dim + 2) if kind == "hydro" else 8
        flops = FLOPS["hydro" if kind == "hydro" else "mhd", dim]
        if kind == "surrogate":
            flops += dim * NET
        return {"bytes": 2 * 8 * nv * cells, "flops": flops * cells}
    if kind == "batch":
        cells = sum(float(p.nx * p.ny * p.nz) for p, _, _ in _batch_members(case, 0))
        return {"bytes": 2 * 64 * cells * case["steps"],
                "flops": FLOPS["mhd", case["dim"]] * cells * case["steps"]}
    params = 4.0 * S.N_PARAMS
    if kind == "train":  # per step: the samples, the weights and Adam's two moments updated
        return {"bytes": case["steps"] * (case["batch"] * 96.0 + 6 * params),
                "flops": case["steps"] * case["batch"] * 3 * NET}
    if kind == "gradient":
        return {"bytes": case["samples"] * 96.0 + 2 * params, "flops": case["samples"] * 3 * NET}
    return {"bytes": case["samples"] * 96.0 + params, "flops": case["samples"] * NET}


def tolerance(case):
    """About four times the largest difference seen between these kernels and exact()."""
    kind = case["kind"]
    if kind in ("infer", "gradient"):
        return {"rel": 0.02, "max": 0.5}  # bf16 activations
    if kind == "train":
        return {"rel": 0.007, "max": 0.5}  # the same, through Adam
    if kind == "surrogate":
        return {"rel": 2e-6, "max": 5e-3}  # bf16 corrections, refused or accepted face by face
    if case["precision"] == "fp32":
        return {"rel": 5e-6, "max": 1e-3}
    return {"rel": 1e-11, "max": 1e-7}  # roundoff, grown over up to 200 steps


# ---- exact: the scheme in plain torch, 64 bits -------------------------------------------------
def _sh(a, d, n):
    """a at index + n along direction d (0 x, 1 y, 2 z)."""
    return torch.roll(a, -n, -1 - d)


def _fill_ghosts(U, dim, gw, bc, vectors):
    """Ghost cells of x, then y, then z; `vectors`: first index of each vector's components."""
    for d in range(dim):
        ax = U[0].dim() - 1 - d
        n = U[0].shape[ax] - 2 * gw
        for up in (0, 1):
            kind = bc[2 * d + up]
            for g in range(gw):
                c = n + gw + g if up else g
                if kind == A.BC_DIRICHLET:
                    src = 2 * n + 2 * gw - 1 - c if up else 2 * gw - 1 - c
                elif kind == A.BC_NEUMANN:
                    src = n + gw - 1 if up else gw
                else:
                    src = c - n if up else c + n
                for v in range(len(U)):
                    flip = kind == A.BC_DIRICHLET and any(v == b + d for b in vectors)
                    x = U[v].select(ax, src)
                    U[v].select(ax, c).copy_(-x if flip else x)


def _inner(a, dim, gw):
    for d in range(dim):
        ax = a.dim() - 1 - d
        a = a.narrow(ax, gw, a.shape[ax] - 2 * gw)
    return a


def _slope(st, q, qp, qm):
    l, r, c = st * (q - qm), st * (qp - q), 0.5 * (qp - qm)
    s = torch.minimum(torch.minimum(l.abs(), r.abs()), c.abs())
    return torch.where(l * r <= 0, torch.zeros_like(s), torch.copysign(s, c))


def _fast(q, n, g):
    """Fast magnetosonic speed of a primitive state along the field component n (0, 1, 2)."""
    c2 = g * q[1] / q[0]
    d2 = 0.5 * ((q[5] ** 2 + q[6] ** 2 + q[7] ** 2) / q[0] + c2)
    return torch.sqrt(d2 + torch.sqrt((d2 * d2 - c2 * q[5 + n] ** 2 / q[0]).clamp_min(0)))


def _cons_flux(q, g):
    """Conservative state and ideal MHD flux (normal x)."""
    d, p, u, v, w, a, b, c = q
    em = 0.5 * (a * a + b * b + c * c)
    e = p / (g - 1) + 0.5 * d * (u * u + v * v + w * w) + em
    pt = p + em
    U = [d, e, d * u, d * v, d * w, a, b, c]
    F = [d * u, (e + pt) * u - a * (a * u + b * v + c * w), d * u * u - a * a + pt,
         d * u * v - a * b, d * u * w - a * c, torch.zeros_like(d), b * u - a * v, c * u - a * w]
    return U, F


def _llf(l, r, g):
    ul, fl = _cons_flux(l, g)
    ur, fr = _cons_flux(r, g)
    s = torch.maximum(_fast(l, 0, g) + l[2].abs(), _fast(r, 0, g) + r[2].abs())
    return [0.5 * (a + b) - 0.5 * s * (y - x) for a, b, x, y in zip(fl, fr, ul, ur)], s, ul, ur, fl, fr


def _hlld(l, r, g):
    """Miyoshi and Kusano (2005); l, r share the normal field l[5]."""
    a = l[5]
    sg = torch.where(a >= 0, 1.0, -1.0).to(a.dtype)
    cf = torch.maximum(_fast(l, 0, g), _fast(r, 0, g))
    sl, sr = torch.minimum(l[2], r[2]) - cf, torch.maximum(l[2], r[2]) + cf

    def side(q):
        em = 0.5 * (a * a + q[6] ** 2 + q[7] ** 2)
        e = q[1] / (g - 1) + 0.5 * q[0] * (q[2] ** 2 + q[3] ** 2 + q[4] ** 2) + em
        return e, q[1] + em, q[2] * a + q[3] * q[6] + q[4] * q[7]

    el, ptl, vbl = side(l)
    er, ptr, vbr = side(r)
    rcl, rcr = l[0] * (l[2] - sl), r[0] * (sr - r[2])
    us = (rcr * r[2] + rcl * l[2] + (ptl - ptr)) / (rcr + rcl)
    pts = (rcr * ptl + rcl * ptr + rcl * rcr * (l[2] - r[2])) / (rcr + rcl)

    def star(q, s, e, pt, vb):
        rs = q[0] * (s - q[2]) / (s - us)
        den = q[0] * (s - q[2]) * (s - us) - a * a
        num = q[0] * (s - q[2]) ** 2 - a * a
        deg = (a * a > 0) & ((den - a * a).abs() <= 1e-8 * a * a)
        den = torch.where(deg, torch.ones_like(den), den)
        vs = torch.where(deg, q[3], q[3] - a * q[6] * (us - q[2]) / den)
        ws = torch.where(deg, q[4], q[4] - a * q[7] * (us - q[2]) / den)
        bs = torch.where(deg, q[6], q[6] * num / den)
        cs = torch.where(deg, q[7], q[7] * num / den)
        vbs = us * a + vs * bs + ws * cs
        es = ((s - q[2]) * e - pt * q[2] + pts * us + a * (vb - vbs)) / (s - us)
        return rs, vs, ws, bs, cs, vbs, es

    rsl, vsl, wsl, bsl, csl, vbsl, esl = star(l, sl, el, ptl, vbl)
    rsr, vsr, wsr, bsr, csr, vbsr, esr = star(r, sr, er, ptr, vbr)
    ql, qr = torch.sqrt(rsl), torch.sqrt(rsr)
    sal, sar = us - a.abs() / ql, us + a.abs() / qr
    sm = ql + qr
    vss = (ql * vsl + qr * vsr + sg * (bsr - bsl)) / sm
    wss = (ql * wsl + qr * wsr + sg * (csr - csl)) / sm
    bss = (ql * bsr + qr * bsl + sg * ql * qr * (vsr - vsl)) / sm
    css = (ql * csr + qr * csl + sg * ql * qr * (wsr - wsl)) / sm
    vbss = us * a + vss * bss + wss * css
    essl, essr = esl - sg * ql * (vbsl - vbss), esr + sg * qr * (vbsr - vbss)
    regions = [(sl > 0, [l[0], l[2], l[3], l[4], l[6], l[7], ptl, el, vbl]),
               (sal > 0, [rsl, us, vsl, wsl, bsl, csl, pts, esl, vbsl]),
               (us > 0, [rsl, us, vss, wss, bss, css, pts, essl, vbss]),
               (sar > 0, [rsr, us, vss, wss, bss, css, pts, essr, vbss]),
               (sr > 0, [rsr, us, vsr, wsr, bsr, csr, pts, esr, vbsr])]
    o = [r[0], r[2], r[3], r[4], r[6], r[7], ptr, er, vbr]
    for cond, val in reversed(regions):
        o = [torch.where(cond, x, y) for x, y in zip(val, o)]
    ro, uo, vo, wo, bo, co, pt, e, vb = o
    return [ro * uo, (e + pt) * uo - a * vb, ro * uo * uo - a * a + pt, ro * uo * vo - a * bo,
            ro * uo * wo - a * co, torch.zeros_like(a), bo * uo - a * vo, co * uo - a * wo]


def _hll(l, r, g):
    ul, fl = _cons_flux(l, g)
    ur, fr = _cons_flux(r, g)
    cf = torch.maximum(_fast(l, 0, g), _fast(r, 0, g))
    sl = (torch.minimum(l[2], r[2]) - cf).clamp_max(0)
    sr = (torch.maximum(l[2], r[2]) + cf).clamp_min(0)
    return [(sr * x - sl * y + sr * sl * (b - c)) / (sr - sl) for x, y, c, b in zip(fl, fr, ul, ur)]


def _surrogate_flux(l, r, g, net):
    """LLF flux plus the network's correction where the gate and the admissibility check allow
    it, HLLD elsewhere."""
    f0, s, ul, ur, fl, fr = _llf(l, r, g)
    hl = _hlld(l, r, g)
    rb = 0.5 * (l[0] + r[0])
    ib, ip = 1 / (torch.sqrt(rb) * s), 1 / (rb * s * s)
    m = lambda v: 0.5 * (l[v] + r[v])  # noqa: E731
    d = lambda v: r[v] - l[v]  # noqa: E731
    x = torch.stack([d(0) / rb, m(2) / s, m(3) / s, m(4) / s, l[5] * ib, m(6) * ib, m(7) * ib,
                     m(1) * ip, torch.zeros_like(s) + (g - 5 / 3), d(2) / s, d(3) / s, d(4) / s,
                     d(6) * ib, d(7) * ib, d(1) * ip, torch.zeros_like(s)], -1).nan_to_num()
    y = _mlp(net, x.reshape(-1, 16))[0].reshape(x.shape[:-1] + (8,))
    sc = [rb * s, rb * s ** 3, rb * s * s, rb * s * s, rb * s * s, torch.zeros_like(s),
          torch.sqrt(rb) * s * s, torch.sqrt(rb) * s * s]
    F = [f0[v] + sc[v] * (net["mu_out"][v] + net["sig_out"][v] * y[..., v]) for v in range(8)]
    ok = (d(0).abs() < 0.005 * torch.minimum(l[0], r[0])) & \
        (d(1).abs() < 0.005 * torch.minimum(l[1], r[1]))
    for U, f, sign in ((ul, fl, -1.0), (ur, fr, 1.0)):
        a = [U[v] + sign * (F[v] - f[v]) / s for v in range(8)]
        pr = a[1] - 0.5 * (a[2] ** 2 + a[3] ** 2 + a[4] ** 2) / a[0] - \
            0.5 * (a[5] ** 2 + a[6] ** 2 + a[7] ** 2)
        ok = ok & (a[0] > 0) & (pr > 0)
    return [torch.where(ok, x, y) for x, y in zip(F, hl)]


def _emf2d(rt, rb, lt, lb, perm, g, smallc):
    """2D HLLD EMF of an edge from its four states; perm: the (u, v) and (a, b, c) indexes."""
    u, v, ia, ib, ic = perm
    top, bot = 0.5 * (rt[ia] + lt[ia]), 0.5 * (rb[ia] + lb[ia])
    right, left = 0.5 * (rt[ib] + rb[ib]), 0.5 * (lt[ib] + lb[ib])
    st = {"LL": (rt, top, right), "RL": (lt, top, left), "LR": (rb, bot, right),
          "RR": (lb, bot, left)}
    q = {k: [s[0], s[1], s[u], s[v], None, a, b, s[ic]] for k, (s, a, b) in st.items()}
    mx = lambda xs: torch.stack(xs).amax(0)  # noqa: E731
    mn = lambda xs: torch.stack(xs).amin(0)  # noqa: E731
    keys = ("LL", "LR", "RL", "RR")
    cx, cy = mx([_fast(q[k], 0, g) for k in keys]), mx([_fast(q[k], 1, g) for k in keys])
    SL, SR = mn([q[k][2] for k in keys]) - cx, mx([q[k][2] for k in keys]) + cx
    SB, ST = mn([q[k][3] for k in keys]) - cy, mx([q[k][3] for k in keys]) + cy
    pt = {k: q[k][1] + 0.5 * (q[k][5] ** 2 + q[k][6] ** 2 + q[k][7] ** 2) for k in keys}
    sx = {"LL": SL, "LR": SL, "RL": SR, "RR": SR}
    sy = {"LL": SB, "RL": SB, "LR": ST, "RR": ST}
    rcx = {k: q[k][0] * (q[k][2] - sx[k]).abs() for k in keys}
    rcy = {k: q[k][0] * (q[k][3] - sy[k]).abs() for k in keys}
    us = (sum(rcx[k] * q[k][2] for k in keys) + (pt["LL"] - pt["RL"] + pt["LR"] - pt["RR"])) / \
        sum(rcx[k] for k in keys)
    vs = (sum(rcy[k] * q[k][3] for k in keys) + (pt["LL"] - pt["LR"] + pt["RL"] - pt["RR"])) / \
        sum(rcy[k] for k in keys)
    fx = {k: (sx[k] - q[k][2]) / (sx[k] - us) for k in keys}
    fy = {k: (sy[k] - q[k][3]) / (sy[k] - vs) for k in keys}
    rx, ry = {k: q[k][0] * fx[k] for k in keys}, {k: q[k][0] * fy[k] for k in keys}
    rr = {k: q[k][0] * fx[k] * fy[k] for k in keys}
    Bs, As = {k: q[k][6] * fx[k] for k in keys}, {k: q[k][5] * fy[k] for k in keys}
    Ex = {k: us * Bs[k] - q[k][3] * q[k][5] for k in keys}
    Ey = {k: q[k][2] * q[k][6] - vs * As[k] for k in keys}
    Ess = {k: us * Bs[k] - vs * As[k] for k in keys}
    E0 = {k: q[k][2] * q[k][6] - q[k][3] * q[k][5] for k in keys}

    def alf(ks, n, r1, ss):
        return mx([q[k][n].abs() / torch.sqrt(r1[k]) for k in ks] +
                  [ss[k].abs() / torch.sqrt(rr[k]) for k in ks]).clamp_min(smallc)

    SAL = (us - alf(("LR", "LL"), 5, rx, As)).clamp_max(0)
    SAR = (us + alf(("RR", "RL"), 5, rx, As)).clamp_min(0)
    SAB = (vs - alf(("LL", "RL"), 6, ry, Bs)).clamp_max(0)
    SAT = (vs + alf(("LR", "RR"), 6, ry, Bs)).clamp_min(0)
    wx, wy = SAR - SAL, SAT - SAB
    AT, AB = (SAR * As["RR"] - SAL * As["LR"]) / wx, (SAR * As["RL"] - SAL * As["LL"]) / wx
    BR, BL = (SAT * Bs["RR"] - SAB * Bs["RL"]) / wy, (SAT * Bs["LR"] - SAB * Bs["LL"]) / wy
    Ec = (SAL * SAB * Ess["RR"] - SAL * SAT * Ess["RL"] - SAR * SAB * Ess["LR"] +
          SAR * SAT * Ess["LL"]) / wx / wy - SAT * SAB / wy * (AT - AB) + SAR * SAL / wx * (BR - BL)
    Eb = (SAR * Ex["LL"] - SAL * Ex["RL"] + SAR * SAL * (q["RL"][6] - q["LL"][6])) / wx
    Et = (SAR * Ex["LR"] - SAL * Ex["RR"] + SAR * SAL * (q["RR"][6] - q["LR"][6])) / wx
    El = (SAT * Ey["LL"] - SAB * Ey["LR"] - SAT * SAB * (q["LR"][5] - q["LL"][5])) / wy
    Er = (SAT * Ey["RL"] - SAB * Ey["RR"] - SAT * SAB * (q["RR"][5] - q["RL"][5])) / wy
    w = torch.where
    low = w(SL >= 0, E0["LL"], w(SR >= 0, Eb, E0["RL"]))
    high = w(SL >= 0, E0["LR"], w(SR >= 0, Et, E0["RR"]))
    mid = w(SL >= 0, El, w(SR >= 0, Ec, Er))
    return w(SB >= 0, low, w(ST >= 0, mid, high))


def _mhd_step(U, p, g, dx, flux):
    """One CFL step of the list U of 8 padded arrays in place (leading dimensions, if any, are
    independent runs: g and dx broadcast over them); returns dt."""
    dim, gw = p.dim, 3
    _fill_ghosts(U, dim, gw, list(p.bc), (2, 5))
    z = dim == 3
    r = U[0].clamp_min(p.smallr)
    u, v, w = U[2] / r, U[3] / r, U[4] / r
    a, b = 0.5 * (U[5] + _sh(U[5], 0, 1)), 0.5 * (U[6] + _sh(U[6], 1, 1))
    c = 0.5 * (U[7] + _sh(U[7], 2, 1)) if z else 0.5 * U[7]
    smallp = p.smallc * p.smallc / g
    e = (U[1] - 0.5 * (a * a + b * b + c * c)) / r - 0.5 * (u * u + v * v + w * w)
    q = [r, torch.maximum((g - 1) * r * e, r * smallp), u, v, w, a, b, c]
    inv = sum((_fast(q, d, g) + q[2 + d].abs()) / dx[d] for d in range(dim))
    dims = tuple(range(-dim, 0))
    dt = p.cfl / _inner(inv, dim, gw).amax(dims, keepdim=True)
    h = [dt / dx[d] for d in range(dim)] + [torch.zeros_like(dt)] * (3 - dim)

    def edge(i, j):  # v_i B_j - v_j B_i at the edge normal to (i, j), lower side of both
        av = lambda f: 0.25 * (f + _sh(f, i, -1) + _sh(f, j, -1) + _sh(_sh(f, i, -1), j, -1))  # noqa: E731
        bi, bj = 0.5 * (U[5 + i] + _sh(U[5 + i], j, -1)), 0.5 * (U[5 + j] + _sh(U[5 + j], i, -1))
        return av(q[2 + i]) * bj - av(q[2 + j]) * bi

    zero = torch.zeros_like(r)
    E = [edge(1, 2), edge(2, 0), edge(0, 1)] if z else [zero, zero, edge(0, 1)]
    st = p.slope_type
    D = [[0.5 * _slope(st, f, _sh(f, d, 1), _sh(f, d, -1)) if d < dim else zero for f in q]
         for d in range(3)]
    face = [U[5], U[6], U[7]]
    dn = [0.5 * (_sh(face[d], d, 1) - face[d]) if d < dim else zero for d in range(3)]
    for d in range(dim):
        D[d][5 + d] = dn[d]
    # transverse slopes of the face fields: dF[n][t], field n along t
    dF = [[0.5 * _slope(st, face[n], _sh(face[n], t, 1), _sh(face[n], t, -1))
           if t != n and t < dim else zero for t in range(3)] for n in range(3)]
    vel, mag = [u, v, w], [a, b, c]
    src = [zero.clone() for _ in range(8)]
    for d in range(dim):
        X = D[d]
        src[0] = src[0] - (vel[d] * X[0] + X[2 + d] * r) * h[d]
        src[1] = src[1] - (vel[d] * X[1] + X[2 + d] * g * q[1]) * h[d]
        for n in range(3):
            t = -vel[d] * X[2 + n]
            if n == d:  # pressure and the transverse magnetic pressure
                t = t - (X[1] + sum(mag[m] * X[5 + m] for m in range(3) if m != d)) / r
            else:  # tension
                t = t + mag[d] * X[5 + n] / r
            src[2 + n] = src[2 + n] + t * h[d]
            if n != d:  # induction: (v_n B_d - v_d B_n) along d
                src[5 + n] = src[5 + n] + (vel[n] * X[5 + d] + mag[d] * X[2 + n] -
                                           vel[d] * X[5 + n] - mag[n] * X[2 + d]) * h[d]
    m = [x + s for x, s in zip(q, src)]
    cd = lambda f, d: _sh(f, d, 1) - f  # noqa: E731
    L = [face[0] + 0.5 * (cd(E[2], 1) * h[1] - (cd(E[1], 2) * h[2] if z else 0)),
         face[1] + 0.5 * (-cd(E[2], 0) * h[0] + (cd(E[0], 2) * h[2] if z else 0)),
         face[2] + 0.5 * (cd(E[1], 0) * h[0] - cd(E[0], 1) * h[1]) if z else face[2]]
    R = [_sh(L[d], d, 1) if d < dim else None for d in range(3)]
    dR = [[_sh(dF[n][t], n, 1) if n < dim else None for t in range(3)] for n in range(3)]

    def floors(s):
        s[0] = s[0].clamp_min(p.smallr)
        s[1] = torch.maximum(smallp + 0 * s[0] if z else smallp * s[0], s[1])
        return s

    def face_state(d, sign):
        s = [m[k] + sign * D[d][k] for k in range(8)]
        s[5 + d] = R[d] if sign > 0 else L[d]
        return floors(s)

    def edge_state(i, j, si, sj):  # corner of the cell in the plane (i, j)
        s = [m[k] + (si * D[i][k] + sj * D[j][k]) for k in range(8)]
        s[5 + i] = R[i] + sj * dR[i][j] if si > 0 else L[i] + sj * dF[i][j]
        s[5 + j] = R[j] + si * dR[j][i] if sj > 0 else L[j] + si * dF[j][i]
        return floors(s)

    new = [x.clone() for x in U]
    hydro = range(5) if z else (0, 1, 2, 3, 4, 7)
    for d in range(dim):
        def rot(s):
            s = list(s)
            if d:
                s[2], s[2 + d] = s[2 + d], s[2]
                s[5], s[5 + d] = s[5 + d], s[5]
            return s

        ql = rot([_sh(x, d, -1) for x in face_state(d, 1)])
        qr = rot(face_state(d, -1))
        ql[5] = qr[5] = 0.5 * (ql[5] + qr[5])
        F = rot(flux(ql, qr, g))
        for k in hydro:
            new[k] = new[k] + (F[k] - _sh(F[k], d, 1)) * h[d]

    def emf(i, j):  # along the third direction; (i, j) in the solver's (u, v) order
        at = lambda s, si, sj: [_sh(_sh(x, i, -si), j, -sj) for x in s]  # noqa: E731
        rt, rb = at(edge_state(i, j, 1, 1), 1, 1), at(edge_state(i, j, 1, -1), 1, 0)
        lt, lb = at(edge_state(i, j, -1, 1), 0, 1), edge_state(i, j, -1, -1)
        k = 3 - i - j
        return _emf2d(rt, rb, lt, lb, (2 + i, 2 + j, 5 + i, 5 + j, 5 + k), g, p.smallc)

    EZ = emf(0, 1)
    new[5] = new[5] + cd(EZ, 1) * h[1]
    new[6] = new[6] - cd(EZ, 0) * h[0]
    if z:
        EX, EY = emf(1, 2), emf(2, 0)
        new[5] = new[5] - cd(EY, 2) * h[2]
        new[6] = new[6] + cd(EX, 2) * h[2]
        new[7] = new[7] + cd(EY, 0) * h[0] - cd(EX, 1) * h[1]
    for k in range(8):
        _inner(U[k], dim, gw).copy_(_inner(new[k], dim, gw))
    return dt


def _two_shock(l, r, p, nv):
    """Two-shock approximate solver with Newton iterations (the solvers' "approx")."""
    g, sr, sc = p.gamma0, p.smallr, p.smallc
    g6, sp, spp = (g + 1) / (2 * g), sc * sc / g, sr * sc * sc / g
    rl, rr = l[0].clamp_min(sr), r[0].clamp_min(sr)
    ul, ur = l[2], r[2]
    pl, pr = torch.maximum(l[1], rl * sp), torch.maximum(r[1], rr * sp)
    cl, cr = g * pl * rl, g * pr * rr
    wl, wr = torch.sqrt(cl), torch.sqrt(cr)
    ps = ((wr * pl + wl * pr + wl * wr * (ul - ur)) / (wl + wr)).clamp_min(0)
    live = torch.ones_like(ps, dtype=torch.bool)
    for _ in range(10):
        a, b = torch.sqrt(cl * (1 + g6 * (ps - pl) / pl)), torch.sqrt(cr * (1 + g6 * (ps - pr) / pr))
        qa, qb = 2 * a ** 3 / (a * a + cl), 2 * b ** 3 / (b * b + cr)
        dp = torch.maximum(qb * qa / (qb + qa) * ((ul - (ps - pl) / a) - (ur + (ps - pr) / b)), -ps)
        ps = torch.where(live, ps + dp, ps)
        live = live & ((dp / (ps + spp)).abs() > 1e-6)
    wl, wr = torch.sqrt(cl * (1 + g6 * (ps - pl) / pl)), torch.sqrt(cr * (1 + g6 * (ps - pr) / pr))
    us = 0.5 * (ul + (pl - ps) / wl + ur - (pr - ps) / wr)
    left = torch.copysign(torch.ones_like(us), us) > 0
    pick = lambda x, y: torch.where(left, x, y)  # noqa: E731
    sg = pick(torch.ones_like(us), -torch.ones_like(us))
    ro, uo, po, wo = pick(rl, rr), pick(ul, ur), pick(pl, pr), pick(wl, wr)
    co = torch.sqrt((g * po / ro).abs()).clamp_min(sc)
    rs = (ro / (1 + ro * (po - ps) / (wo * wo))).clamp_min(sr)
    cs = torch.sqrt((g * ps / rs).abs()).clamp_min(sc)
    so, si, sk = co - sg * uo, cs - sg * us, wo / ro - sg * uo
    shock = ps >= po
    so, si = torch.where(shock, sk, so), torch.where(shock, sk, si)
    scr = torch.maximum(so - si, sc + (so + si).abs())
    f = (0.5 * (1 + (so + si) / scr)).nan_to_num(0).clamp(0, 1)
    d, un, pg = f * rs + (1 - f) * ro, f * us + (1 - f) * uo, f * ps + (1 - f) * po
    out, ins = so < 0, si > 0
    d, un, pg = (torch.where(ins, x, torch.where(out, y, w))
                 for x, y, w in ((rs, ro, d), (us, uo, un), (ps, po, pg)))
    t = [pick(l[k], r[k]) for k in range(3, nv)]
    e = pg / (g - 1) + 0.5 * d * (un * un + sum(x * x for x in t))
    return [d * un, un * (e + pg), d * un * un + pg] + [d * un * x for x in t]


def _hydro_flux(l, r, p, nv, solver):
    if solver == "approx":
        return _two_shock(l, r, p, nv)
    g, sp = p.gamma0, p.smallc ** 2 / p.gamma0
    rl, rr = l[0].clamp_min(p.smallr), r[0].clamp_min(p.smallr)
    pl, pr = torch.maximum(l[1], rl * sp), torch.maximum(r[1], rr * sp)
    ul, ur = l[2], r[2]
    cl, cr = torch.sqrt(g * pl / rl), torch.sqrt(g * pr / rr)
    cm = torch.maximum(cl, cr)
    if solver == "hllc":
        cm = torch.maximum(cm, torch.full_like(cm, p.smallc))
        sl, sr = torch.minimum(ul, ur) - cm, torch.maximum(ul, ur) + cm
        el = pl / (g - 1) + 0.5 * rl * sum(l[k] ** 2 for k in range(2, nv))
        er = pr / (g - 1) + 0.5 * rr * sum(r[k] ** 2 for k in range(2, nv))
        rcl, rcr = rl * (ul - sl), rr * (sr - ur)
        us = (rcr * ur + rcl * ul + (pl - pr)) / (rcr + rcl)
        ps = (rcr * pl + rcl * pr + rcl * rcr * (ul - ur)) / (rcr + rcl)
        rsl, rsr = rl * (sl - ul) / (sl - us), rr * (sr - ur) / (sr - us)
        esl = ((sl - ul) * el - pl * ul + ps * us) / (sl - us)
        esr = ((sr - ur) * er - pr * ur + ps * us) / (sr - us)
        o = [rr, ur, pr, er]
        for cond, val in ((sr > 0, [rsr, us, ps, esr]), (us > 0, [rsl, us, ps, esl]),
                          (sl > 0, [rl, ul, pl, el])):
            o = [torch.where(cond, x, y) for x, y in zip(val, o)]
        ro, uo, pt, e = o
        f0 = ro * uo
        return [f0, (e + pt) * uo, ro * uo * uo + pt] + \
            [f0 * torch.where(f0 > 0, l[k], r[k]) for k in range(3, nv)]

    def cons(q):
        U = [q[0], q[1] / (g - 1) + 0.5 * q[0] * sum(q[k] ** 2 for k in range(2, nv))]
        U += [q[0] * q[k] for k in range(2, nv)]
        return U, [U[2], q[2] * (U[1] + q[1]), q[1] + U[2] * q[2]] + \
            [U[2] * q[k] for k in range(3, nv)]

    UL, FL = cons(l)
    UR, FR = cons(r)
    if solver == "hll":
        sl, sr = (torch.minimum(ul, ur) - cm).clamp_max(0), (torch.maximum(ul, ur) + cm).clamp_min(0)
        return [(sr * a - sl * b + sr * sl * (y - x)) / (sr - sl)
                for a, b, x, y in zip(FL, FR, UL, UR)]
    s = torch.maximum(ul.abs() + cl, ur.abs() + cr)
    return [0.5 * (a + b - s * (y - x)) for a, b, x, y in zip(FL, FR, UL, UR)]


def _hydro_step(U, p, solver):
    dim, gw, nv, g = p.dim, 2, p.dim + 2, p.gamma0
    _fill_ghosts(U, dim, gw, list(p.bc), (2,))
    dx = (p.dx, p.dy, p.dz)
    r = U[0].clamp_min(p.smallr)
    vel = [U[2 + d] / r for d in range(dim)]
    e = U[1] / r - 0.5 * sum(x * x for x in vel)
    pr = torch.maximum((g - 1) * r * e, r * (p.smallc ** 2 / g))
    q = [r, pr] + vel
    cs = torch.sqrt(g * pr / r)
    dt = p.cfl / _inner(sum((cs + vel[d].abs()) / dx[d] for d in range(dim)), dim, gw).amax()
    D = [[_slope(p.slope_type, f, _sh(f, d, 1), _sh(f, d, -1)) for f in q] for d in range(dim)]
    div = sum(D[d][2 + d] for d in range(dim))
    adv = [sum(vel[d] * D[d][k] for d in range(dim)) for k in range(nv)]
    src = [-adv[0] - div * r, -adv[1] - div * g * pr] + \
        [-adv[2 + d] - D[d][1] / r for d in range(dim)]
    new = [x.clone() for x in U]
    for d in range(dim):
        h = dt / dx[d]

        def rot(s):
            s = list(s)
            s[2], s[2 + d] = s[2 + d], s[2]
            return s

        def state(sign):
            s = [q[k] + 0.5 * sign * D[d][k] + 0.5 * src[k] * h for k in range(nv)]
            s[0] = s[0].clamp_min(p.smallr)
            return s

        F = rot(_hydro_flux(rot([_sh(x, d, -1) for x in state(1)]), rot(state(-1)), p, nv, solver))
        for k in range(nv):
            new[k] = new[k] + (F[k] - _sh(F[k], d, 1)) * h
    for k in range(nv):
        _inner(U[k], dim, gw).copy_(_inner(new[k], dim, gw))
    return float(dt)


def _net(P):
    P = torch.from_numpy(np.asarray(P, dtype=np.float64)).cuda()
    n = {"W1": P[S.W1:S.B1].view(128, 16), "b1": P[S.B1:S.W2], "W2": P[S.W2:S.B2].view(128, 128),
         "b2": P[S.B2:S.W3], "W3": P[S.W3:S.B3].view(8, 128), "b3": P[S.B3:S.N_TRAINED]}
    for k, lo, hi in (("mu_in", S.MU_IN, S.ISIG_IN), ("isig_in", S.ISIG_IN, S.MU_OUT),
                      ("mu_out", S.MU_OUT, S.SIG_OUT), ("sig_out", S.SIG_OUT, S.N_PARAMS)):
        n[k] = P[lo:hi]
    return n


def _mlp(n, X):
    xs = (X - n["mu_in"]) * n["isig_in"]
    h1 = torch.relu(xs @ n["W1"].T + n["b1"])
    h2 = torch.relu(h1 @ n["W2"].T + n["b2"])
    return h2 @ n["W3"].T + n["b3"], (xs, h1, h2)


def _mlp_grad(n, X, T):
    y, (xs, h1, h2) = _mlp(n, X)
    dy = 2 * (y - (T - n["mu_out"]) / n["sig_out"]) / y.numel()
    d2 = (dy @ n["W3"]) * (h2 > 0)
    d1 = (d2 @ n["W2"]) * (h1 > 0)
    return torch.cat([(d1.T @ xs).reshape(-1), d1.sum(0), (d2.T @ h1).reshape(-1), d2.sum(0),
                      (dy.T @ h2).reshape(-1), dy.sum(0)])


def _minibatch(seed, step, batch, n):
    """The sample indexes of a training step: SplitMix64's output function of a counter."""
    with np.errstate(over="ignore"):
        i = np.arange(batch, dtype=np.uint64)
        z = np.uint64(seed) + np.uint64(0x9E3779B97F4A7C15) * (np.uint64(step * 0x10001 + 1) + i)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        return ((z ^ (z >> np.uint64(31))) % np.uint64(n)).astype(np.int64)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("train", "gradient", "infer"):
        P = _net_params(seed, False)
        X, T = (torch.from_numpy(x).cuda().double() for x in _samples(case["samples"], seed))
        if kind == "infer":
            return _mlp(_net(P), X)[0].cpu().numpy()
        if kind == "gradient":
            return _mlp_grad(_net(P), X, T).cpu().numpy()
        n = _net(P)
        flat = torch.cat([n[k].reshape(-1) for k in ("W1", "b1", "W2", "b2", "W3", "b3")])
        m, v = torch.zeros_like(flat), torch.zeros_like(flat)
        rest = torch.from_numpy(P[S.N_TRAINED:].astype(np.float64)).cuda()
        for s in range(case["steps"]):
            i = torch.from_numpy(_minibatch(seed & 0xFFFF, s, case["batch"], case["samples"])).cuda()
            gr = _mlp_grad(_net(torch.cat([flat, rest]).cpu().numpy()), X[i], T[i])
            m, v = 0.9 * m + 0.1 * gr, 0.999 * v + 0.001 * gr * gr
            flat = flat - 1e-3 * (m / (1 - 0.9 ** (s + 1))) / \
                (torch.sqrt(v / (1 - 0.999 ** (s + 1))) + 1e-8)
        return torch.cat([flat, rest]).cpu().numpy()
    if kind == "batch":
        members = _batch_members(case, seed)
        flux = {"hlld": _hlld, "hll": _hll, "llf": lambda l, r, g: _llf(l, r, g)[0]}[case["riemann"]]
        groups = {}
        for k, (p, _, _) in enumerate(members):
            groups.setdefault((p.nx, p.ny, p.nz), []).append(k)
        if len(groups) * case["steps"] > 700 and case["dim"] == 3:
            return None
        out = [None] * len(members)
        for ks in groups.values():
            p = members[ks[0]][0]
            tail = (1,) * p.dim
            g = torch.tensor([members[k][0].gamma0 for k in ks], dtype=torch.float64,
                             device="cuda").view((-1,) + tail)
            U = torch.stack([_initial(*members[k], "cuda") for k in ks])
            if p.dim == 2:
                U = U[:, :, 0]
            U = [x.contiguous() for x in U.unbind(1)]
            for _ in range(case["steps"]):
                _mhd_step(U, p, g, (p.dx, p.dy, p.dz), flux)
            U = torch.stack(U, 1).cpu().numpy()
            for n, k in enumerate(ks):
                out[k] = U[n].reshape(p.shape)
        return out
    p = _params(case)
    U = _initial(p, case["problem"], seed, "cuda")
    U = [(x if p.dim == 3 else x[0]).contiguous() for x in U]
    net = _net(_net_params(seed, True)) if kind == "surrogate" else None
    t = 0.0
    for _ in range(case["steps"]):
        if kind == "hydro":
            t += _hydro_step(U, p, case["riemann"])
            continue
        if net is not None:
            flux = lambda l, r, g: _surrogate_flux(l, r, g, net)  # noqa: E731
        else:
            flux = {"hlld": _hlld, "hll": _hll,
                    "llf": lambda l, r, g: _llf(l, r, g)[0]}[case["riemann"]]
        t += float(_mhd_step(U, p, p.gamma0, (p.dx, p.dy, p.dz), flux))
    return {"t": t, "U": torch.stack(U).view(p.shape)}
