"""The work that this framework is timed on: each of its public paths at the
sizes, meshes, precisions and solvers its users run.

A case names a kind of call (`kind`), the mesh it runs on (`mesh`, `n` quads
per direction or `nx` x `ny`) and the options that change the path.  The plan
of a case is what a user's program builds once and keeps: the mesh, its
variational-reconstruction setup and the device context.  The inputs are made
from the seed: cell means with their reconstruction, or training rows.

`run` makes one pass through the host classes of `dnds_amd.host` and then
waits for the device as a program does before it looks at a result
(`Device.sync`, which also reports a failed state).  Arrays stay on the
device: `Outputs` reads one back in the reference's host layout when it is
asked for it.
"""
from __future__ import annotations

import functools
import math
import os

import numpy as np
import torch

from dnds_amd import _capi as A
from dnds_amd import cases as workloads
from dnds_amd.host import (RIEMANN_VR_SETTING, CompactFacedMeshSerialRW, EulerEvaluator, ExplicitSSPRK3LocalDt,
                           ImplicitEulerDualTimeStep, ImplicitSDIRK4DualTimeStep, VRFiniteVolume2D, WarmStart,
                           vr_setting)

GAMMA = workloads.GAMMA
CFL = 0.5
SWEEPS = 5  # reconstruction sweeps per stage, as in the benchmark
THREADS = min(16, len(os.sched_getaffinity(0)))  # of the host setup
N_IN, N_OUT = 58, 36  # the warm-start network's features and outputs


def listed() -> list[dict]:
    return [
        # the 40 x 40 isentropic vortex, the smallest documented run: every
        # launch is a few workgroups, so latency and launches are all of it
        {"name": "vortex_step_3k", "kind": "step", "mesh": "vortex", "n": 40, "mixed": False, "limiter": 0},
        # a four-quadrant Riemann step at an ordinary size, WBAP V2 limiter
        {"name": "riemann_step_33k", "kind": "step", "mesh": "riemann", "n": 128, "mixed": False, "limiter": 2},
        # the benchmark's Mach-3 shock on a mixed tri/quad mesh, wall and
        # inflow boundaries, WBAP V2: the production step, larger than any cache
        {"name": "mach3_step_1m", "kind": "step", "mesh": "mach3", "n": 819, "mixed": False, "limiter": 2},
        # the mixed-precision arm (FP32 correction sweeps and face values)
        {"name": "vortex_mixed_step_264k", "kind": "step", "mesh": "vortex", "n": 363, "mixed": True, "limiter": 0},
        # reconstruction of a new state to a tolerance (start of a run, and
        # the harvest of training pairs), Jacobi sweeps with their increments
        {"name": "reconstruct_66k", "kind": "reconstruct", "mesh": "vortex", "n": 181, "sweeps": 20},
        # the in-place sweep that the reference's Riemann configuration sets
        {"name": "sor_sweeps_131k", "kind": "sweeps", "mesh": "riemann", "n": 256, "sor": True, "sweeps": 4},
        # sweeps called one by one by a program that drives them itself
        {"name": "jacobi_sweeps_525k", "kind": "sweeps", "mesh": "riemann", "n": 512, "sor": False, "sweeps": 5},
        # time step and right-hand side of the laminar Navier-Stokes model
        {"name": "viscous_rhs_262k", "kind": "rhs", "mesh": "riemann", "n": 362, "viscous": True, "riemann": "HLLC"},
        # the limiter by itself, V3, on the mixed mesh
        {"name": "wbap_v3_135k", "kind": "limiter", "mesh": "mach3", "n": 300, "procedure": 3},
        # steady laminar flat plate: implicit Euler iterations with LU-SGS
        {"name": "plate_lusgs_31k", "kind": "implicit", "mesh": "plate", "nx": 385, "ny": 79, "order": 3,
         "scheme": "euler", "gmres": 0, "iterations": 10},
        # bump in a channel with GMRES preconditioned by LU-SGS: many short
        # kernels and reductions on a small mesh
        {"name": "bump_gmres_2k", "kind": "implicit", "mesh": "bump", "nx": 48, "ny": 16, "order": 3,
         "scheme": "euler", "gmres": 1, "iterations": 4},
        # the learned warm start: one epoch of training in batches of 4096
        {"name": "warmstart_train_66k", "kind": "train", "rows": 65536, "batch": 4096},
    ]


def _size(rng, lo: int, hi: int) -> int:
    """lo..hi, spread over the logarithm"""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["step", "step", "step", "reconstruct", "sweeps", "rhs", "limiter", "implicit", "warmstart"])
    if kind == "step":
        mesh = rng.choice(["vortex", "riemann", "mach3"])
        limiter = 0 if mesh == "vortex" else rng.choice([2, 2, 3])
        return {"kind": "step", "mesh": mesh, "n": _size(rng, 24, 420), "mixed": rng.random() < 0.4,
                "limiter": limiter}
    if kind == "reconstruct":
        return {"kind": "reconstruct", "mesh": "vortex", "n": _size(rng, 24, 300), "sweeps": rng.randint(5, 25)}
    if kind == "sweeps":
        return {"kind": "sweeps", "mesh": rng.choice(["riemann", "mach3", "vortex"]), "n": _size(rng, 24, 400),
                "sor": rng.random() < 0.5, "sweeps": rng.randint(1, 6)}
    if kind == "rhs":
        mesh = rng.choice(["riemann", "mach3", "vortex"])
        return {"kind": "rhs", "mesh": mesh, "n": _size(rng, 24, 400), "viscous": rng.random() < 0.5,
                "riemann": rng.choice(["Roe", "HLLC", "HLLEP"])}
    if kind == "limiter":
        return {"kind": "limiter", "mesh": rng.choice(["riemann", "mach3"]), "n": _size(rng, 24, 350),
                "procedure": rng.choice([2, 3])}
    if kind == "implicit":
        mesh = rng.choice(["plate", "bump"])
        nx = _size(rng, 24, 420)
        return {"kind": "implicit", "mesh": mesh, "nx": nx, "ny": max(8, nx // rng.randint(2, 5)),
                "order": rng.choice([1, 3]) if mesh == "plate" else 3,
                "scheme": rng.choice(["euler", "sdirk4"]) if mesh == "bump" else "euler",
                "gmres": rng.choice([0, 0, 1, 2]) if mesh == "bump" else 0, "iterations": rng.randint(2, 8)}
    if rng.random() < 0.5:
        return {"kind": "predict", "mesh": "vortex", "n": _size(rng, 24, 400)}
    batch = rng.choice([1000, 2048, 4096, 8192])
    return {"kind": "train", "rows": batch * rng.randint(2, 12) + rng.randint(0, batch - 1), "batch": batch}


# ------------------------------------------------------------------ plans ----

class Plan:
    """Mesh, setup and evaluator of a case, kept by the program."""

    def __init__(self, mesh, vfv, far, base, riemann="HLLC", gas=None):
        self.mesh, self.vfv, self.base = mesh, vfv, base
        self.ev = EulerEvaluator(mesh, vfv, riemannSolverType=riemann, farFieldStaticValue=far, **(gas or {}))


def _riemann_mesh(n: int, limiter: bool, sor: bool):
    bc = A.BC_SPECIAL_2DRIEMANNFAR
    mesh = CompactFacedMeshSerialRW.generate(A.MESH_TRI_SPLIT, n, n, 0.0, 1.0, 0.0, 1.0, jitter=0.2, seed=2,
                                             bc=(bc, bc, bc, bc))
    vfv = VRFiniteVolume2D(mesh, vr_setting(**RIEMANN_VR_SETTING, build_limiter_data=int(limiter),
                                            sor_instead=int(sor)))
    vfv.Initialization(THREADS)
    bary = vfv.arrays(["cell_bary"])["cell_bary"].reshape(-1, 2)
    return mesh, vfv, workloads.RIEMANN_FAR, workloads.riemann_state(bary)


def _mach3_mesh(n: int, limiter: bool, sor: bool):
    bcs = (A.BC_FARFIELD, A.BC_WALL_EULER, A.BC_WALL_EULER, A.BC_WALL_EULER)
    mesh = CompactFacedMeshSerialRW.generate(A.MESH_MIXED, n, n, 0.0, 4.0, 0.0, 1.0, jitter=0.15, seed=5, bc=bcs)
    vfv = VRFiniteVolume2D(mesh, vr_setting(**dict(RIEMANN_VR_SETTING, far_weight=1.0),
                                            build_limiter_data=int(limiter), sor_instead=int(sor)))
    vfv.Initialization(THREADS)
    bary = vfv.arrays(["cell_bary"])["cell_bary"].reshape(-1, 2)
    prim = np.where((bary[:, 0] < 0.5)[:, None], np.array(workloads.MACH3_LEFT), np.array(workloads.MACH3_RIGHT))
    far = tuple(_conservative(*(np.array(v) for v in workloads.MACH3_LEFT)).tolist())
    return mesh, vfv, far, _conservative(*prim.T)


def _vortex_mesh(n: int, limiter: bool, sor: bool):
    mesh = CompactFacedMeshSerialRW.generate(A.MESH_TRI_SPLIT, n, n, 0.0, 10.0, 0.0, 10.0, periodic=(True, True),
                                             jitter=0.0, seed=1)
    vfv = VRFiniteVolume2D(mesh, vr_setting(**RIEMANN_VR_SETTING, build_limiter_data=int(limiter),
                                            sor_instead=int(sor)))
    vfv.Initialization(THREADS)
    return mesh, vfv, (1.0, 1.0, 1.0, 3.5), None


@functools.lru_cache(maxsize=2)
def _plan(mesh: str, n, nx, ny, order, limiter: bool, sor: bool, riemann: str, viscous: bool) -> Plan:
    if mesh == "plate":
        c = workloads.flat_plate(nx, ny, reynolds=1e5, rec_order=order, nthreads=THREADS)
        return Plan(c.mesh, c.vfv, c.far, c.u0, c.riemann, c.gas)
    if mesh == "bump":
        c = workloads.bump_channel(nx, ny, nthreads=THREADS)
        return Plan(c.mesh, c.vfv, c.far, c.u0, c.riemann)
    make = {"riemann": _riemann_mesh, "mach3": _mach3_mesh, "vortex": _vortex_mesh}[mesh]
    m, vfv, far, base = make(n, limiter, sor)
    gas = dict(muGas=1e-3, prGas=0.72, TRef=1.0, CSutherland=0.5) if viscous else None
    return Plan(m, vfv, far, base, riemann, gas)


def _plan_of(case: dict) -> Plan:
    mesh = case.get("mesh", "vortex")
    riemann = case.get("riemann", "Roe" if mesh == "vortex" else "HLLC")
    limiter = case["kind"] == "limiter" or bool(case.get("limiter", 0))
    return _plan(mesh, case.get("n", 16), case.get("nx"), case.get("ny"), case.get("order"), limiter,
                 bool(case.get("sor", False)), riemann, bool(case.get("viscous", False)))


# ----------------------------------------------------------------- inputs ----

def _conservative(rho, u, v, p):
    return np.stack([rho, rho * u, rho * v, p / (GAMMA - 1) + 0.5 * rho * (u * u + v * v)], axis=-1)


def _means(case: dict, plan: Plan, seed: int) -> np.ndarray:
    """Cell means: the workload's state with seeded density noise at its
    velocity and pressure; the vortex at a seeded time of its travel."""
    rng = np.random.default_rng(seed)
    if plan.base is None:
        t = rng.uniform(0.0, 10.0)
        vol = plan.vfv.arrays(["volume"])["volume"]
        return workloads.cell_means(plan.mesh, vol, lambda x, y: workloads.vortex_exact(x, y, t))
    u = plan.base.copy()
    e = 1e-3 * rng.uniform(-1.0, 1.0, u.shape[0])
    kinetic = 0.5 * (u[:, 1] ** 2 + u[:, 2] ** 2) / u[:, 0]
    u[:, :3] *= (1.0 + e)[:, None]
    u[:, 3] += e * kinetic
    return u


def _training_rows(rows: int, seed: int):
    """Features as the network meets them (scaled differences in [-1, 1],
    moments, a log size) and targets of their order: a fixed linear map of
    the differences plus a small remainder."""
    rng = np.random.default_rng(seed)
    X = rng.uniform(-1.0, 1.0, (rows, N_IN)).astype(np.float32)
    X[:, 48:57] *= 0.2
    X[:, 57] = -3.0 + 0.1 * X[:, 57]
    W = np.random.default_rng(7).standard_normal((48, N_OUT)).astype(np.float32) * np.float32(0.1)
    T = X[:, :48] @ W + np.float32(0.01) * rng.standard_normal((rows, N_OUT)).astype(np.float32)
    return X, np.ascontiguousarray(T, dtype=np.float32)


def _network_parameters(seed: int, n_param: int) -> np.ndarray:
    return (np.random.default_rng(seed).standard_normal(n_param) * 0.1).astype(np.float32)


class Outputs(dict):
    """A pass's results; indexing reads a device array back to the host."""

    def __getitem__(self, key):
        v = dict.__getitem__(self, key)
        return v.download() if hasattr(v, "download") else v


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    plan = _plan_of(case)
    ev, vfv = plan.ev, plan.vfv
    s = {"case": case, "plan": plan}
    if kind == "train":
        X, T = _training_rows(case["rows"], seed)
        ws = WarmStart(ev, seed=seed, capacity=case["rows"])
        ws.add_rows(X, T)
        s.update(ws=ws, p0=ws.get_params())
        return s
    u0 = _means(case, plan, seed)
    s["u"] = ev.BuildMean().upload(u0)
    if kind == "predict":
        ws = WarmStart(ev, seed=seed)
        ws.set_params(_network_parameters(seed, ws.n_param))
        s.update(ws=ws, uRec=vfv.BuildRec())
        ev.device.sync()
        return s
    s["uRec"], s["uRecNew"] = vfv.BuildRec().setConstant(0.0), vfv.BuildRec()
    if kind != "reconstruct":
        # the reconstruction a running program holds: a few sweeps on the means
        for _ in range(4):
            vfv.ReconstructionJacobiStep(s["u"], s["uRec"], s["uRecNew"], 0.0)
    if kind in ("step", "implicit"):
        s["u_start"] = ev.BuildMean().copy_from(s["u"])
        s["uRec_start"] = vfv.BuildRec().copy_from(s["uRec"])
    if kind == "step":
        s["ode"] = ExplicitSSPRK3LocalDt(ev, nInternalRecStep=SWEEPS, CFL=CFL, useLimiter=case["limiter"] > 0,
                                         mixedPrecision=case["mixed"],
                                         limiterProcedure=1 if case["limiter"] == 3 else 0)
    elif kind == "rhs":
        s.update(dt=ev.BuildScalar(), rhs=ev.BuildMean())
    elif kind == "limiter":
        s.update(ind=ev.BuildScalar(), uRecLim=vfv.BuildRec())
    elif kind == "implicit":
        steady = case["mesh"] == "plate"
        scheme = ImplicitSDIRK4DualTimeStep if case["scheme"] == "sdirk4" else ImplicitEulerDualTimeStep
        s["ode"] = scheme(ev, nInternalRecStep=1, CFL=20.0 if steady else 10.0,
                          nTimeStepInternal=case["iterations"], rhsThresholdInternal=0.0)
        s["dt"] = 1e100 if steady else 0.2
    ev.device.sync()
    return s


# ------------------------------------------------------------------- pass ----

def run(s: dict) -> dict:
    case, ev, vfv = s["case"], s["plan"].ev, s["plan"].vfv
    kind = case["kind"]
    if kind == "train":
        s["ws"].set_params(s["p0"])
        loss = s["ws"].train(1, batch=case["batch"])
        return {"loss": float(loss[-1]), "params": s["ws"].get_params()}
    u, r, rn = s["u"], s["uRec"], s.get("uRecNew")
    if kind == "predict":
        s["ws"].predict(u, r)
        out = Outputs(uRec=r)
    elif kind == "step":
        # every pass is the step from the prepared state
        u.copy_from(s["u_start"])
        r.copy_from(s["uRec_start"])
        out = Outputs(dt=s["ode"].Step(u, r, rn, 0.0), u=u, uRec=r)
    elif kind == "reconstruct":
        r.setConstant(0.0)
        sweeps, increment = vfv.ReconstructToTolerance(u, r, rn, 1e-20, case["sweeps"])
        out = Outputs(uRec=r, sweeps=sweeps, increment=increment)
    elif kind == "sweeps":
        for _ in range(case["sweeps"]):
            vfv.ReconstructionJacobiStep(u, r, rn, 0.0)
        out = Outputs(uRec=r)
    elif kind == "rhs":
        dtmin = ev.EvaluateDt(s["dt"], u, CFL, 1e100, True)
        ev.EvaluateRHS(s["rhs"], u, r, 0.0)
        out = Outputs(dtMin=dtmin, dt=s["dt"], rhs=s["rhs"])
    elif kind == "limiter":
        limit = vfv.ReconstructionWBAPLimitFacialV3 if case["procedure"] == 3 else vfv.ReconstructionWBAPLimitFacialV2
        limit(u, r, s["uRecLim"], None, s["ind"])
        out = Outputs(uRec=s["uRecLim"], indicator=s["ind"])
    else:
        u.copy_from(s["u_start"])
        r.copy_from(s["uRec_start"])
        ev.SetLinearSolver(case["gmres"], 10, 2)
        h = s["ode"].Step(u, r, rn, s["dt"])
        out = Outputs(u=u, uRec=r, increments=h[1] if case["scheme"] == "sdirk4" else h)
    ev.device.sync()
    return out


# ------------------------------------------------------------------- work ----

def _counts(case: dict):
    """(cells, faces, cell-face pairs) of a case's mesh"""
    mesh = case["mesh"]
    if mesh in ("plate", "bump"):
        quads = case["nx"] * case["ny"]
        return (quads, 2 * quads, 4 * quads) if mesh == "plate" else (2 * quads, 3 * quads, 6 * quads)
    quads = case["n"] ** 2
    return (1.5 * quads, 2.5 * quads, 5 * quads) if mesh == "mach3" else (2 * quads, 3 * quads, 6 * quads)


def _sweep(nc, pairs, real=8):
    """A^-1 B and A^-1 b of each cell-face pair, its neighbour, the
    coefficients in and out, the means; a multiply and an add per entry and
    variable"""
    return pairs * (90 * real + 4) + nc * (2 * 36 * real + 32), pairs * (2 * 81 * 4 + 3 * 36)


def _rhs(nc, nf, viscous):
    """face: cells, point coordinates of both sides, a normal; cell: moments,
    coefficients, means, volume, result; three points of two
    reconstructions and a flux"""
    return (nf * (8 + 96 + 16) + nc * (288 + 72 + 32 + 8 + 32),
            nf * 3 * (2 * 9 * (3 + 8) + 250 + (2 * 18 * 8 + 150 if viscous else 0)))


def _dt(nc, nf):
    return nf * (8 + 16 + 16 + 8) + nc * (32 + 8 + 8), nf * 60


def _limiter(nc, nf, copied):
    """indicator only (limited cells are few): point 0 of both sides, weights,
    normal, cells; rho and E coefficients, moments, scales; where it copies,
    the other coefficients in and out"""
    return nf * (32 + 80 + 16 + 8) + nc * (144 + 72 + 16 + 16 + 8 + (288 + 144 if copied else 0)), nf * 1500


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "train":
        rows = case["rows"] // case["batch"] * case["batch"]
        weights = N_IN * 128 + 128 * 128 + 128 * N_OUT
        steps = rows // case["batch"]
        return {"bytes": rows * 4 * (N_IN + N_OUT) + steps * weights * 4 * 6, "flops": rows * (6 * weights - 2 * N_IN * 128)}
    nc, nf, pairs = _counts(case)
    if kind == "predict":
        weights = N_IN * 128 + 128 * 128 + 128 * N_OUT
        return {"bytes": nc * (32 + 12 * 4 + 40 + 288) + weights * 4, "flops": nc * 2 * weights}
    parts = []
    if kind == "reconstruct" or kind == "sweeps":
        parts = [_sweep(nc, pairs)] * case["sweeps"]
    elif kind == "rhs":
        parts = [_dt(nc, nf), _rhs(nc, nf, case["viscous"])]
    elif kind == "limiter":
        parts = [_limiter(nc, nf, True)]
    elif kind == "step":
        parts = [_dt(nc, nf)] + 3 * [_rhs(nc, nf, False), (nc * 96, nc * 24)]
        parts += 3 * ([_sweep(nc, pairs)] + (SWEEPS - 1) * [_sweep(nc, pairs, 4 if case["mixed"] else 8)])
        if case["limiter"]:
            parts += 3 * [_limiter(nc, nf, False)]
    else:
        lusgs = (2 * (nc * (4 + 8 + 8 + 64) + pairs * 4 + pairs / 2 * 100), pairs * 60)
        one = [_dt(nc, nf), _sweep(nc, pairs), _rhs(nc, nf, case["mesh"] == "plate"), lusgs, (nc * 160, nc * 32)]
        if case["gmres"]:
            # per restart 10 vectors: product, both sweeps, projections on the
            # vectors so far, update
            vec = nc * 32
            one += 2 * ([(nc * 84 + pairs * 108, pairs * 70), lusgs] * 11 + [(vec * (2 * 55 + 4 * 10), nc * 4 * 4 * 55)])
        parts = one * case["iterations"] * (3 if case["scheme"] == "sdirk4" else 1)
    return {"bytes": float(sum(p[0] for p in parts)), "flops": float(sum(p[1] for p in parts))}


# ---------------------------------------------- values in 64 bits, by torch ----

class _Exact:
    """The sweeps on a mesh of triangles without walls and, on a periodic
    one, the time step and the Roe right-hand side, in plain torch.  The mesh and
    the matrices of the reconstruction are inputs, as they are for `run`."""

    def __init__(self, plan: Plan):
        m, v = plan.mesh.arrays(), plan.vfv.arrays(["volume", "face_area", "face_norm", "face_norm_center", "face_d0",
                                                   "ainv_b", "ainv_bvec"])
        t = torch.from_numpy
        self.nc, self.nf = m["n_cell"], m["n_face"]
        self.lr = t(m["face2cell"].copy())
        slot = t(m["cell2face"].copy()).reshape(self.nc, 3)
        ends, own = self.lr[slot], torch.arange(self.nc)[:, None]
        # a far-field face couples a cell to itself
        self.nbr = torch.where(ends[..., 1] == A.NO_CELL, own, ends.sum(-1) - own)
        self.M = t(v["ainv_b"]).reshape(self.nc, 3, 9, 9)
        self.b = t(v["ainv_bvec"]).reshape(self.nc, 3, 9)
        self.vol, self.area = t(v["volume"]), t(v["face_area"])
        self.norm = t(v["face_norm"]).reshape(self.nf, 3, 2)
        n = t(v["face_norm_center"]).reshape(self.nf, 2)
        self.nhat = n / n.norm(dim=1, keepdim=True)
        self.d0 = t(v["face_d0"]).reshape(self.nf, 3, 2, 9)

    def sweep(self, u, x):
        """x [cell][variable][9] of the Jacobi map"""
        new = torch.zeros_like(x)
        for s in range(3):
            j = self.nbr[:, s]
            new += torch.bmm(x[j], self.M[:, s].transpose(1, 2).contiguous())
            new += (u[j] - u)[:, :, None] * self.b[:, s, None, :]
        return new

    @staticmethod
    def pressure(u):
        return (GAMMA - 1) * (u[..., 3] - 0.5 * (u[..., 1] ** 2 + u[..., 2] ** 2) / u[..., 0])

    def time_step(self, u):
        """the global minimum and the faces' jump of the wave speeds"""
        L, R = u[self.lr[:, 0]], u[self.lr[:, 1]]
        pL, pR = self.pressure(L), self.pressure(R)
        vL, vR = L[:, 1:3] / L[:, :1], R[:, 1:3] / R[:, :1]
        vn = 0.5 * ((vL + vR) * self.nhat).sum(1)
        a = torch.sqrt(GAMMA * 0.5 * (pL + pR) / (0.5 * (L[:, 0] + R[:, 0])))
        lam = torch.zeros(self.nc, dtype=u.dtype)
        for side in (0, 1):
            lam.index_add_(0, self.lr[:, side], (vn.abs() + a) * self.area)
        jump = ((vR - vL) * self.nhat).sum(1).abs()
        jump = jump + 0.7071 * torch.sqrt((GAMMA * pR / R[:, 0] - GAMMA * pL / L[:, 0]).abs())
        return float((CFL * self.vol / lam).min()), jump

    def rhs(self, u, x, jump):
        out = torch.zeros_like(u)
        for g, w in ((0, 5 / 9), (1, 8 / 9), (2, 5 / 9)):
            n = self.norm[:, g]
            length = n.norm(dim=1, keepdim=True)
            n = n / length
            state = []
            for side in (0, 1):
                c = self.lr[:, side]
                state.append(u[c] + (x[c] * self.d0[:, g, side, None, :]).sum(2))
            f = self.roe(state[0], state[1], n, jump) * length * w
            out.index_add_(0, self.lr[:, 0], -f)
            out.index_add_(0, self.lr[:, 1], f)
        return out / self.vol[:, None]

    def roe(self, UL, UR, n, jump):
        """Roe's flux through unit normals n, Harten and Yee's fix on the
        acoustic waves"""
        def turned(U, s):
            return torch.stack([U[:, 0], n[:, 0] * U[:, 1] + s * n[:, 1] * U[:, 2],
                                n[:, 0] * U[:, 2] - s * n[:, 1] * U[:, 1], U[:, 3]], 1)

        L, R = turned(UL, 1.0), turned(UR, 1.0)
        pL, pR = self.pressure(L), self.pressure(R)

        def flux(U, p):
            v = U[:, 1:2] / U[:, :1]
            z = torch.zeros_like(p)
            return U * v + torch.stack([z, p, z, p * v[:, 0]], 1)

        wL, wR = torch.sqrt(L[:, 0]), torch.sqrt(R[:, 0])

        def mean(a, b):
            return (wL * a + wR * b) / (wL + wR)

        vx, vy = mean(L[:, 1] / L[:, 0], R[:, 1] / R[:, 0]), mean(L[:, 2] / L[:, 0], R[:, 2] / R[:, 0])
        H = mean((L[:, 3] + pL) / L[:, 0], (R[:, 3] + pR) / R[:, 0])
        q = vx * vx + vy * vy
        a = torch.sqrt((GAMMA - 1) * (H - 0.5 * q))
        eps = torch.maximum(0.05 * (torch.sqrt(q) + a), jump)

        def fixed(lam):
            return torch.where(lam < eps, (lam * lam + eps * eps) / (2 * eps), lam)

        d = R - L
        s = d[:, 2] - vy * d[:, 0]
        e = (GAMMA - 1) / (a * a) * (d[:, 0] * (H - vx * vx) + vx * d[:, 1] - (d[:, 3] - s * vy))
        m = (d[:, 0] * (vx + a) - d[:, 1] - a * e) / (2 * a)
        p = d[:, 0] - m - e
        m, p = m * fixed((vx - a).abs()), p * fixed((vx + a).abs())
        e, s = e * vx.abs(), s * vx.abs()
        diss = torch.stack([m + e + p, m * (vx - a) + e * vx + p * (vx + a), vy * (m + e + p) + s,
                            m * (H - vx * a) + e * 0.5 * q + s * vy + p * (H + vx * a)], 1)
        return turned(0.5 * (flux(L, pL) + flux(R, pR) - diss), -1.0)


def exact(case: dict, seed: int):
    """The sweeps and the periodic, unlimited steps; the others have walls,
    limiters or solvers whose restatement is a program of its own."""
    kind, mesh = case["kind"], case.get("mesh")
    if not (kind in ("step", "reconstruct") and mesh == "vortex" or
            kind == "sweeps" and mesh in ("vortex", "riemann") and not case["sor"]):
        return None
    if kind == "step" and case["n"] > 380:
        return None  # over 20 seconds
    plan = _plan_of(case)
    ex = _Exact(plan)
    u = torch.from_numpy(_means(case, plan, seed))
    x = torch.zeros(ex.nc, 4, 9, dtype=torch.float64)
    if kind == "reconstruct":
        for _ in range(case["sweeps"]):
            new = ex.sweep(u, x)
            inc = float(((new - x) ** 2).sum() / ex.nc)
            x = new
        return {"uRec": x.reshape(ex.nc, 36).numpy(), "sweeps": None, "increment": inc}
    for _ in range(4):
        x = ex.sweep(u, x)
    if kind == "sweeps":
        for _ in range(case["sweeps"]):
            x = ex.sweep(u, x)
        return {"uRec": x.reshape(ex.nc, 36).numpy()}
    dt, jump = ex.time_step(u)
    last = u
    for c in (1.0, 0.25, 2.0 / 3.0):
        for _ in range(SWEEPS):
            x = ex.sweep(u, x)
        u = (1 - c) * last + c * (u + dt * ex.rhs(u, x, jump))
    return {"dt": dt, "u": u.numpy(), "uRec": x.reshape(ex.nc, 36).numpy()}
