"""Workloads that stand for what a program does with the MPFA-O Richards path.

A program lays out one context per problem (mesh, boundary types, materials:
``MPFAO``) and then either drives its own nonlinear solver through the
callbacks (residual, Jacobian), or hands whole time steps to the device
solver, and reads diagnostics and velocities back.  Meshes are the jittered
boxes and extruded Delaunay prisms of ``tdycore_amd.workloads``; the mesh of
a size is fixed, permeability, porosity and the state come from the seed.

Kinds of case (``kind``):
  residual   one TS residual (what a line search or a matrix-free solver calls)
  callbacks  residual and Jacobian, as a Newton iteration calls them
             (``form`` "ts": IFunction + IJacobian, "snes": SNESFunction + SNESJacobian)
  recover    Diagnostics and RecoverVelocity at an output time
  step       one implicit time step on the device (``driver`` "snes", "ts" or "tdyti"),
             FP64 or FP32 Krylov, with or without the coarse correction

``exact`` is the same mathematics in plain numpy, FP64, from the mesh and the
materials: one local system per vertex solved directly, fluxes, Jacobian, and
for small problems the time step by Newton with dense solves.
"""
import functools
import math

import numpy as np
import torch

from tdycore_amd import meshgen as mg
from tdycore_amd import workloads
from tdycore_amd.mpfao import MPFAO

PREF, GRAVITY, VISCOSITY = 101325.0, 9.8068, 9.94e-4
VG_M, VG_ALPHA = 1.0 / 3.0, 1e-4
POLY = (0.995, 0.99, 1.0, 0.005)
DAY, HOUR = 86400.0, 3600.0
EXACT_CELLS = 210_000     # numpy takes about 20 s beyond this
EXACT_STEP_CELLS = 4_500  # time steps: dense Newton


def listed():
    return [
        # the smallest call: one residual of a cache-resident problem, launches and latency count
        dict(name="residual_4k", kind="residual", mesh="cube", nx=16, ny=16, nz=16, density="constant"),
        # one residual of the benchmark's 1M-cell layered box: HBM-bound
        dict(name="residual_1m", kind="residual", mesh="layered", nx=128, ny=128, nz=64, density="constant"),
        # one Newton iteration's callbacks of a mid-size problem, odd sizes, compressible water
        dict(name="snes_callbacks_95k", kind="callbacks", form="snes", mesh="cube", nx=61, ny=47, nz=33,
             density="exponential"),
        # the callbacks PETSc's TS makes per Newton iteration at 1M cells
        dict(name="ts_callbacks_1m", kind="callbacks", form="ts", mesh="layered", nx=128, ny=128, nz=64,
             density="constant"),
        # the same on an extruded Delaunay mesh: regions and rows of uneven size
        dict(name="prism_callbacks_200k", kind="callbacks", form="ts", mesh="prism", tri=10_000, layers=20,
             density="constant"),
        # output time: saturation, masses and face velocities
        dict(name="recover_442k", kind="recover", mesh="layered", nx=96, ny=96, nz=48, density="exponential"),
        # a step of the smallest configuration: many short dependent launches
        dict(name="step_4k", kind="step", driver="snes", mesh="cube", nx=16, ny=16, nz=16, density="constant",
             fp32=False, coarse=True, block=64),
        # one request of a serving ensemble, advanced by the time integrator
        dict(name="step_request_63k", kind="step", driver="tdyti", mesh="cube", nx=56, ny=40, nz=28,
             density="constant", fp32=False, coarse=True, block=256),
        # TS backward Euler with PETSc's default preconditioner (one-level block Jacobi)
        dict(name="step_ts_onelevel_46k", kind="step", driver="ts", mesh="layered", nx=48, ny=40, nz=24,
             density="constant", fp32=False, coarse=False, block=256),
        # the FP32 Krylov form
        dict(name="step_fp32_442k", kind="step", driver="snes", mesh="layered", nx=96, ny=96, nz=48,
             density="constant", fp32=True, coarse=True, block=256),
        # the benchmark's step: 1M cells in FP64
        dict(name="step_1m", kind="step", driver="snes", mesh="layered", nx=128, ny=128, nz=64, density="constant",
             fp32=False, coarse=True, block=256),
        # infiltration into an extruded Delaunay mesh, vertical-column blocks
        dict(name="step_prism_100k", kind="step", driver="snes", mesh="prism", tri=5_000, layers=20,
             density="constant", fp32=False, coarse=False, block=64),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case: any kind, sizes spread over their logarithm from a few
    thousand cells to about half a million, odd and ragged sizes included."""
    kind = rng.choice(["residual", "callbacks", "callbacks", "recover", "step", "step", "step"])
    case = dict(kind=kind, mesh=rng.choice(["cube", "layered", "prism"]))
    if kind == "callbacks":
        case["form"] = rng.choice(["ts", "snes"])
    if case["mesh"] == "prism":
        case["layers"] = rng.randint(4, 24)
        case["tri"] = _log_int(rng, 400, 200_000 // case["layers"])
    else:
        cells = _log_int(rng, 2_500, 450_000)
        ax, ay = rng.uniform(0.7, 1.4), rng.uniform(0.7, 1.4)
        s = (2.0 * cells / (ax * ay)) ** (1.0 / 3.0)  # about twice as wide as high
        case["nx"], case["ny"] = max(8, round(s * ax)), max(8, round(s * ay))
        case["nz"] = max(6, round(cells / (case["nx"] * case["ny"])))
    case["density"] = rng.choice(["constant", "exponential"])
    if kind == "step":
        case["driver"] = rng.choice(["snes", "tdyti"] if case["mesh"] == "prism" else ["snes", "ts", "tdyti"])
        case["fp32"] = rng.random() < 0.4
        case["coarse"] = case["mesh"] != "prism" and rng.random() < 0.7
        case["block"] = 64 if case["mesh"] == "prism" or rng.random() < 0.25 else 256
    return case


# ---------------------------------------------------------------- problems

MESH_SEED = 20261203


@functools.lru_cache(maxsize=2)
def _box_mesh(mesh, nx, ny, nz):
    upper = (1.0, 1.0, 1.0) if mesh == "cube" else (1000.0, 1000.0, 100.0)
    m = mg.box_mesh(nx, ny, nz, upper=upper, jitter=0.1, seed=MESH_SEED)
    zt = 0.5 * upper[2]
    fbc = m.face_bc(dirichlet=["z-", "z+"], neumann=["x-", "x+", "y-", "y+"])
    pb = mg.boundary_values(m, lambda x: mg.hydrostatic_pressure(x[:, 2], zt))
    return m, fbc, pb, mg.hydrostatic_pressure(m.cell_cen[:, 2], zt)


@functools.lru_cache(maxsize=2)
def _prism_mesh(tri, layers, block_tris):
    P = workloads.prism_problem(n_tri=tri, nlayers=layers, seed=MESH_SEED, length=50.0 * math.sqrt(tri), lattice=64,
                                infiltration=True, block_tris=block_tris)
    return P["mesh"], P["face_bc"], P["kw"]["p_bnd_fn"], P["U0"], P["pc_part"]


def _problem(case, seed):
    """The problem's inputs as numpy arrays: mesh, boundary types and values,
    permeability, porosity, residual saturation, hydrostatic state, and the
    preconditioner's blocks."""
    rng = np.random.default_rng([int(seed), 7])
    part = None
    if case["mesh"] == "prism":
        m, fbc, pb, U0, part = _prism_mesh(case["tri"], case["layers"], max(1, min(6, 64 // case["layers"])))
        nl = case["layers"]
        z, layer = np.unique(np.round(m.cell_cen[:, 2], 9), return_inverse=True)
        field = mg.layered_K(64, 64, nl, rng)[:, 0].reshape(nl, 64, 64)
        hi = m.vert_xyz.max(axis=0)
        ix = np.clip((m.cell_cen[:, 0] / hi[0] * 64).astype(np.int64), 0, 63)
        iy = np.clip((m.cell_cen[:, 1] / hi[1] * 64).astype(np.int64), 0, 63)
        k = field[layer.ravel(), iy, ix]
        K = np.zeros((m.nc, 9))
        K[:, 0] = K[:, 4] = k
        K[:, 8] = k / 10.0
    else:
        m, fbc, pb, U0 = _box_mesh(case["mesh"], case["nx"], case["ny"], case["nz"])
        if case["mesh"] == "cube":
            K = mg.random_rotated_K(m.nc, rng, -12.0, 0.5)
        else:
            K = mg.layered_K(case["nx"], case["ny"], case["nz"], rng)
        if case.get("coarse") or case.get("block") == 64:
            part = mg.brick_partition(m, *((8, 8, 4) if case.get("block") == 256 else (4, 4, 4)))
    phi = rng.uniform(0.2, 0.4, size=m.nc)
    return dict(mesh=m, face_bc=fbc, p_bnd=pb, K=K, phi=phi, Sr=np.full(m.nc, 0.1), U0=U0, part=part,
                density=case["density"], rng=rng)


def _states(case, P):
    """The host inputs of a call: a state away from equilibrium and its rate."""
    rng, nc = P["rng"], P["mesh"].nc
    U = P["U0"] + 2e4 * (rng.random(nc) - 0.5)
    Ud = 1e-2 * (rng.random(nc) - 0.5)
    Uprev = U + 500.0 * (rng.random(nc) - 0.5)
    return U, Ud, Uprev


def _dt(case):
    return DAY if case["mesh"] == "layered" else HOUR


def prepare(case, seed):
    P = _problem(case, seed)
    g = MPFAO(P["mesh"], P["face_bc"], P["K"], P["phi"], P["Sr"], vg_m=VG_M, vg_alpha=VG_ALPHA, poly=POLY,
              gravity=GRAVITY, density=P["density"], gmatrix="mpfao", pref=PREF, p_bnd_fn=P["p_bnd"])
    dev = lambda a: torch.tensor(a, dtype=torch.float64, device="cuda")  # noqa: E731
    s = dict(case=case, g=g, dt=_dt(case))
    if case["kind"] == "step":
        if P["part"] is not None:
            g.set_pc_partition(P["part"])
        s["U0"] = dev(P["U0"])
        s["U"] = torch.empty_like(s["U0"])
        s["opts"] = g.solver_options(snes_rtol=1e-10, ksp_rtol=1e-5, pc_block=case["block"],
                                     krylov_fp32=int(case["fp32"]), pc_coarse=int(case["coarse"]))
        return s
    U, Ud, Uprev = _states(case, P)
    s["U"] = dev(U)
    if case["kind"] == "recover":
        return s
    s["Ud"], s["R"] = dev(Ud), torch.empty_like(s["U"])
    if case["kind"] == "callbacks":
        s["J"] = torch.empty(g.jac_nnz, dtype=torch.float64, device="cuda")
        if case["form"] == "snes":
            g.SetDtime(s["dt"])
            g.SNESPreSolve(dev(Uprev))
    return s


def run(s):
    case, g = s["case"], s["g"]
    if case["kind"] == "residual":
        g.IFunction(0.0, s["U"], s["Ud"], s["R"])
        return s["R"]
    if case["kind"] == "callbacks":
        if case["form"] == "ts":
            g.IFunction(0.0, s["U"], s["Ud"], s["R"])
            g.IJacobian(0.0, s["U"], s["Ud"], 1.0 / s["dt"], s["J"])
        else:
            g.SNESFunction(s["U"], s["R"])
            g.SNESJacobian(s["U"], s["J"])
        return s["R"], s["J"]
    if case["kind"] == "recover":
        S, mass, water = g.Diagnostics(s["U"])
        vel, cnt = g.RecoverVelocity(s["U"])
        return {"S": S, "mass": mass, "water": water, "vel": vel, "count": cnt}
    U, dt = s["U"], s["dt"]
    U.copy_(s["U0"])
    if case["driver"] == "snes":
        g.run_snes_steps(U, dt, 1, s["opts"])
    elif case["driver"] == "ts":
        g.run_ts_be(U, dt, 1, s["opts"])
    else:
        g.run_tdyti(U, dt, 1.5, 4 * dt, dt, s["opts"])
    return U


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    """Bytes: each input read and each output written once (transmissibilities
    T, gravity term, connectivity, per-cell materials and state, residual,
    Jacobian).  A time step: NEWTON Newton iterations of residual, Jacobian,
    factorisation and KRYLOV Krylov steps each (matrix, factor and two passes
    over half a restart's basis), counts typical of these problems."""
    if case["mesh"] == "prism":
        nc = case["tri"] * case["layers"]
        nf, nv, ncol, row = 2.55 * nc, 0.53 * nc, 12.0, 39.0
        trow = 9.5 * nc
    else:
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        nc = nx * ny * nz
        nf = (nx + 1) * ny * nz + nx * (ny + 1) * nz + nx * ny * (nz + 1)
        nv, ncol, row = (nx + 1) * (ny + 1) * (nz + 1), 8.0, 27.0
        trow = 4.0 * nf - 8.0 * (nx + ny) * nz
    t_bytes = trow * (ncol * 8 + 8) + nv * ncol * 4 + nf * 24
    res_bytes = t_bytes + nc * 8 * 7
    res_flops = trow * (2 * ncol + 12) + nc * 60
    jac_bytes = nc * row * 8
    jac_flops = trow * ncol * 6
    if case["kind"] == "residual":
        return {"bytes": res_bytes, "flops": res_flops}
    if case["kind"] == "callbacks":
        return {"bytes": res_bytes + jac_bytes, "flops": res_flops + jac_flops}
    if case["kind"] == "recover":
        return {"bytes": t_bytes + nc * 8 * 7 + nf * 12, "flops": trow * 2 * ncol + nc * 60}
    newton, krylov = 5.0, 60.0
    tv = 4 if case["fp32"] else 8
    it = nc * tv * (27 * 2 + 2 * 15 + 4)
    return {"bytes": newton * (2 * res_bytes + jac_bytes + nc * 27 * (8 + tv) + krylov * it),
            "flops": newton * (2 * res_flops + jac_flops + nc * 700.0 + krylov * nc * (4 * 27 + 4 * 15))}


# ---------------------------------------------------------------- plain FP64 mathematics

def _saturation(Sr, Pc):
    """van Genuchten S, dS/dp, d2S/dp2 at capillary pressure Pc = pref - p."""
    m, a, n = VG_M, VG_ALPHA, 1.0 / (1.0 - VG_M)
    dry = Pc > 0
    pc = np.where(dry, Pc, 1.0)
    pan = (pc * a) ** n
    Se = (1 + pan) ** -m
    dSe = -m * n * pan / pc * (1 + pan) ** (-m - 1)
    d2Se = m * n * pan * (1 + pan) ** (-m - 2) * ((m * n + 1) * pan - n + 1) / pc ** 2
    return (np.where(dry, (1 - Sr) * Se + Sr, 1.0), np.where(dry, -dSe * (1 - Sr), 0.0),
            np.where(dry, (1 - Sr) * d2Se, 0.0))


def _kr_unsmoothed(Se):
    m = VG_M
    x = np.clip(Se, 1e-300, 1 - 1e-16)
    s1 = x ** (1 / m)
    t = (1 - s1) ** m
    kr = np.sqrt(x) * (1 - t) ** 2
    return kr, 0.5 * kr / x + 2 * x ** (1 / m - 0.5) * (1 - s1) ** (m - 1) * (1 - t)


def _mualem(Se):
    """Relative permeability and its derivative, a cubic above Se = POLY[1]
    that meets the curve (value and slope) there and 1 (slope 0) at POLY[2]."""
    x0, x1, x2, dx = POLY
    kr1, dkr1 = _kr_unsmoothed(np.float64(x1))
    row = lambda x: [1, x, x * x, x ** 3]  # noqa: E731
    slope = lambda x: [0, 1 / dx, 2 * x / dx, 3 * x * x / dx]  # noqa: E731
    t1, t2 = (x1 - x0) / dx, (x2 - x0) / dx
    c = np.linalg.solve(np.array([row(t2), row(t1), slope(t1), slope(t2)], dtype=np.float64),
                        np.array([1.0, kr1, dkr1, 0.0]))
    kr, dkr = _kr_unsmoothed(Se)
    t = (Se - x0) / dx
    top = Se > x1
    return (np.where(top, c[0] + t * (c[1] + t * (c[2] + t * c[3])), kr),
            np.where(top, (c[1] + t * (2 * c[2] + t * 3 * c[3])) / dx, dkr))


def _density(kind, p):
    if kind == "constant":
        return np.full_like(p, 998.0), np.zeros_like(p), np.zeros_like(p)
    rho = np.where(p < PREF, 997.16, 997.16 * np.exp(1e-8 * np.maximum(p - PREF, 0)))
    d = np.where(p < PREF, 0.0, 1e-8 * rho)
    return rho, d, 1e-8 * d


class _Plain:
    """The discretisation of one problem from mesh and materials."""

    def __init__(self, P):
        self.P, m = P, P["mesh"]
        nc, nf, nv = m.nc, m.nf, m.nv
        fv, cv, fc = m.face_verts, m.cell_verts, m.face_cells
        self.up, self.dn = fc[:, 0].astype(np.int64), fc[:, 1].astype(np.int64)
        nvf = (fv >= 0).sum(1)
        self.area = m.face_area / nvf
        bc = P["face_bc"]
        self.noflow = bc == mg.BC_NEUMANN
        self.dirichlet = (self.up < 0) & ~self.noflow
        # rank of every (face, vertex) and (cell, vertex) among those of the vertex
        def ranks(v):
            flat = v.ravel()
            live = np.nonzero(flat >= 0)[0]
            o = live[np.argsort(flat[live], kind="stable")]
            s = flat[o]
            start = np.searchsorted(s, s)
            r = np.full(flat.shape[0], -1, np.int64)
            r[o] = np.arange(o.shape[0]) - start
            return r.reshape(v.shape), int(r.max()) + 1
        self.frank, F = ranks(fv)
        crank, C = ranks(cv)
        self.F, self.C = F, C
        self.vcell = np.full((nv, C), -1, np.int64)
        K = P["K"].reshape(-1, 3, 3)
        A = np.zeros((nv, F, F))
        B = np.zeros((nv, F, C))
        self.g_up = np.zeros((nf, 4, 3))                 # flux of the up side: coefficients of (x_k - p)
        self.k_up = np.zeros((nf, 4, 3), np.int64)       # and the ranks k of the three faces
        cf = m.cell_faces
        for s in range(8):
            c = np.nonzero(cv[:, s] >= 0)[0]
            if not c.size:
                continue
            v = cv[c, s].astype(np.int64)
            self.vcell[v, crank[c, s]] = c
            faces = cf[c]
            at = (fv[np.maximum(faces, 0)] == v[:, None, None]) & (faces >= 0)[:, :, None]
            lf = np.argsort(~at.any(2), axis=1, kind="stable")[:, :3]
            fid = np.take_along_axis(faces, lf, 1).astype(np.int64)
            q = np.take_along_axis(at.argmax(2), lf, 1)
            k = self.frank[fid, q]
            e = m.face_cen[fid] - m.cell_cen[c][:, None]
            nu = np.stack([np.cross(e[:, 1], e[:, 2]), np.cross(e[:, 2], e[:, 0]), np.cross(e[:, 0], e[:, 1])], 1)
            nu /= np.einsum("id,id->i", e[:, 0], nu[:, 0])[:, None, None]
            kn = np.einsum("iab,ijb->ija", K[c], nu)
            g = np.einsum("ila,ija->ilj", m.face_normal[fid], kn) * self.area[fid][:, :, None]
            i = crank[c, s]
            for l in range(3):
                f, kl = fid[:, l], k[:, l]
                first = (self.up[f] == c) | (self.up[f] < 0)
                w = np.where(self.dirichlet[f], 0.0, np.where(first, 1.0, -1.0))
                for j in range(3):
                    np.add.at(A, (v, kl, k[:, j]), w * g[:, l, j])
                    np.add.at(B, (v, kl, i), w * g[:, l, j])
                fs, qs = f[first], q[first, l]
                self.g_up[fs, qs] = g[first, l]
                self.k_up[fs, qs] = k[first]
        # Dirichlet faces hold their pressure; absent faces are the identity
        self.fv, self.live = fv.astype(np.int64), fv >= 0
        present = np.zeros((nv, F), bool)
        present[fv[self.live], self.frank[self.live]] = True
        held = ~present
        self.df, self.dq = np.nonzero(self.live & self.dirichlet[:, None])
        held[fv[self.df, self.dq], self.frank[self.df, self.dq]] = True
        hv, hk = np.nonzero(held)
        A[hv, hk, hk] = 1.0
        self.A, self.B = A, B
        self._gravity(K)

    def _gravity(self, K):
        m, up, dn = self.P["mesh"], self.up, self.dn
        fc = m.face_cen
        cu = np.where((up >= 0)[:, None], m.cell_cen[np.maximum(up, 0)], fc)
        cd = m.cell_cen[dn]
        u = cd - cu
        u /= np.linalg.norm(u, axis=1)[:, None]
        du = np.where(up >= 0, np.linalg.norm(cu - fc, axis=1), 0.0)
        w = du / (du + np.linalg.norm(cd - fc, axis=1))
        Ki, Kj = np.linalg.inv(K[np.where(up >= 0, up, dn)]), np.linalg.inv(K[dn])
        Kf = np.linalg.inv(w[:, None, None] * Ki + (1 - w)[:, None, None] * Kj)
        Kf[(Kf < 0) | (np.abs(Kf) < 2.220446049250313e-16)] = 0.0
        self.G = self.area * np.einsum("fa,fab,fb->f", m.face_normal, Kf, u) * GRAVITY * u[:, 2]

    def face_pressures(self, p, pb):
        """x (nv, F): the pressures at the vertices' sub-faces."""
        pc = np.where(self.vcell >= 0, p[np.maximum(self.vcell, 0)], 0.0)
        rhs = np.einsum("vfc,vc->vf", self.B, pc)
        rhs[self.fv[self.df, self.dq], self.frank[self.df, self.dq]] = pb[-self.up[self.df] - 1]
        return np.linalg.solve(self.A, rhs[:, :, None])[:, :, 0]

    def rows_tp(self, p, pb):
        """T.P of every flux row (nf, 4)."""
        x = self.face_pressures(p, pb)
        own = p[np.where(self.up >= 0, self.up, self.dn)]
        v = np.maximum(self.fv, 0)
        tp = ((x[v[:, :, None], self.k_up] - own[:, None, None]) * self.g_up).sum(2)
        return np.where(self.live & ~self.noflow[:, None], tp, 0.0)

    def rows_T(self):
        """Coefficients of every flux row in its vertex's cells (nf, 4, C)."""
        X = np.linalg.solve(self.A, self.B)
        v = np.maximum(self.fv, 0)
        T = np.zeros(self.fv.shape + (self.C,))
        for j in range(3):
            T += self.g_up[:, :, j, None] * X[v, self.k_up[:, :, j]]
        own = np.where(self.up >= 0, self.up, self.dn)
        T -= np.where(self.vcell[v] == own[:, None, None], self.g_up.sum(2)[:, :, None], 0.0)
        T[~self.live | self.noflow[:, None]] = 0.0
        return T

    def state(self, p, Sr):
        S, dS, d2S = _saturation(Sr, PREF - p)
        kr, dkr = _mualem((S - Sr) / (1 - Sr))
        return S, dS, d2S, kr / VISCOSITY, dkr / (1 - Sr) * dS / VISCOSITY

    def evaluate(self, p, form, rate, jac):
        """(R, J values by (row, col) or None); rate: Udot and shift (TS), or
        the accumulation of the previous state and dt (SNES)."""
        P, m = self.P, self.P["mesh"]
        up, dn, nc = self.up, self.dn, m.nc
        phi, V, pb = P["phi"], m.cell_vol, P["p_bnd"]
        S, dS, d2S, uk, duk = self.state(p, P["Sr"])
        rho, dr, d2r = _density(P["density"], p)
        rb = _density(P["density"], np.array([PREF]))[0][0]
        uk_b = self.state(pb, P["Sr"][dn[m.bnd_face]])[3]
        u0, b0 = np.maximum(up, 0), np.maximum(-up - 1, 0)
        inner = up >= 0
        den = 0.5 * (np.where(inner, rho[u0], rb) + rho[dn])[:, None]
        tp, G = self.rows_tp(p, pb), self.G[:, None]
        from_up = tp + den * G < 0
        lam = np.where(from_up, np.where(inner, uk[u0], uk_b[b0] if pb.size else 0.0)[:, None], uk[dn][:, None])
        live = self.live & ~self.noflow[:, None]
        flux = np.where(live, -den * lam * tp - den ** 2 * lam * G, 0.0)
        fs = flux.sum(1)
        R = np.bincount(up[inner], fs[inner], nc) - np.bincount(dn, fs, nc)
        dM = (dr * S + rho * dS) * phi
        d2M = (2 * dS * dr + S * d2r + d2S * rho) * phi
        if form == "ts":
            Ud, shift = rate
            R += dM * Ud * V
            diag = (shift * dM + d2M * Ud) * V
        else:
            prev, dt = rate
            R += rho * phi * S * V / dt - prev
            diag = dM * V / dt
        if not jac:
            return R, None
        T = self.rows_T()
        v = np.maximum(self.fv, 0)
        cols = self.vcell[v]
        D = (den * lam)[:, :, None] * T
        for side, c in ((True, np.where(inner, up, -2)), (False, dn)):
            dd = 0.5 * np.where(c >= 0, dr[np.maximum(c, 0)], 0.0)[:, None]
            dl = np.where((from_up == side) & (c >= 0)[:, None], duk[np.maximum(c, 0)][:, None], 0.0)
            own = dd * lam * tp + den * dl * tp + 2 * den * dd * lam * G + den ** 2 * dl * G
            D += np.where(cols == c[:, None, None], own[:, :, None], 0.0)
        ok = (cols >= 0) & live[:, :, None]
        keep = ok & inner[:, None, None]
        r = np.concatenate([np.broadcast_to(up[:, None, None], ok.shape)[keep],
                            np.broadcast_to(dn[:, None, None], ok.shape)[ok], np.arange(nc)])
        cc = np.concatenate([cols[keep], cols[ok], np.arange(nc)])
        return R, (r, cc, np.concatenate([-D[keep], D[ok], diag]))

    def csr_values(self, r, c, val):
        """The entries summed into the vertex-adjacency pattern, rows then
        columns ascending."""
        nc = self.P["mesh"].nc
        i, j = np.broadcast_arrays(self.vcell[:, :, None], self.vcell[:, None, :])
        ok = (i >= 0) & (j >= 0)
        keys = np.unique(i[ok] * nc + j[ok])
        return np.bincount(np.searchsorted(keys, r * nc + c), val, keys.shape[0])

    def accumulation(self, p):
        P = self.P
        S = _saturation(P["Sr"], PREF - p)[0]
        return _density(P["density"], p)[0] * P["phi"] * S * P["mesh"].cell_vol

    def step(self, p, dt, ts):
        """One backward-Euler step by damped Newton with dense solves, or None
        where that does not converge."""
        prev = self.accumulation(p) / dt
        old = p.copy()
        ev = lambda x, jac: self.evaluate(  # noqa: E731
            x, *(("ts", ((x - old) / dt, 1 / dt)) if ts else ("snes", (prev, dt))), jac)
        nc = p.shape[0]
        R, J = ev(p, True)
        r0 = np.linalg.norm(R)
        for _ in range(40):
            M = np.zeros((nc, nc))
            np.add.at(M, (J[0], J[1]), J[2])
            d = torch.linalg.solve(torch.from_numpy(M), torch.from_numpy(R)).numpy()
            lam, n0 = 1.0, np.linalg.norm(R)
            while lam > 1e-4 and not np.linalg.norm(ev(p - lam * d, False)[0]) < n0:
                lam *= 0.5
            if lam <= 1e-4:
                break
            p = p - lam * d
            R, J = ev(p, True)
            if np.linalg.norm(R) <= 1e-13 * r0:
                break
        return p if np.linalg.norm(R) <= 1e-11 * r0 else None


def exact(case, seed):
    if case["mesh"] == "prism":
        nc = case["tri"] * case["layers"] * 3  # their local systems are larger
    else:
        nc = case["nx"] * case["ny"] * case["nz"]
    if nc > (EXACT_STEP_CELLS if case["kind"] == "step" else EXACT_CELLS):
        return None
    P = _problem(case, seed)
    plain, dt = _Plain(P), _dt(case)
    if case["kind"] == "step":
        p = plain.step(P["U0"].copy(), dt, case["driver"] == "ts")
        return None if p is None else torch.from_numpy(p)
    U, Ud, Uprev = _states(case, P)
    t = torch.from_numpy
    if case["kind"] == "residual":
        return t(plain.evaluate(U, "ts", (Ud, 0.0), False)[0])
    if case["kind"] == "callbacks":
        rate = (Ud, 1.0 / dt) if case["form"] == "ts" else (plain.accumulation(Uprev) / dt, dt)
        R, J = plain.evaluate(U, case["form"], rate, True)
        return t(R), t(plain.csr_values(*J))
    S = _saturation(P["Sr"], PREF - U)[0]
    rho, V = _density(P["density"], U)[0], P["mesh"].cell_vol
    tp = plain.rows_tp(U + rho * GRAVITY * P["mesh"].cell_cen[:, 2], P["p_bnd"])
    vel = -(tp / P["mesh"].face_area[:, None]).sum(1)
    return {"S": t(S), "mass": t(rho * V), "water": t(rho * P["phi"] * S * V), "vel": t(vel), "count": None}
