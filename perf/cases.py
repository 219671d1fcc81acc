"""Performance cases of the explicit residual / update path and its adjoints on one GPU.

Every case drives `mose_amd.lib.GpuSolver` as a host program does: a context per case, marches of
many steps with the state resident on the device, the state fetched at the end of a march.

  march     advance `steps` explicit steps from the present state, then fetch every block's state
  vjp       one residual adjoint: upload the residual adjoints, mose_residual_vjp, fetch
  solve     `steps` iterations of the steady adjoint solve, fetch the residual adjoint
  reverse   a fixed-dt march of `steps` steps and its reverse sweep for the kinetic energy
"""
import math

import numpy as np
import torch

from mose_amd import abi, cases
from mose_amd.lib import GpuSolver

GAMMA = cases.GAMMA
RGAS = cases.RGAS_NONDIM
RK = {1: (1.0,), 2: (1.0, 0.5), 3: (1.0, 0.25, 2.0 / 3.0)}


def _case(kind, flow, ni, nj, nk, steps, name=None, limiter="vanleer", riemann="HLLC", fp32=False, sd=False, irs=0.0,
          blocks=1, layout=0, tune=False):
    c = {"kind": kind, "flow": flow, "ni": ni, "nj": nj, "nk": nk, "steps": steps, "limiter": limiter, "riemann": riemann,
         "fp32": fp32, "sd": sd, "irs": irs, "blocks": blocks, "layout": layout, "tune": tune}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the shock tube of the 1-D test family: steps of a few microseconds of work each
        _case("march", "sod", 1000, 1, 1, 200, "sod_1000", limiter="minmod"),
        # a small periodic box of odd sizes, as in parameter studies and tests
        _case("march", "vortex", 33, 25, 17, 100, "vortex_33x25x17", riemann="HLLE"),
        # the 2-D body-fitted channel marched to its steady state with local time steps
        _case("march", "bump", 512, 256, 1, 100, "bump_512x256", limiter="minmod"),
        # a mid-size box of ragged sizes with the other flux scheme, library defaults
        _case("march", "vortex", 131, 97, 75, 100, "vortex_131x97x75_ausm", riemann="AUSM+"),
        # the headline workload: the largest box, tiling picked by the tuner as a long run does
        _case("march", "vortex", 256, 256, 256, 60, "vortex_256", tune=True),
        # many unequal blocks joined 1-to-1, FP32 fluxes
        _case("march", "chain", 16, 72, 0, 60, "chain_32_fp32", fp32=True, blocks=32, layout=1234),
        # batched viscous Taylor-Green boxes, FP64 and FP32 fluxes
        _case("march", "tgv", 128, 128, 128, 40, "tgv_2x128", riemann="AUSM+", blocks=2),
        _case("march", "tgv", 96, 96, 96, 60, "tgv_3x96_fp32", riemann="AUSM+", fp32=True, blocks=3),
        # shock-detector reconstruction, and implicit residual smoothing
        _case("march", "vortex", 120, 120, 120, 60, "vortex_120_muscl_sd", limiter="minmod", riemann="HLLE", sd=True),
        _case("march", "vortex", 128, 96, 80, 60, "vortex_128x96x80_irs", irs=0.5),
        # the steady adjoint of the channel
        _case("solve", "bump", 384, 192, 1, 100, "bump_384x192_adjoint"),
        # Reynolds-number sensitivity through the march of viscous boxes
        _case("reverse", "tgv", 96, 96, 96, 8, "tgv_2x96_reverse", riemann="AUSM+", blocks=2),
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    flow = rng.choice(["sod", "vortex", "vortex", "vortex", "bump", "chain", "tgv", "tgv", "solve", "reverse", "vjp"])
    limiter = rng.choice(["vanleer", "vanalbada", "mc"])
    if flow == "sod":
        return _case("march", "sod", _size(rng, 100, 4000), 1, 1, rng.randint(50, 200), limiter=rng.choice(["minmod", "vanleer"]),
                     riemann=rng.choice(["HLLC", "HLLE", "AUSM+"]))
    if flow == "vortex":
        sd = rng.random() < 0.25
        irs = 0.5 if not sd and rng.random() < 0.25 else 0.0
        n = [_size(rng, 16, 200) for _ in range(3)]
        return _case("march", "vortex", n[0], n[1], n[2], rng.randint(20, 60), limiter="minmod" if sd else limiter,
                     riemann=rng.choice(["HLLC", "AUSM+", "HLLE"]), sd=sd, irs=irs)
    if flow == "bump":
        return _case("march", "bump", _size(rng, 48, 640), _size(rng, 24, 320), 1, rng.randint(20, 100), limiter="minmod")
    if flow == "chain":
        return _case("march", "chain", 16, rng.randint(32, 80), 0, rng.randint(20, 50), limiter="vanleer", fp32=rng.random() < 0.5,
                     blocks=rng.randint(4, 40), layout=rng.randint(1, 10 ** 6))
    if flow in ("tgv", "reverse"):
        n = _size(rng, 20, 96 if flow == "reverse" else 130)
        kind = "march" if flow == "tgv" else "reverse"
        return _case(kind, "tgv", n, n, n, rng.randint(4, 8) if kind == "reverse" else rng.randint(20, 50),
                     riemann=rng.choice(["AUSM+", "HLLC"]), fp32=kind == "march" and rng.random() < 0.4, blocks=rng.randint(1, 3))
    if flow == "solve":
        return _case("solve", "bump", _size(rng, 48, 512), _size(rng, 24, 256), 1, rng.randint(20, 100))
    n = [_size(rng, 16, 120) for _ in range(3)]
    return _case("vjp", "vortex", n[0], n[1], n[2], 1, limiter=rng.choice(["vanleer", "vanalbada"]), riemann=rng.choice(["HLLC", "AUSM+"]))


# ------------------------------------------------------------------------------------ inputs
def _cfg(case, cfl, time_accurate=True):
    return abi.make_cfg(GAMMA, RGAS, cfl, case["limiter"], case["riemann"], 3, time_accurate,
                        precision=abi.PREC_FP32_FLUX if case["fp32"] else abi.PREC_FP64, muscl_sd=case["sd"], irs_beta=case["irs"])


def _perturb(prim, rng, amp, nmodes=2):
    """Smooth seeded modes on every variable (no direction stays uniform): prim (nk, nj, ni, 5)."""
    shape = prim.shape[:-1]
    for v in range(5):
        s = 0.0
        for _ in range(nmodes):
            waves = [np.sin(2.0 * np.pi * rng.integers(1, 4) * (np.arange(n) + 0.5) / n + 2.0 * np.pi * rng.random()) for n in shape]
            s = s + waves[0][:, None, None] * (waves[1][:, None] * waves[2])
        if v in (0, 4):
            prim[..., v] *= 1.0 + amp * s
        else:
            prim[..., v] += amp * s
    return prim


def _vortex(case, rng):
    dims = (case["ni"], case["nj"], case["nk"])
    L = 10.0
    nodes = cases.cartesian_nodes(dims, (0.0, 0.0, 0.0), (L, L, L))
    x, y = ((np.arange(n) + 0.5) * (L / n) for n in dims[:2])
    xc = np.zeros((1, dims[1], dims[0], 3))
    xc[..., 0], xc[..., 1] = x, y[:, None]
    plane = cases.vortex_exact(xc, 0.0, x0=4.0 + 2.0 * rng.random(), y0=4.0 + 2.0 * rng.random())
    prim = _perturb(np.repeat(plane, dims[2], axis=0), rng, 0.02)
    bc = cases.bc_records([{"dims": dims, "faces": cases.periodic_faces(1)}])
    return cases.Case("vortex", _cfg(case, 0.4), [cases.Block(dims, nodes, cases.padded_state(dims, prim))], bc)


def _sod(case, rng):
    c = cases.sod(n=case["ni"], limiter=case["limiter"], riemann=case["riemann"])
    P = c.blocks[0].P
    left = P[..., 0] > 0.5
    for v in (0, 4):
        P[..., v] *= np.where(left, 0.9 + 0.2 * rng.random(), 0.9 + 0.2 * rng.random())
    return c


def _bump(case, rng):
    heights = 0.002 * rng.random(16)
    c = cases.bump_channel(ni=case["ni"], nj=case["nj"], ncontrol=16, heights=heights, limiter=case["limiter"],
                           riemann=case["riemann"], alpha=0.02 * rng.random())
    if case["kind"] == "solve":      # the state about which the adjoint is taken: a smooth supersonic flow
        prim = _perturb(np.ascontiguousarray(abi.interior(c.blocks[0].P)), rng, 0.02)
        c.blocks[0].P = cases.padded_state(c.blocks[0].dims, prim)
    return c


def _chain(case, rng):
    c = cases.multiblock_chain(nblocks=case["blocks"], seed=case["layout"], lo=case["ni"], hi=case["nj"], riemann=case["riemann"],
                               limiter=case["limiter"], precision=abi.PREC_FP32_FLUX if case["fp32"] else abi.PREC_FP64)
    waves = [(rng.integers(1, 4, 3) * 2.0, 2.0 * np.pi * rng.random(3)) for _ in range(5)]
    for q, blk in enumerate(c.blocks):
        prim = np.ascontiguousarray(abi.interior(blk.P))
        for v, (k, ph) in enumerate(waves):
            s = [np.sin(k[d] * (c.meta["origin"][q][d] + c.meta["h"] * (np.arange(blk.dims[d]) + 0.5)) + ph[d]) for d in range(3)]
            s = s[2][:, None, None] * (s[1][:, None] * s[0])
            if v in (0, 4):
                prim[..., v] *= 1.0 + 0.01 * s
            else:
                prim[..., v] += 0.01 * s
        blk.P = cases.padded_state(blk.dims, prim)
    return c


def _tgv(case, rng):
    c = cases.taylor_green(n=case["ni"], nbox=case["blocks"], seed=int(rng.integers(1 << 30)), limiter=case["limiter"],
                           riemann=case["riemann"], precision=abi.PREC_FP32_FLUX if case["fp32"] else abi.PREC_FP64)
    for blk in c.blocks:
        prim = np.ascontiguousarray(abi.interior(blk.P))
        pert = _perturb(np.ones_like(prim), rng, 1.0) - 1.0
        prim[..., 0] += 0.002 * pert[..., 0]
        prim[..., 1:4] += 0.05 * pert[..., 1:4]
        prim[..., 4] += 0.1 * pert[..., 4]
        blk.P = cases.padded_state(blk.dims, prim)
    return c


_FLOWS = {"vortex": _vortex, "sod": _sod, "bump": _bump, "chain": _chain, "tgv": _tgv}


def _bars(case, c, rng):
    """Adjoint inputs per block, blk%R layout with ghost entries 0."""
    out = []
    for blk in c.blocks:
        x = np.zeros(abi.padded_shape(blk.dims))
        inner = abi.interior(x)
        if case["kind"] == "solve":      # an objective of the wall pressure (first row of cells)
            inner[:, 0, :, 4] = 1e-2 * (1.0 + 0.5 * np.sin(np.linspace(0.0, 6.0, blk.dims[0]) + 6.0 * rng.random()))
        else:
            inner[...] = rng.standard_normal(inner.shape)
        out.append(x)
    return out


def _inputs(case, seed):
    rng = np.random.default_rng([seed, 7])
    c = _FLOWS[case["flow"]](case, rng)
    bars = _bars(case, c, rng) if case["kind"] in ("vjp", "solve") else None
    return c, bars


def _fixed_dt(case):
    """Time step of the fixed-dt march: CFL 0.4 of the Taylor-Green flow (Mach 0.1, speeds below 1.5)."""
    return 0.4 * (2.0 * math.pi / case["ni"]) / 11.5


def prepare(case, seed):
    c, bars = _inputs(case, seed)
    g = GpuSolver(c)
    if case["tune"]:
        g.autotune(3)
    return {"case": case, "solver": g, "bars": bars, "P": [b.P for b in c.blocks] if case["flow"] == "sod" else None}


# --------------------------------------------------------------------------------------- run
def run(state):
    case, g = state["case"], state["solver"]
    nb = len(g.dims)
    if case["kind"] == "march":
        if state["P"] is not None:       # a whole run from the initial state, as a shock-tube study does
            g.put_state(1, state["P"][0])
        t, norms = g.advance(case["steps"])
        return {"states": [abi.interior(g.get_state(b)) for b in range(1, nb + 1)], "norms": norms} if nb < 60 else [
            abi.interior(g.get_state(b)) for b in range(1, nb + 1)]
    if case["kind"] == "vjp":
        return [abi.interior(p) for p in g.residual_vjp(state["bars"])]
    if case["kind"] == "solve":
        psi, it, r0, r = g.adjoint_solve(state["bars"], max_iter=case["steps"], rtol=0.0, check_every=case["steps"])
        return {"psi": [abi.interior(p) for p in psi], "res": np.array([r0, r])}
    ke, mub, P0b = g.march_kinetic_energy(case["steps"], _fixed_dt(case))
    return {"ke": ke, "mu_bar": mub, "P0_bar": [abi.interior(p) for p in P0b]}


def _cells(case):
    if case["flow"] == "chain":      # seeded sizes
        return float(_chain(case, np.random.default_rng(0)).ncells)
    return case["blocks"] * case["ni"] * case["nj"] * case["nk"]


def work(case):
    """Per cell and RK stage: the stage input and U^n read and the result written (5 FP64 each), the
    slopes and Riemann problems of three faces (two in the plane cases); an adjoint stage reads the state
    and the residual adjoint and writes the state adjoint, and does about three times the operations."""
    n, steps = _cells(case), case["steps"]
    faces = {"sod": 1, "bump": 2}.get(case["flow"], 3)
    ops = 250 * faces + 60 + (200 * faces if case["flow"] == "tgv" else 0)
    if case["kind"] == "march":
        return {"bytes": 120.0 * 3 * steps * n + 40.0 * n, "flops": 1.0 * ops * 3 * steps * n}
    if case["kind"] == "vjp":
        return {"bytes": 120.0 * n, "flops": 3.0 * ops * n}
    if case["kind"] == "solve":
        return {"bytes": 240.0 * 3 * steps * n, "flops": 3.0 * ops * 3 * steps * n}
    return {"bytes": (120.0 + 240.0) * 3 * steps * n, "flops": 5.0 * ops * 3 * steps * n}


# ------------------------------------------------------- the same numbers in plain torch, 64 bits
class _Plain:
    """Rectilinear uniform blocks with faces of type 101 / 201 (aligned), 400 or 0: the scheme in
    torch on primitive fields (5, nk, nj, ni), differentiable."""

    def __init__(self, case, c, dev):
        self.case, self.dev = case, dev
        self.dims = [b.dims for b in c.blocks]
        self.h = [[float((b.nodes[-1, -1, -1, d] - b.nodes[0, 0, 0, d]) / b.dims[d]) for d in range(3)] for b in c.blocks]
        self.face = {}
        for r in c.bc[np.unique(c.bc[["b", "f"]], return_index=True)[1]]:
            self.face[int(r["b"]) - 1, int(r["f"]) - 1] = (int(r["type"]), int(r["bs"]) - 1, int(r["fs"]) - 1)
        self.ndir = 1 if case["flow"] == "sod" else 3
        self.visc = {b - 1: [torch.tensor(float(p), dtype=torch.float64, device=dev) for p in prm] for b, prm in c.meta.get("viscous", [])}
        self.cfl = float(c.cfg.cfl)

    def pad(self, P, b):
        """P[b] with two ghost layers on every face (edges and corners by periodic wrap only)."""
        X = P[b]
        if all(self.face[b, f][:2] == (201, b) for f in range(6)):
            return torch.nn.functional.pad(X[None], (2,) * 6, mode="circular")[0]
        out = torch.nn.functional.pad(X, (2,) * 6, value=1.0)
        for d in range(self.ndir):
            for side in range(2):
                typ, bs, fs = self.face[b, 2 * d + side]
                ax, n = 3 - d, self.dims[b][d]
                if typ in (101, 201):
                    m = self.dims[bs][d]
                    near, far = (0, 1) if fs % 2 == 0 else (m - 1, m - 2)
                    g1, g2 = P[bs].select(ax, near), P[bs].select(ax, far)
                else:
                    q = [X.select(ax, s if side == 0 else n - 1 - s) for s in range(3)]
                    g1 = 3.0 * q[0] - 3.0 * q[1] + q[2]
                    g2 = 3.0 * g1 - 3.0 * q[0] + q[1]
                mid = [slice(None)] + [slice(2, -2)] * 3
                for layer, g in ((1, g1), (2, g2)):
                    at = list(mid)
                    at[ax] = 2 - layer if side == 0 else n + 1 + layer
                    out[tuple(at)] = g
        return out

    def limiter(self, x, y):
        lim = self.case["limiter"]
        if lim == "minmod":
            return torch.where(x * y < 0, torch.zeros_like(x), torch.where(x.abs() > y.abs(), y, x))
        if lim == "vanleer":
            ok = x * y > 0
            return torch.where(ok, 2.0 * x * y / torch.where(ok, x + y, torch.ones_like(x)), torch.zeros_like(x))
        if lim == "vanalbada":
            q = x * x + y * y
            return torch.where(q > 0, x * y * (x + y) / torch.where(q > 0, q, torch.ones_like(q)), torch.zeros_like(x))
        m = torch.minimum(2.0 * torch.minimum(x.abs(), y.abs()), 0.5 * (x.abs() + y.abs()))      # mc
        return torch.where(x * y > 0, torch.sign(x) * m, torch.zeros_like(x))

    @staticmethod
    def physical(P, d):
        r, u, p = P[0], P[1:4], P[4]
        m = r * u[d]
        e = p / (GAMMA - 1.0) + 0.5 * r * (u * u).sum(0)
        F = [m, m * u[0], m * u[1], m * u[2], (e + p) * u[d]]
        F[1 + d] = F[1 + d] + p
        return torch.stack(F)

    @staticmethod
    def cons(P):
        r, u, p = P[0], P[1:4], P[4]
        return torch.stack([r, r * u[0], r * u[1], r * u[2], p / (GAMMA - 1.0) + 0.5 * r * (u * u).sum(0)])

    @staticmethod
    def prim(U):
        r, u = U[0], U[1:4] / U[0]
        return torch.stack([r, u[0], u[1], u[2], (GAMMA - 1.0) * (U[4] - 0.5 * r * (u * u).sum(0))])

    def riemann(self, L, R, d):
        if self.case["riemann"] == "AUSM+":
            aL, aR = torch.sqrt(GAMMA * L[4] / L[0]), torch.sqrt(GAMMA * R[4] / R[0])
            a = torch.sqrt(aL * aR)
            mL, mR = L[1 + d] / a, R[1 + d] / a
            sub, sup = mL.abs() < 1, mR.abs() < 1
            Mp = torch.where(sub, 0.25 * (mL + 1) ** 2 + 0.125 * (mL * mL - 1) ** 2, 0.5 * (mL + mL.abs()))
            Pp = torch.where(sub, 0.25 * (mL + 1) ** 2 * (2 - mL) + 0.1875 * mL * (mL * mL - 1) ** 2, (mL >= 0).to(mL.dtype))
            Mm = torch.where(sup, -0.25 * (mR - 1) ** 2 - 0.125 * (mR * mR - 1) ** 2, 0.5 * (mR - mR.abs()))
            Pm = torch.where(sup, 0.25 * (mR - 1) ** 2 * (2 + mR) - 0.1875 * mR * (mR * mR - 1) ** 2, (mR < 0).to(mR.dtype))
            M, p = Mp + Mm, Pp * L[4] + Pm * R[4]
            HL = GAMMA / (GAMMA - 1.0) * L[4] / L[0] + 0.5 * (L[1:4] ** 2).sum(0)
            HR = GAMMA / (GAMMA - 1.0) * R[4] / R[0] + 0.5 * (R[1:4] ** 2).sum(0)
            zero = torch.zeros_like(M)
            ml, mr = L[0] * a * torch.maximum(M, zero), R[0] * a * torch.minimum(M, zero)
            F = [ml + mr] + [ml * L[q] + mr * R[q] for q in (1, 2, 3)] + [ml * HL + mr * HR]
            F[1 + d] = F[1 + d] + p
            return torch.stack(F)
        aL, aR = torch.sqrt(GAMMA * L[4] / L[0]), torch.sqrt(GAMMA * R[4] / R[0])
        HL = GAMMA / (GAMMA - 1.0) * L[4] / L[0] + 0.5 * (L[1:4] ** 2).sum(0)
        HR = GAMMA / (GAMMA - 1.0) * R[4] / R[0] + 0.5 * (R[1:4] ** 2).sum(0)
        sL, sR = torch.sqrt(L[0]), torch.sqrt(R[0])
        u = (sL * L[1:4] + sR * R[1:4]) / (sL + sR)
        a = torch.sqrt((GAMMA - 1.0) * ((sL * HL + sR * HR) / (sL + sR) - 0.5 * (u * u).sum(0)))
        zero = torch.zeros_like(a)
        S1 = torch.minimum(zero, torch.minimum(L[1 + d] - aL, u[d] - a))
        S4 = torch.maximum(zero, torch.maximum(R[1 + d] + aR, u[d] + a))
        FL, FR, UL, UR = self.physical(L, d), self.physical(R, d), self.cons(L), self.cons(R)
        if self.case["riemann"] == "HLLE":
            return (S4 * FL - S1 * FR + S1 * S4 * (UR - UL)) / (S4 - S1)
        cl, cr = L[0] * (S1 - L[1 + d]), R[0] * (S4 - R[1 + d])
        Ss = (R[4] - L[4] + cl * L[1 + d] - cr * R[1 + d]) / (cl - cr)
        left = (S1 >= 0) | (Ss >= 0)
        Q, UQ, FQ = torch.where(left, L, R), torch.where(left, UL, UR), torch.where(left, FL, FR)
        S = torch.where(left, S1, S4)
        pstar = L[0] * (L[1 + d] - S1) * (L[1 + d] - Ss) + L[4]
        star = torch.where(left, S1 < 0, S4 > 0)
        inv = 1.0 / torch.where(star, S - Ss, torch.ones_like(S))
        m = (S - Q[1 + d]) * Q[0]
        W = [m, m * Q[1], m * Q[2], m * Q[3], (S - Q[1 + d]) * UQ[4] - Q[4] * Q[1 + d] + pstar * Ss]
        W[1 + d] = W[1 + d] + pstar - Q[4]
        return torch.where(star, FQ + S * (torch.stack(W) * inv - UQ), FQ)

    def mu(self, T, prm):
        return prm[0] * (T / prm[1]) ** 1.5 * (prm[1] + prm[2]) / (T + prm[2])

    def detector(self, X):
        p = X[4]
        kap = 0.0
        for ax in range(3):
            mid = [slice(2, -2)] * 3
            lo, hi = list(mid), list(mid)
            lo[ax], hi[ax] = slice(1, -3), slice(3, -1)
            a, b, q = p[tuple(lo)], p[tuple(hi)], p[tuple(mid)]
            k = ((b - 2.0 * q + a) / (b + 2.0 * q + a)).abs()
            kap = torch.maximum(kap, k) if ax else k
        return torch.where(kap < 0.05, 1.0 - torch.tanh(10.0 * (kap / 20.0) ** 3), torch.zeros_like(kap))

    def viscous(self, X, b, d):
        """Viscous flux through the n + 1 faces of direction d (fully padded periodic block)."""
        h, prm = self.h[b], self.visc[b]
        V = torch.stack([X[1], X[2], X[3], X[4] / (X[0] * RGAS)])
        ax, n = 3 - d, self.dims[b][d]

        def cut(A, shift, lo):      # interior in the other directions (shifted), n + 1 cells from `lo` along d
            at = [slice(None)]
            for a in (1, 2, 3):
                s = shift.get(a, 0)
                at.append(slice(lo, lo + n + 1) if a == ax else slice(2 + s, A.shape[a] - 2 + s))
            return A[tuple(at)]
        G = [None] * 3
        G[d] = (cut(V, {}, 2) - cut(V, {}, 1)) / h[d]
        for e in range(3):
            if e != d:
                t = 3 - e
                G[e] = 0.25 * (cut(V, {t: 1}, 1) - cut(V, {t: -1}, 1) + cut(V, {t: 1}, 2) - cut(V, {t: -1}, 2)) / h[e]
        Pf = 0.5 * (cut(X, {}, 1) + cut(X, {}, 2))
        mu = self.mu(Pf[4] / (Pf[0] * RGAS), prm)
        div = G[0][0] + G[1][1] + G[2][2]
        tau = [mu * (G[d][e] + G[e][d]) for e in range(3)]
        tau[d] = tau[d] - 2.0 / 3.0 * mu * div
        cp = GAMMA * RGAS / (GAMMA - 1.0)
        heat = mu * cp / prm[3] * G[d][3]
        return torch.stack([torch.zeros_like(mu), tau[0], tau[1], tau[2], tau[0] * Pf[1] + tau[1] * Pf[2] + tau[2] * Pf[3] + heat])

    def rate(self, P, b):
        """Residual of block b over its cell volume."""
        X = self.pad(P, b)
        beta = self.detector(X) if self.case["sd"] else None
        out = 0.0
        for d in range(self.ndir):
            ax, n = 3 - d, self.dims[b][d]
            at = [slice(None)] + [slice(None) if a == ax else slice(2, -2) for a in (1, 2, 3)]
            Y = X[tuple(at)]
            dif = Y.narrow(ax, 1, n + 3) - Y.narrow(ax, 0, n + 3)
            half = 0.5 * self.limiter(dif.narrow(ax, 1, n + 2), dif.narrow(ax, 0, n + 2))
            mid = Y.narrow(ax, 1, n + 2)
            hl, hr = half.narrow(ax, 0, n + 1), half.narrow(ax, 1, n + 1)
            if beta is not None:
                w = torch.cat([beta.narrow(ax - 1, 0, 1), beta], ax - 1)
                hl, hr = w * hl, w * hr
            F = self.riemann(mid.narrow(ax, 0, n + 1) + hl, mid.narrow(ax, 1, n + 1) - hr, d)
            for side in range(2):
                if self.face[b, 2 * d + side][0] == 400:
                    Fb = self.physical(P[b].narrow(ax, 0 if side == 0 else n - 1, 1), d)
                    F = torch.cat([Fb, F.narrow(ax, 1, n)] if side == 0 else [F.narrow(ax, 0, n), Fb], ax)
            if b in self.visc:
                F = F - self.viscous(X, b, d)
            out = out + (F.narrow(ax, 1, n) - F.narrow(ax, 0, n)) / self.h[b][d]
        return out

    def smooth(self, R):
        beta = self.case["irs"]
        for ax in (3, 2, 1):
            n = R.shape[ax]
            lo, hi = R.narrow(ax, 0, 1), R.narrow(ax, n - 1, 1)
            S = R
            for _ in range(2):
                S = (R + beta * (torch.cat([lo, S.narrow(ax, 0, n - 1)], ax) + torch.cat([S.narrow(ax, 1, n - 1), hi], ax))) / (1.0 + 2.0 * beta)
            R = S
        return R

    def dt(self, P):
        best = 1e5
        for b, Q in enumerate(P):
            a = torch.sqrt(GAMMA * Q[4] / Q[0])
            for d in range(self.ndir):
                best = min(best, self.cfl * float((self.h[b][d] / (Q[1 + d].abs() + a)).min()))
                if b in self.visc:
                    mu = self.mu(Q[4] / (Q[0] * RGAS), self.visc[b])
                    best = min(best, float((Q[0] * self.h[b][d] ** 2 * self.visc[b][4] / mu).min()))
        return best

    def stage(self, U, Un, c, dt):
        P = [self.prim(u) for u in U]
        out = []
        for b in range(len(U)):
            R = -dt * self.rate(P, b)
            if self.case["irs"] > 0.0:
                R = self.smooth(R)
            out.append(Un[b] + c * (U[b] - Un[b] + R))
        return out


def _to_torch(c, dev):
    return [torch.from_numpy(np.ascontiguousarray(np.moveaxis(abi.interior(b.P), -1, 0))).to(dev) for b in c.blocks]


def _back(x):
    return np.moveaxis(x.detach().cpu().numpy(), 0, -1)


def exact(case, seed):
    # the channel's general metrics are the discretisation's own: no independent value
    if case["flow"] == "bump" or _cells(case) * case["steps"] > 1.1e9:
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    c, bars = _inputs(case, seed)
    s = _Plain(case, c, dev)
    P = _to_torch(c, dev)
    if case["kind"] == "vjp":
        P = [p.requires_grad_(True) for p in P]
        tot = 0.0
        for b, x in enumerate(bars):
            w = torch.from_numpy(np.ascontiguousarray(np.moveaxis(abi.interior(x), -1, 0))).to(dev)
            tot = tot + (w * s.rate(P, b)).sum() * (s.h[b][0] * s.h[b][1] * s.h[b][2])
        return [_back(g) for g in torch.autograd.grad(tot, P)]
    U = [s.cons(p) for p in P]
    if case["kind"] == "march":
        with torch.no_grad():
            for _ in range(case["steps"]):
                P0 = [s.prim(u) for u in U]
                Un, dt = U, s.dt(P0)
                for co in RK[3]:
                    U = s.stage(U, Un, co, dt)
            P = [s.prim(u) for u in U]
            norms = np.sqrt(sum(((p - q) ** 2).sum((1, 2, 3)).cpu().numpy() for p, q in zip(P, P0)))
        states = [_back(p) for p in P]
        return {"states": states, "norms": norms} if len(states) < 60 else states
    # reverse: the adjoint of the stages, one at a time
    dt, vol = _fixed_dt(case), [h[0] * h[1] * h[2] for h in s.h]
    tape = []
    with torch.no_grad():
        for _ in range(case["steps"]):
            Un = U
            for co in RK[3]:
                tape.append((U, Un, co))
                U = s.stage(U, Un, co, dt)
    U = [u.requires_grad_(True) for u in U]
    ke = [0.5 * (u[1:4] ** 2 / u[0]).sum() * v for u, v in zip(U, vol)]
    lam = list(torch.autograd.grad(sum(ke), U))
    lam_n = [torch.zeros_like(x) for x in lam]
    mub = torch.zeros(len(U), dtype=torch.float64, device=dev)
    for Us, Un, co in reversed(tape):
        Us = [u.detach().requires_grad_(True) for u in Us]
        Uc = [u.detach().requires_grad_(True) for u in Un]
        for prm in s.visc.values():
            prm[0] = prm[0].detach().requires_grad_(True)
        mus = [s.visc[b][0] for b in range(len(U))]
        got = torch.autograd.grad(s.stage(Us, Uc, co, dt), Us + Uc + mus, lam)
        nb = len(U)
        mub = mub + torch.stack(got[2 * nb:])
        lam_n = [a + x for a, x in zip(lam_n, got[nb:2 * nb])]
        lam = list(got[:nb])
        if co == RK[3][0]:
            lam = [a + x for a, x in zip(lam, lam_n)]
            lam_n = [torch.zeros_like(x) for x in lam]
    P = [p.requires_grad_(True) for p in P]
    P0b = torch.autograd.grad([s.cons(p) for p in P], P, lam)
    return {"ke": torch.stack(ke).detach().cpu().numpy(), "mu_bar": mub.detach().cpu().numpy(), "P0_bar": [_back(x) for x in P0b]}
