"""Timed cases of the solve-and-sensitivity path, through the entry points that a design program calls.

Kinds of case ("kind" of the dict):

  ku        y = K u on resident vectors (vf_sim_apply_K): the product a program's own Krylov or time loop calls.
  vcycle    s = M^-1 r (vf_mg_precondition) with the hierarchy built: the multigrid preconditioner by itself, for a
            program's own Krylov loop and as the inner block of every solve.
  solve     one design step: new densities, hierarchy, MG-PCG from zero to 1e-8, compliance and sensitivity
            (vf_sim_set_densities, vf_mg_pcg, vf_sim_dot, vf_sim_compliance_gradient), everything on the device.
  chain     the design filters forward and backward: smoothing, Heaviside projection, and both adjoints.
  autograd  compliance and its gradient through CompliancePipeline (filter, projection, solve, backward).
  lbl       LayerByLayerEvaluator.run with the zero guess: all layer solves of a build, objective and gradient.
  planar    the design step on a [1, 1] grid with the full-multigrid preconditioner of the 2D demos.

Densities are smoothed noise (mean 0.3, standard deviation 0.1, clamped to [1e-3, 1]), as designs in progress are; a
smoothing radius r is the hat of support r + 1. Loads and supports are the package's cantilever and MBB beams.
"""
import ctypes
import itertools
import math

import numpy as np
import torch

from voxelfem_amd import capi, optMGLevel, pyVoxelFEM as pv
from voxelfem_amd import workloads as wl
from voxelfem_amd.autograd import CompliancePipeline

DEV = "cuda:0"
NU = 0.3
EMIN = 1e-9
GAMMA = 3.0


def listed():
    return [
        # the smallest product: an odd part-sized grid, bound by the launch
        {"name": "ku_24x17x19", "kind": "ku", "nx": 24, "ny": 17, "nz": 19},
        # the product on the headline grid
        {"name": "ku_384x192x192", "kind": "ku", "nx": 384, "ny": 192, "nz": 192},
        # single-precision V-cycle of a mid-sized design (13M unknowns)
        {"name": "vcycle_fp32_256x128x128", "kind": "vcycle", "nx": 256, "ny": 128, "nz": 128, "precision": "fp32",
         "fmg": False, "nu": 1},
        # double-precision full multigrid cycle with two sweeps (the compliance objective's default preconditioner)
        # on a grid that no tile divides
        {"name": "vcycle_fp64_fmg_176x88x72", "kind": "vcycle", "nx": 176, "ny": 88, "nz": 72, "precision": "fp64",
         "fmg": True, "nu": 2},
        # a small interactive design step, bound by launches and latency
        {"name": "solve_fp64_64x32x32", "kind": "solve", "nx": 64, "ny": 32, "nz": 32, "precision": "fp64",
         "fmg": False, "nu": 1},
        # an ordinary design step in double precision, on sizes that are no power of two
        {"name": "solve_fp64_208x112x96", "kind": "solve", "nx": 208, "ny": 112, "nz": 96, "precision": "fp64",
         "fmg": False, "nu": 1},
        # the headline design step: 43M unknowns, single-precision cycles in the double-precision PCG
        {"name": "solve_fp32_384x192x192", "kind": "solve", "nx": 384, "ny": 192, "nz": 192, "precision": "fp32",
         "fmg": False, "nu": 1},
        # filter chain of the headline design, radius 3
        {"name": "chain_384x192x192_r3", "kind": "chain", "nx": 384, "ny": 192, "nz": 192, "radius": 3, "beta": 8.0},
        # filter chain of a small part with odd sides, radius 2
        {"name": "chain_97x61x45_r2", "kind": "chain", "nx": 97, "ny": 61, "nz": 45, "radius": 2, "beta": 4.0},
        # differentiable compliance of the MBB half-beam, forward and backward
        {"name": "autograd_fp32_128x64x64", "kind": "autograd", "nx": 128, "ny": 64, "nz": 64, "precision": "fp32",
         "radius": 2, "beta": 8.0},
        # all 40 layer solves of a 160x80x80 build
        {"name": "lbl_fp64_160x80x80", "kind": "lbl", "nx": 160, "ny": 80, "nz": 80, "precision": "fp64", "inc": 2},
        # the design step of the 2D demo
        {"name": "planar_384x192", "kind": "planar", "nx": 384, "ny": 192},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mg_grid(rng, most, hi):
    """A grid whose sides are multiples of 8 (16 for the longer ones), at most `most` elements, with a coarsest level
    of the size that the level heuristic aims at."""
    while True:
        nx = 8 * _logint(rng, 4, hi // 8)
        q = 8 if nx <= 96 else 16
        nx = nx // q * q
        ny, nz = (q * max(16 // q, round(min(hi / 2, nx * rng.uniform(0.3, 0.7)) / q)) for _ in range(2))
        if nx * ny * nz <= most and _coarse_unknowns((nx, ny, nz)) < 9000:
            return nx, ny, nz


def _coarse_unknowns(ne):
    lv = optMGLevel(ne, 3)
    return 3 * math.prod((n >> lv) + 1 for n in ne)


def draw(rng):
    kind = rng.choice(["ku", "vcycle", "solve", "solve", "chain", "autograd", "lbl", "planar"])
    if kind == "ku":
        nx = _logint(rng, 16, 380)
        ny, nz = (max(8, min(190, round(nx * rng.uniform(0.3, 0.9)))) for _ in range(2))
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz}
    if kind == "chain":
        nx = _logint(rng, 24, 380)
        ny, nz = (max(12, min(190, round(nx * rng.uniform(0.3, 0.9)))) for _ in range(2))
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "radius": rng.randint(1, 3),
                "beta": float(rng.choice([1, 2, 4, 8]))}
    if kind == "vcycle":
        nx, ny, nz = _mg_grid(rng, 256 * 128 * 128, 256)
        fmg = rng.random() < 0.4
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "precision": rng.choice(["fp64", "fp32"]), "fmg": fmg,
                "nu": 2 if fmg else 1}
    if kind == "solve":
        nx, ny, nz = _mg_grid(rng, 256 * 128 * 128, 256)
        fmg = rng.random() < 0.3
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "precision": rng.choice(["fp64", "fp32"]), "fmg": fmg,
                "nu": 2 if fmg else 1}
    if kind == "autograd":
        nx, ny, nz = _mg_grid(rng, 128 * 64 * 64, 128)
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "precision": rng.choice(["fp64", "fp32"]),
                "radius": rng.randint(1, 3), "beta": float(rng.choice([2, 4, 8]))}
    if kind == "lbl":
        nx = 16 * rng.randint(4, 8)
        ny, nz = 16 * rng.randint(2, 4), 16 * rng.randint(2, 4)
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "precision": rng.choice(["fp64", "fp32"]),
                "inc": rng.choice([2, 3, 4])}
    nx = 16 * _logint(rng, 4, 24)
    return {"kind": "planar", "nx": nx, "ny": 16 * max(2, round(nx / 16 * rng.uniform(0.4, 0.6)))}


# ---- inputs ----------------------------------------------------------------------------------------------------


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _blur(x, passes=3):
    """Box blurs of width 5 along every axis (about a Gaussian of 2.4 voxels)."""
    d = x.dim()
    pool = torch.nn.functional.avg_pool3d if d == 3 else torch.nn.functional.avg_pool2d
    x = x[None, None]
    for _ in range(passes):
        x = pool(x, 5, stride=1, padding=2, count_include_pad=False)
    return x[0, 0]


def _density(ne, seed, mean=0.3, std=0.1):
    z = _blur(torch.rand(ne, dtype=torch.float32, device=DEV, generator=_gen(seed)).double())
    z = (z - z.mean()) / z.std() * std + mean
    return z.clamp(1e-3, 1.0).contiguous()


def _field(ne, seed):
    """A nodal vector field [d, *nn]: smoothed noise plus a little noise of every wavelength, as residuals and
    directions in the middle of a solve are."""
    d = len(ne)
    nn = [n + 1 for n in ne]
    g = _gen(seed + 7919)
    out = torch.empty([d] + nn, dtype=torch.float64, device=DEV)
    for c in range(d):
        r = torch.rand(nn, dtype=torch.float32, device=DEV, generator=g).double() - 0.5
        out[c] = 8.0 * _blur(r, 2) + 0.1 * r
    return out


def _dims(case):
    return (case["nx"], case["ny"], case["nz"]) if "nz" in case else (case["nx"], case["ny"])


def _prec(case):
    return capi.VF_PREC_FP32 if case.get("precision") == "fp32" else capi.VF_PREC_FP64


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def prepare(case, seed):
    kind, ne = case["kind"], _dims(case)
    st = {"kind": kind, "case": case}
    L = capi.lib()
    if kind == "ku":
        tps = wl.configure(pv, ne, wl.CANTILEVER_BC if ne[2] % 2 == 0 else None, None)
        capi.check(L.vf_sim_set_densities(tps._handle(), _p(_density(ne, seed)), capi.VF_DEVICE))
        u = _field(ne, seed)
        st.update(tps=tps, u=u, y=torch.empty_like(u))
    elif kind == "vcycle":
        tps = wl.configure(pv, ne, wl.CANTILEVER_BC, None)
        capi.check(L.vf_sim_set_densities(tps._handle(), _p(_density(ne, seed)), capi.VF_DEVICE))
        mg = tps.multigridSolver(optMGLevel(ne, 3))
        r = _field(ne, seed)
        r[:, 0] = 0  # the residual of a clamped system vanishes on the clamped face
        capi.check(L.vf_mg_update_stiffness(mg._handle()))
        capi.check(L.vf_mg_finish_update(mg._handle()))
        st.update(tps=tps, mg=mg, r=r, s=torch.empty_like(r))
    elif kind in ("solve", "planar"):
        if kind == "solve":
            tps = wl.configure(pv, ne, wl.CANTILEVER_BC, None)
        else:
            tps = wl.configure2d(pv, ne, wl.CANTILEVER2D_BC, None)
        mg = tps.multigridSolver(optMGLevel(ne, len(ne)))
        if kind == "solve":
            mg.useGraphs = True
        f = torch.empty([len(ne)] + [n + 1 for n in ne], dtype=torch.float64, device=DEV)
        capi.check(L.vf_sim_build_load(tps._handle(), _p(f), capi.VF_DEVICE))
        rho = _density(ne, seed)
        st.update(tps=tps, mg=mg, f=f, rho=rho, u=torch.empty_like(f), g=torch.empty_like(rho))
    elif kind == "chain":
        x = _density(ne, seed)
        g = -_density(ne, seed + 104729)  # sensitivities have one sign
        st.update(x=x, gr=g, s=torch.empty_like(x), rho=torch.empty_like(x), t=torch.empty_like(x),
                  gx=torch.empty_like(x), dims=(ctypes.c_int64 * 3)(*ne))
    elif kind == "autograd":
        tps = wl.configure(pv, ne, wl.MBB_BC, None, symmetry_x=True)
        pipe = CompliancePipeline(tps, optMGLevel(ne, 3), rmin=case["radius"] + 1.0, filter_type=1, beta=case["beta"],
                                  tol=1e-8, precision=case["precision"])
        st.update(pipe=pipe, x=_density(ne, seed, mean=0.45, std=0.1).reshape(-1))
    elif kind == "lbl":
        full = wl.configure(pv, ne, None, _density(ne, seed).reshape(-1).cpu().numpy())
        sim = full.getIntermediateFabricationShape(1.0, False, pv.InterpolationLaw.SIMP)
        mg = sim.multigridSolver(optMGLevel(ne, 3))
        ev = pv.LayerByLayerEvaluator(sim)
        ev.selectInitMethod("zero")
        ev.precision = case["precision"]
        st.update(full=full, sim=sim, mg=mg, ev=ev)
    else:
        raise ValueError(kind)
    torch.cuda.synchronize()
    return st


def run(st):
    kind, case = st["kind"], st["case"]
    L = capi.lib()
    if kind == "ku":
        capi.check(L.vf_sim_apply_K(st["tps"]._handle(), _p(st["u"]), _p(st["y"]), capi.VF_DEVICE))
        return st["y"]
    if kind == "vcycle":
        capi.check(L.vf_mg_precondition(ctypes.c_void_p(st["mg"]._handle()), _p(st["r"]), _p(st["s"]), ctypes.c_int64(1),
                                        ctypes.c_int64(case["nu"]), int(case["fmg"]), _prec(case), capi.VF_DEVICE))
        return st["s"]
    if kind in ("solve", "planar"):
        fmg, nu = (True, 2) if kind == "planar" else (case["fmg"], case["nu"])
        sim = st["tps"]._handle()
        capi.check(L.vf_sim_set_densities(sim, _p(st["rho"]), capi.VF_DEVICE))
        st["u"].zero_()
        capi.pcg(st["mg"]._handle(), st["u"].data_ptr(), st["f"].data_ptr(), 1000, 1e-8, 1, nu, fmg, _prec(case))
        c = ctypes.c_double()
        capi.check(L.vf_sim_dot(sim, _p(st["f"]), _p(st["u"]), 0, capi.VF_DEVICE, ctypes.byref(c)))
        capi.check(L.vf_sim_compliance_gradient(sim, _p(st["u"]), _p(st["g"]), capi.VF_DEVICE))
        return {"compliance": 0.5 * c.value, "u": st["u"], "gradient": st["g"]}
    if kind == "chain":
        n, beta, rmin = st["x"].numel(), case["beta"], case["radius"] + 1.0
        capi.check(L.vf_smoothing_filter(st["dims"], rmin, 1, _p(st["x"]), _p(st["s"]), capi.VF_DEVICE, None))
        capi.check(L.vf_projection(beta, n, _p(st["s"]), _p(st["rho"]), capi.VF_DEVICE, None))
        capi.check(L.vf_projection_backprop(beta, n, _p(st["gr"]), _p(st["s"]), _p(st["t"]), capi.VF_DEVICE, None))
        capi.check(L.vf_smoothing_filter(st["dims"], rmin, 1, _p(st["t"]), _p(st["gx"]), capi.VF_DEVICE, None))
        return {"rho": st["rho"], "gradient": st["gx"]}
    if kind == "autograd":
        x = st["x"].clone().requires_grad_(True)
        c = st["pipe"](x)
        c.backward()
        return {"compliance": c.detach(), "gradient": x.grad}
    ev = st["ev"]
    ev.run(st["mg"], True, case["inc"], 1000, 1e-8)
    return {"objective": ev.objective(), "gradient": ev.gradient()}


# ---- what a pass cannot do without -----------------------------------------------------------------------------


def _cycle_work(ne, levels, word, fmg, nu):
    """Least traffic and operations of one cycle: per level, nu sweeps down and up (each reads iterate, right-hand side
    and moduli and writes the iterate; the first down-sweep starts from zero) and one residual; the moduli stand for
    the operators of the coarse levels too. Operations: a node row is 27 blocks of 3 x 3."""
    d = len(ne)
    bytes_, flops = 0.0, 0.0
    for lv in range(levels):
        nn = math.prod((n >> lv) + 1 for n in ne)
        nel = math.prod(n >> lv for n in ne)
        visits = (lv + 1) if fmg else 1
        vec = d * nn * word
        bytes_ += visits * ((2 * nu) * (3 * vec + nel * word) - vec + (3 * vec + nel * word))
        flops += visits * (2 * nu + 1) * 2 * d * d * 3 ** d * nn
    return bytes_, flops


def work(case):
    kind, ne = case["kind"], _dims(case)
    d = len(ne)
    nn, nel = math.prod(n + 1 for n in ne), math.prod(ne)
    vec = 8.0 * d * nn
    ku_b, ku_f = 2 * vec + 8.0 * nel, 2.0 * 9 * 2 * 48 * nel if d == 3 else 2.0 * 64 * nel
    if kind == "ku":
        return {"bytes": ku_b, "flops": 240.0 * nel}
    if kind == "chain":
        taps = (2 * case["radius"] + 1) ** 3 * 0.55  # voxels within the hat's support
        return {"bytes": 8.0 * nel * 6, "flops": 2 * 2 * taps * nel}
    levels = optMGLevel(ne, d)
    word = 4.0 if case.get("precision") == "fp32" else 8.0
    fmg, nu = (True, 2) if kind == "planar" else (case.get("fmg", False), case.get("nu", 1))
    cyc_b, cyc_f = _cycle_work(ne, levels, word, fmg, nu)
    if kind == "vcycle":
        return {"bytes": cyc_b, "flops": cyc_f}
    # about ten iterations to 1e-8: the cycle, K d, and the vector updates (x, r, d read and written, s and K d read)
    its = 10
    it_b, it_f = cyc_b + ku_b + 8 * vec, cyc_f + ku_f
    if kind == "lbl":  # the layers' structures fill half the grid on average
        layers = -(-ne[1] // case["inc"])
        return {"bytes": 0.5 * layers * 15 * it_b, "flops": 0.5 * layers * 15 * it_f}
    return {"bytes": its * it_b + vec + 16.0 * nel, "flops": its * it_f}


def tolerance(case):
    """About four times what the path differs by from the 64-bit reference below."""
    kind = case["kind"]
    if kind in ("ku", "chain"):  # measured 1e-16 to 6e-16
        return {"rel": 4e-15, "max": 1e-13}
    if kind == "vcycle":  # measured 8e-14 (the coarsest solve's conditioning) and 7e-8
        return {"rel": 1e-12, "max": 1e-10} if case["precision"] == "fp64" else {"rel": 1e-6, "max": 1e-4}
    # solves stop at a relative residual of 1e-8, which leaves u and its sensitivity up to 2e-9 off; a sum in another
    # order can move the stop by one iteration, which gains or loses about a factor of ten
    return {"rel": 1e-7, "max": 1e-5}


# ---- the same in 64 bits with plain torch ----------------------------------------------------------------------


def _k0(d, nu=NU):
    """Unit element stiffness by two-point Gauss quadrature (2D: plane stress), DoF order (node, component)."""
    mu = 1 / (2 * (1 + nu))
    lam = nu / ((1 + nu) * (1 - 2 * nu)) if d == 3 else nu / ((1 + nu) * (1 - nu))
    corners = list(itertools.product((0, 1), repeat=d))
    n = len(corners)
    K = np.zeros((n * d, n * d))
    a = 0.5 / math.sqrt(3)
    for q in itertools.product((0.5 - a, 0.5 + a), repeat=d):
        G = np.zeros((n, d))
        for i, c in enumerate(corners):
            for k in range(d):
                G[i, k] = math.prod((1.0 if c[m] else -1.0) if m == k else (q[m] if c[m] else 1 - q[m]) for m in range(d))
        g = G @ G.T
        for i in range(n):
            for j in range(n):
                B = lam * np.outer(G[i], G[j]) + mu * np.outer(G[j], G[i]) + mu * g[i, j] * np.eye(d)
                K[i * d:(i + 1) * d, j * d:(j + 1) * d] += B / 2 ** d
    return torch.tensor(K, dtype=torch.float64, device=DEV)


class _Reference:
    """The multigrid hierarchy of one density field, each level an array of element matrices (the finest: one matrix
    scaled by the moduli); `free` marks unconstrained components."""

    def __init__(self, E, free, levels):
        d = self.d = E.dim()
        self.corners = list(itertools.product((0, 1), repeat=d))
        K0 = _k0(d)
        self.ops, self.free = [(K0, E)], [free]
        P = [self._child(c) for c in self.corners]
        for lv in range(levels):
            K, Em = self.ops[-1]
            out = 0
            for c, p in zip(self.corners, P):
                sl = tuple(slice(k, None, 2) for k in c)
                if lv == 0:
                    out = out + (p.T @ K @ p)[(...,) + (None,) * d] * Em[sl]
                else:
                    sub = K[(slice(None), slice(None)) + sl]
                    shape, n = sub.shape, sub.shape[0]
                    t = (p.T @ sub.reshape(n, -1)).reshape(n, n, -1).transpose(0, 1).reshape(n, -1)
                    out = out + (p.T @ t).reshape(n, n, -1).transpose(0, 1).reshape(shape)
            self.ops.append((out, None))
            self.free.append(self.free[-1][(slice(None),) + (slice(None, None, 2),) * d])
        self.Dinv = [self._diag_inverse(i) for i in range(levels)]
        self._factor()

    def _child(self, child):
        """Interpolation of a coarse element's DoFs to child element `child`."""
        d, n = self.d, len(self.corners)
        P = np.zeros((n * d, n * d))
        for i, f in enumerate(self.corners):
            for j, c in enumerate(self.corners):
                x = [0.5 * (a + b) for a, b in zip(child, f)]
                w = math.prod(x[k] if c[k] else 1 - x[k] for k in range(d))
                for k in range(d):
                    P[i * d + k, j * d + k] = w
        return torch.tensor(P, dtype=torch.float64, device=DEV)

    def _slices(self, shape):
        return [(slice(None),) + tuple(slice(c, c + n) for c, n in zip(cor, shape)) for cor in self.corners]

    def apply(self, lv, u):
        K, E = self.ops[lv]
        ne = [n - 1 for n in u.shape[1:]]
        sl = self._slices(ne)
        ue = torch.cat([u[s] for s in sl])
        if E is not None:
            fe = (K @ ue.reshape(ue.shape[0], -1)).reshape(ue.shape) * E
        else:
            fe = torch.stack([(K[i] * ue).sum(0) for i in range(K.shape[0])])
        y = torch.zeros_like(u)
        for k, s in enumerate(sl):
            y[s] += fe[self.d * k:self.d * (k + 1)]
        return y * self.free[lv]

    def _diag_inverse(self, lv):
        d, (K, E) = self.d, self.ops[lv]
        nn = self.free[lv].shape[1:]
        ne = [n - 1 for n in nn]
        A = torch.zeros([d, d] + list(nn), dtype=torch.float64, device=DEV)
        for k, s in enumerate(self._slices(ne)):
            blk = K[d * k:d * (k + 1), d * k:d * (k + 1)]
            A[(slice(None),) + s] += blk[(...,) + (None,) * d] * E if E is not None else blk
        f = self.free[lv]
        A = A * f[None] * f[:, None]
        for c in range(d):
            A[c, c] += 1 - f[c]
        if d == 2:
            det = A[0, 0] * A[1, 1] - A[0, 1] * A[1, 0]
            adj = torch.stack([torch.stack([A[1, 1], -A[0, 1]]), torch.stack([-A[1, 0], A[0, 0]])])
        else:
            cof = [[A[(i + 1) % 3, (j + 1) % 3] * A[(i + 2) % 3, (j + 2) % 3]
                    - A[(i + 1) % 3, (j + 2) % 3] * A[(i + 2) % 3, (j + 1) % 3] for i in range(3)] for j in range(3)]
            adj = torch.stack([torch.stack(r) for r in cof])
            det = sum(A[0, k] * adj[k, 0] for k in range(3))
        return adj / det * f[None] * f[:, None]

    def _factor(self):
        K, E = self.ops[-1]
        nn = list(self.free[-1].shape[1:])
        ne, d = [n - 1 for n in nn], self.d
        ids = torch.arange(d * math.prod(nn), device=DEV).reshape([d] + nn)
        m = torch.cat([ids[s] for s in self._slices(ne)]).reshape(d * len(self.corners), -1)
        Kf = (K[(...,) + (None,) * d] * E).reshape(K.shape[0], K.shape[1], -1) if E is not None else K.reshape(
            K.shape[0], K.shape[1], -1)
        N = ids.numel()
        A = torch.zeros(N * N, dtype=torch.float64, device=DEV)
        for i in range(m.shape[0]):
            for j in range(m.shape[0]):
                A.index_add_(0, m[i] * N + m[j], Kf[i, j])
        keep = self.free[-1].reshape(-1).nonzero()[:, 0]
        A = A.reshape(N, N)[keep][:, keep].cpu()
        self.keep, self.chol = keep, torch.linalg.cholesky(0.5 * (A + A.T))

    def coarse(self, b):
        x = torch.zeros_like(b).reshape(-1)
        rhs = b.reshape(-1)[self.keep].cpu()[:, None]
        x[self.keep] = torch.cholesky_solve(rhs, self.chol)[:, 0].to(DEV)
        return x.reshape(b.shape)

    def sweep(self, lv, u, b, forward):
        colours = self.corners if forward else self.corners[::-1]
        for c in colours:
            s = (slice(None),) + tuple(slice(k, None, 2) for k in c)
            r = (b - self.apply(lv, u))[s]
            u[s] += (self.Dinv[lv][(slice(None),) + s] * r[None]).sum(1)

    def restrict(self, f):
        for ax in range(1, self.d + 1):
            n = f.shape[ax]
            ev = f.index_select(ax, torch.arange(0, n, 2, device=DEV))
            od = 0.5 * f.index_select(ax, torch.arange(1, n, 2, device=DEV))
            m = ev.shape[ax]
            ev.narrow(ax, 0, m - 1).add_(od)
            ev.narrow(ax, 1, m - 1).add_(od)
            f = ev
        return f

    def interpolate(self, c):
        for ax in range(1, self.d + 1):
            m = c.shape[ax]
            shape = list(c.shape)
            shape[ax] = 2 * m - 1
            f = torch.empty(shape, dtype=c.dtype, device=DEV)
            idx = [slice(None)] * (self.d + 1)
            idx[ax] = slice(0, None, 2)
            f[tuple(idx)] = c
            idx[ax] = slice(1, None, 2)
            f[tuple(idx)] = 0.5 * (c.narrow(ax, 0, m - 1) + c.narrow(ax, 1, m - 1))
            c = f
        return c

    def vcycle(self, lv, u, b, nu):
        if lv == len(self.ops) - 1:
            return self.coarse(b)
        for _ in range(nu):
            self.sweep(lv, u, b, True)
        r = b * self.free[lv] - self.apply(lv, u)
        rc = self.restrict(r)
        u += self.interpolate(self.vcycle(lv + 1, torch.zeros_like(rc), rc, nu)) * self.free[lv]
        for _ in range(nu):
            self.sweep(lv, u, b, False)
        return u

    def fmg(self, lv, b, nu):
        if lv == len(self.ops) - 1:
            return self.coarse(b)
        u = self.interpolate(self.fmg(lv + 1, self.restrict(b), nu)) * self.free[lv]
        return self.vcycle(lv, u, b, nu)

    def solve(self, f, tol=1e-13, most=120):
        b = f * self.free[0]
        x, r = torch.zeros_like(b), b.clone()
        d, rz, bn = None, None, b.norm()
        for _ in range(most):
            if r.norm() <= tol * bn:
                break
            s = self.vcycle(0, torch.zeros_like(r), r, 1)
            rz, old = (r * s).sum(), rz
            d = s if d is None else s + rz / old * d
            q = self.apply(0, d)
            a = rz / (d * q).sum()
            x, r = x + a * d, r - a * q
        return x


def _supports(case):
    """(free components, load) of the kind's beam."""
    ne = _dims(case)
    d, nn = len(ne), [n + 1 for n in ne]
    free = torch.ones([d] + nn, dtype=torch.float64, device=DEV)
    f = torch.zeros_like(free)
    if case["kind"] == "autograd":
        free[0, 0] = 0
        free[1:, -1, 0] = 0
        f[1, 0, -1] = -1.0 / nn[2]
    elif d == 3:
        free[:, 0] = 0
        f[2, -1, :, ne[2] // 2] = -1.0 / nn[1]
    else:
        free[:, 0] = 0
        f[1, -1, 0] = -1.0
    return free, f


def _modulus(rho):
    return EMIN + rho ** GAMMA * (1 - EMIN)


def _gradient(rho, u):
    d = rho.dim()
    corners = itertools.product((0, 1), repeat=d)
    ue = torch.cat([u[(slice(None),) + tuple(slice(c, c + n) for c, n in zip(cor, rho.shape))] for cor in corners])
    ue = ue.reshape(ue.shape[0], -1)
    e = ((_k0(d) @ ue) * ue).sum(0).reshape(rho.shape)
    return -0.5 * GAMMA * rho ** (GAMMA - 1) * (1 - EMIN) * e


def _smooth(x, radius):
    rmin, R = radius + 1.0, radius
    for ax in range(x.dim()):  # mirrored with the edge value repeated
        n = x.shape[ax]
        at = torch.arange(-R, n + R, device=DEV)
        at = torch.where(at < 0, -at - 1, torch.where(at >= n, 2 * n - 1 - at, at))
        x = x.index_select(ax, at)
    out, W = 0, 0.0
    shape = [n - 2 * R for n in x.shape]
    for o in itertools.product(range(-R, R + 1), repeat=x.dim()):
        w = rmin - math.sqrt(sum(k * k for k in o))
        if w > 0:
            out = out + w * x[tuple(slice(k + R, k + R + n) for k, n in zip(o, shape))]
            W += w
    return out / W


def exact(case, seed):
    kind, ne = case["kind"], _dims(case)
    if kind == "lbl" or math.prod(ne) > 5_000_000 and kind not in ("ku", "chain"):
        return None
    if kind == "ku":
        free = torch.ones([3] + [n + 1 for n in ne], dtype=torch.float64, device=DEV)
        ref = _Reference.__new__(_Reference)
        ref.d, ref.corners = 3, list(itertools.product((0, 1), repeat=3))
        ref.ops, ref.free = [(_k0(3), _modulus(_density(ne, seed)))], [free]
        return ref.apply(0, _field(ne, seed))
    if kind == "chain":
        s = _smooth(_density(ne, seed), case["radius"])
        th, t = math.tanh(case["beta"] / 2), torch.tanh(case["beta"] * (s - 0.5))
        g = -_density(ne, seed + 104729) * case["beta"] * (1 - t * t) / (2 * th)
        return {"rho": (th + t) / (2 * th), "gradient": _smooth(g, case["radius"])}
    free, f = _supports(case)
    levels = optMGLevel(ne, len(ne))
    if kind == "vcycle":
        ref = _Reference(_modulus(_density(ne, seed)), free, levels)
        r = _field(ne, seed)
        r[:, 0] = 0
        return ref.fmg(0, r, case["nu"]) if case["fmg"] else ref.vcycle(0, torch.zeros_like(r), r, case["nu"])
    if kind == "autograd":
        s = _smooth(_density(ne, seed, mean=0.45, std=0.1), case["radius"])
        th, t = math.tanh(case["beta"] / 2), torch.tanh(case["beta"] * (s - 0.5))
        rho = (th + t) / (2 * th)
    else:
        rho = _density(ne, seed)
    u = _Reference(_modulus(rho), free, levels).solve(f)
    c, g = 0.5 * float((f * u).sum()), _gradient(rho, u)
    if kind == "autograd":
        g = _smooth(g * case["beta"] * (1 - t * t) / (2 * th), case["radius"])
        return {"compliance": torch.tensor(c, dtype=torch.float64), "gradient": g.reshape(-1)}
    return {"compliance": c, "u": u, "gradient": g}
