"""Performance cases: the calls a user of tetmag_amd makes, over the range of meshes and batches it is used on.

A case is a dict of plain values: what is called (``kind``), the mesh (a Kuhn cuboid of nx x ny x nz cells or a layered
prism disk), the material terms switched on and the sizes of the call.  ``prepare`` builds what a program has in hand
before the call (mesh, operators, context, batch, magnetisation), ``run`` makes one call and returns its outputs.

Magnetisations move from pass to pass, as along a trajectory: the demag solves then start from what earlier solves
left, as they do in use.  The cold solves have right-hand sides that have nothing to do with each other.
"""
import ctypes as C
import functools
import math

import numpy as np
import torch

from tetmag_amd import _native as N
from tetmag_amd import mesh as M
from tetmag_amd import problem as P

MU0 = 4e-7 * math.pi
PRECISIONS = {"fp64": N.TM_PREC_FP64, "mixed": N.TM_PREC_MIXED, "mixed-int8": N.TM_PREC_MIXED_BEMI8}


def listed():
    c2k = {"mesh": "cuboid", "nx": 20, "ny": 20, "nz": 4, "h": 5.0, "jitter": 0.0}
    c283k = {"mesh": "cuboid", "nx": 128, "ny": 128, "nz": 16, "h": 3.0, "jitter": 0.1, "ku": True}
    disk26k = {"mesh": "disk", "diameter": 200.0, "thickness": 10.0, "h": 2.5}
    return [
        # the smallest use: a host program (TheLLG) that asks the GPU classes for one field after the other on host
        # arrays, 2,205 nodes (latency, launches, small copies)
        {"name": "classes-2k", "kind": "classes", **c2k, "ku": True, "dmi": True},
        # one sparse product on device vectors at the benchmark mesh (282,897 nodes): SpMatCUDA::mvp
        {"name": "spmv-283k", "kind": "spmv", **c283k},
        # an initial solve, or one whose right-hand side has nothing to do with the last (a new state, a line search):
        # the Neumann system of 71,825 nodes from zero
        {"name": "solve-72k", "kind": "solve", "mesh": "cuboid", "nx": 64, "ny": 64, "nz": 16, "h": 3.0, "jitter": 0.1},
        # fixed-step relaxation of a small element, ten steps between two records of m
        {"name": "rk4-2k", "kind": "rk4", **c2k, "steps": 10, "fs": 20.0},
        # adaptive integration of a thin disk over one recording interval
        {"name": "ode-26k", "kind": "ode", **disk26k, "fs": 400.0},
        # right-hand sides for an integrator on the host, bulk DMI, an odd mesh of 29,760 nodes
        {"name": "rhs-30k", "kind": "rhs", "mesh": "cuboid", "nx": 61, "ny": 47, "nz": 9, "h": 3.0, "jitter": 0.1,
         "ku": True, "dmi": True, "fs": 20.0},
        # the same at the benchmark mesh: the dense boundary matrix is 13.4 GB
        {"name": "rhs-283k", "kind": "rhs", **c283k, "fs": 20.0},
        # gradients through one RK4 step (forward and backward) of a skyrmion film with interfacial DMI
        {"name": "vjp-24k", "kind": "vjp", "mesh": "disk", "diameter": 60.0, "thickness": 1.0, "h": 0.6, "ku": True,
         "idmi": True, "fs": 2.5},
        # the benchmark: 64 states advanced together, boundary product from int8 digits
        {"name": "batch64-283k", "kind": "batch", **c283k, "samples": 64, "precision": "mixed-int8", "fs": 20.0},
        # a hysteresis loop's 64 field values advanced together, two RK4 steps
        {"name": "batch64-rk4-26k", "kind": "batch_rk4", **disk26k, "samples": 64, "precision": "mixed", "steps": 2,
         "fs": 50.0},
        # a batch that does not fill 64 samples, all in FP64, fields wanted too
        {"name": "batch24-38k", "kind": "batch", "mesh": "cuboid", "nx": 64, "ny": 64, "nz": 8, "h": 3.0,
         "jitter": 0.1, "ku": True, "samples": 24, "precision": "fp64", "heff": True, "fs": 20.0},
        # a few samples of a small element (finite differences over parameters)
        {"name": "batch7-2k", "kind": "batch", **c2k, "samples": 7, "precision": "mixed", "fs": 20.0},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["classes", "spmv", "solve", "rk4", "ode", "rhs", "rhs", "vjp", "batch", "batch", "batch_rk4"])
    top = {"classes": 20000, "spmv": 280000, "solve": 100000, "rk4": 12000, "ode": 30000, "rhs": 90000, "vjp": 24000,
           "batch": 45000, "batch_rk4": 20000}[kind]
    case = {"kind": kind}
    if kind in ("ode", "vjp", "batch_rk4") and rng.random() < 0.6:
        if kind == "vjp":
            case.update(mesh="disk", diameter=round(rng.uniform(20.0, 60.0), 1), thickness=1.0, h=0.6)
        else:
            case.update(mesh="disk", diameter=round(rng.uniform(60.0, 180.0), 1), thickness=10.0, h=2.5)
    else:
        n = _log_int(rng, 1500, top)
        nz = rng.randint(3, max(3, min(17, int(n ** (1 / 3)))))
        a = math.sqrt(n / (nz + 1.0))
        nx = max(4, int(a * math.exp(rng.uniform(-0.4, 0.4))))
        ny = max(4, int(n / ((nz + 1.0) * (nx + 1.0))))
        case.update(mesh="cuboid", nx=nx, ny=ny, nz=nz, h=rng.choice([3.0, 4.0, 5.0]), jitter=0.1)
    if kind in ("classes", "rhs", "rk4"):
        case["dmi"] = kind == "classes" or rng.random() < 0.3
    case["ku"] = kind in ("classes", "vjp") or rng.random() < 0.5
    if kind == "vjp":
        case["idmi"] = case["mesh"] == "disk"
        case["fs"] = 2.5
    elif kind == "ode":
        case["fs"] = round(rng.uniform(150.0, 400.0), 1)
    elif kind == "batch_rk4":
        case["fs"] = 20.0
    elif kind in ("rk4", "rhs", "batch"):
        case["fs"] = 20.0
    if kind == "rk4":
        case["steps"] = rng.randint(5, 20)
    if kind.startswith("batch"):
        case["samples"] = rng.choice([64, rng.randint(2, 63)])
        case["precision"] = rng.choice(["mixed", "mixed-int8", "fp64"])
        if kind == "batch":
            case["heff"] = rng.random() < 0.3
        else:
            case["steps"] = rng.randint(1, 3)
    return case


# -- meshes and inputs ---------------------------------------------------------
@functools.lru_cache(maxsize=4)
def _problem_of(key):
    c = dict(key)
    skyrmion = bool(c.get("idmi"))
    mat = P.Material(Ms=1.1e6 if skyrmion else 8.0e5, A=1.6e-11 if skyrmion else 1.3e-11,
                     Ku=(8e5 if skyrmion else 5e4) if c.get("ku") else 0.0,
                     ku_axis=(0.0, 0.0, 1.0) if skyrmion else (0.36, 0.48, 0.8), D=1e-3 if c.get("dmi") else 0.0,
                     Di=3e-3 if skyrmion else 0.0, alpha=0.3 if skyrmion else 0.5, B_ext=(0.02, -0.01, 0.03))
    if c["mesh"] == "disk":
        return P.mesh_problem("disk", M.disk_prism(c["diameter"], c["thickness"], c["h"], 0.15, 2027), mat, "vortex")
    return P.cuboid_problem("cuboid", c["nx"], c["ny"], c["nz"], c["h"], c["jitter"], 2025, mat, "vortex", True)


def _problem(case):
    """The mesh and its operators: a program reads its mesh once."""
    keys = ("mesh", "nx", "ny", "nz", "h", "jitter", "diameter", "thickness", "ku", "dmi", "idmi")
    return _problem_of(tuple((k, case[k]) for k in keys if k in case))


def _smooth(prob, samples, seed, dev):
    """(3, n, S) smooth unit fields: normalised sums of eight plane waves (wavelengths 20 to 200 mesh units)."""
    g = torch.Generator().manual_seed(int(seed))
    xyz = torch.from_numpy(prob.mesh.xyz).to(dev)
    out = torch.empty((3, prob.n, samples), dtype=torch.float64, device=dev)
    for s in range(samples):
        u = torch.rand((8, 8), generator=g, dtype=torch.float64)
        ct, ph = 2 * u[:, 2] - 1, 2 * math.pi * u[:, 1]
        st = torch.sqrt(1 - ct * ct)
        q = torch.stack([st * torch.cos(ph), st * torch.sin(ph), ct]) * (2 * math.pi / (20.0 + 180.0 * u[:, 0]))
        a = (2 * u[:, 4:7] - 1).to(dev)
        v = (torch.cos(xyz @ q.to(dev) + (2 * math.pi * u[:, 3]).to(dev)) @ a).T
        out[:, :, s] = v / torch.linalg.vector_norm(v, dim=0, keepdim=True)
    return out


def _tau(prob, fs):
    return 1e-3 * fs * prob.time_scale()


def _fields(case, prob):
    """(3, S) applied fields of a batch, A/m: a sweep along x."""
    s = case["samples"]
    return np.stack([np.linspace(-0.08, 0.08, s), np.full(s, 0.004), np.zeros(s)]) / MU0


def _context(case, prob):
    from tetmag_amd.context import FieldContext
    # the large matrix in the default (reference) form of the solid angle, the others in the one that keeps all digits
    return FieldContext(prob, bem_formula=N.TM_BEM_REFERENCE if prob.n > 100000 else N.TM_BEM_ACCURATE)


class _Handle:
    """A solver of the C interface."""

    def __init__(self, rp, col, val):
        self.h = C.c_void_p()
        N.check(N.lib().tm_solver_create(len(rp) - 1, N.ptr(rp), N.ptr(col), N.ptr(val), N.TM_PRECOND_AMG,
                                         C.byref(self.h)), "tm_solver_create")

    def __del__(self):
        if self.h:
            N.lib().tm_solver_destroy(self.h)


def _csr(prob, values):
    return values, prob.ops.col, prob.ops.rowptr


def prepare(case, seed):
    prob, kind = _problem(case), case["kind"]
    dev = torch.device("cuda")
    s = {"case": case, "prob": prob}
    if kind == "classes":
        from tetmag_amd.gpu import EffFieldGPU
        e = EffFieldGPU(prob.n)
        e.init(prob.n)
        o = prob.ops
        e.setExchangeMatOnDev(_csr(prob, prob.exchange_values()))
        e.setGradientMatsOnDev(_csr(prob, -o.tgx), _csr(prob, -o.tgy), _csr(prob, -o.tgz))
        e.setUniaxialAnisotropy(prob.kaxis, prob.Ku)
        e.setDMIdata(prob.D, 1.0 / o.nodevol, prob.bnd.node_normal, prob.bnd.node_area)
        s["eff"] = e
        s["m"] = [np.ascontiguousarray(_smooth(prob, 1, 7 * seed + k, dev)[:, :, 0].T.cpu().numpy()) for k in range(4)]
        s["at"] = 0
    elif kind == "spmv":
        from tetmag_amd.gpu import SpMatCUDA
        s["A"] = SpMatCUDA(_csr(prob, prob.exchange_values()))
        g = torch.Generator(device=dev).manual_seed(seed)
        s["x"] = torch.randn(prob.n, generator=g, dtype=torch.float64, device=dev)
    elif kind == "solve":
        rp, col, val = prob.neumann_matrix()
        s["solver"] = _Handle(N.i32(rp), N.i32(col), N.f64(val))
        s["b"] = [_charge(prob, _smooth(prob, 1, 7 * seed + k, dev))[:, 0].contiguous() for k in range(3)]
        s["x"] = torch.zeros(prob.n, dtype=torch.float64, device=dev)
        s["at"] = 0
    elif kind in ("rk4", "ode", "rhs"):
        s["ctx"] = _context(case, prob)
        s["ctx"].set_mag(_smooth(prob, 1, seed, dev)[:, :, 0].reshape(-1).contiguous())
        s["m"] = torch.empty(3 * prob.n, dtype=torch.float64, device=dev)
        s["h"] = 0.0
    elif kind == "vjp":
        s["ctx"] = _context(case, prob)
        s["m"] = _smooth(prob, 1, seed, dev)[:, :, 0].reshape(-1).contiguous()
        s["w"] = _smooth(prob, 1, seed + 1, dev)[:, :, 0].reshape(-1).contiguous()
        s["hext"] = torch.tensor(prob.hext, dtype=torch.float64, device=dev, requires_grad=True)
        s["ku"] = torch.tensor(prob.Ku, dtype=torch.float64, device=dev, requires_grad=True) if case.get("ku") else None
        s["di"] = torch.tensor(prob.Di, dtype=torch.float64, device=dev, requires_grad=True) if case.get("idmi") else None
    else:
        from tetmag_amd.batch import BatchContext
        s["ctx"] = _context(case, prob)
        b = s["batch"] = BatchContext(s["ctx"], case["samples"], PRECISIONS[case["precision"]])
        b.set_zeeman(_fields(case, prob))
        m = _smooth(prob, case["samples"], seed, dev)
        torch.cuda.synchronize()
        b.set_mag(m)
        s["m"] = m
    torch.cuda.synchronize()
    return s


def run(s):
    case, kind, prob = s["case"], s["case"]["kind"], s["prob"]
    if kind == "classes":
        e = s["eff"]
        m = s["m"][s["at"] % 4]
        s["at"] += 1
        e.setMagDev(m)
        hx, hu, hd = e.ExchangeFieldGPU(), e.UniaxialAnisotropyField(), e.DMIField()
        H = (hx + hu + hd) / prob.mat.Js
        return {"exchange": hx, "uniaxial": hu, "dmi": hd, "dmdt": e.ClassicLLG_hst(H, prob.alpha),
                "torque": e.MaxTorque(H)}
    if kind == "spmv":
        return s["A"].mvp(s["x"])
    if kind == "solve":
        b = s["b"][s["at"] % 3]
        s["at"] += 1
        N.check(N.lib().tm_solver_solve(s["solver"].h, N.ptr(b), N.TM_DEVICE, N.ptr(s["x"]), N.TM_DEVICE, 1e-10, 10000,
                                        0, None, None), "tm_solver_solve")
        return s["x"]
    if kind == "rhs":
        ctx = s["ctx"]
        ctx.eval_rhs(want_heff=True, stats=False)
        ctx.step_euler(_tau(prob, case["fs"]))
        return {"dmdt": ctx.dmdt, "heff": ctx.heff}
    if kind in ("rk4", "ode"):
        ctx = s["ctx"]
        if kind == "rk4":
            ctx.run_rk4(_tau(prob, case["fs"]), case["steps"])
        else:
            s["h"] = ctx.integrate(_tau(prob, case["fs"]), h0=s["h"])["h_next"]
        N.check(N.lib().tm_ctx_get_mag(ctx.h, N.ptr(s["m"]), N.TM_DEVICE), "tm_ctx_get_mag")
        return s["m"]
    if kind == "vjp":
        from tetmag_amd import autograd as A
        m = s["m"].detach().requires_grad_(True)
        wrt = {"m": m, "hext": s["hext"], "ku": s["ku"], "di": s["di"]}
        wrt = {k: t for k, t in wrt.items() if t is not None}
        m1 = A.rk4_step(s["ctx"], m, _tau(prob, case["fs"]), s["hext"], s["ku"], None, di=s["di"])
        grads = torch.autograd.grad((m1 * s["w"]).sum(), list(wrt.values()))
        s["m"] = m1.detach()
        return {"m1": s["m"], **{"grad_" + k: g for k, g in zip(wrt, grads)}}
    b = s["batch"]
    if kind == "batch_rk4":
        b.run_rk4(_tau(prob, case["fs"]), case["steps"], use_graph=True)
        N.check(N.lib().tm_batch_get_mag(b.h, N.ptr(s["m"]), N.TM_DEVICE), "tm_batch_get_mag")
        return s["m"]
    if case.get("heff"):
        b.eval_rhs(want_heff=True, stats=False)
        b.step_euler(_tau(prob, case["fs"]))
        return {"dmdt": b.dmdt, "heff": b.heff}
    return b.eval_euler(_tau(prob, case["fs"]), stats=False)


def work(case):
    """Operators, boundary matrix and vectors read or written once per right-hand side; each demag solve as one pass
    over its matrix."""
    prob, kind = _problem(case), case["kind"]
    n, nnz, b = prob.n, prob.ops.nnz, prob.bnd.bnx
    s = case.get("samples", 1)
    if kind == "classes":
        return {"bytes": nnz * 36.0 + n * 8.0 * 35, "flops": nnz * 2.0 * 9 + n * 60.0}
    if kind == "spmv":
        return {"bytes": nnz * 12.0 + n * 16.0, "flops": nnz * 2.0}
    if kind == "solve":
        return {"bytes": nnz * 12.0 + n * 24.0, "flops": nnz * 2.0}
    ops = 4 + 3 * bool(case.get("dmi")) + 3
    b_entry = 5.0 if case.get("precision") == "mixed-int8" else 8.0
    once = {"bytes": b_entry * b * b + nnz * (4.0 + 8.0 * ops) + 2 * nnz * 12.0 + n * s * 8.0 * 16 + n * 8.0 * 6,
            "flops": (2.0 * b * b + nnz * 2.0 * (3 * ops + 2) + n * 60.0) * s}
    times = {"rhs": 1, "batch": 1, "vjp": 8}.get(kind) or (4 * case["steps"] if "steps" in case else 6 * case["fs"] / 50)
    return {k: v * times for k, v in once.items()}


# -- the same from the definitions, in 64 bits -----------------------------------
class _Fem:
    """P1 elements, the double layer and the demag problem from their definitions (dense boundary matrix, conjugate
    gradients to rounding)."""

    def __init__(self, prob, demag=True):
        self.prob = prob
        self.dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        self.n = prob.n
        xyz = torch.from_numpy(prob.mesh.xyz).to(self.dev)
        fel = torch.from_numpy(prob.mesh.fel.astype(np.int64)).to(self.dev)
        X = xyz[fel]
        J = X[:, 1:] - X[:, :1]
        inv = torch.linalg.inv(J)  # columns: gradients of the last three shape functions
        g = torch.cat([-inv.sum(2, keepdim=True), inv], 2).transpose(1, 2).contiguous()
        vol = torch.linalg.det(J).abs() / 6.0
        self.fel, self.g, self.vol = fel, g, vol
        self.node_vol = torch.zeros(self.n, dtype=torch.float64, device=self.dev).index_add(
            0, fel.reshape(-1), (vol / 4).repeat_interleave(4))
        k = torch.einsum("eid,ejd->eij", g, g) * vol[:, None, None]
        i = fel[:, :, None].expand(-1, 4, 4).reshape(-1)
        j = fel[:, None, :].expand(-1, 4, 4).reshape(-1)
        K = torch.sparse_coo_tensor(torch.stack([i, j]), k.reshape(-1), (self.n, self.n)).coalesce()
        self.K = K.to_sparse_csr()
        ii = K.indices()
        self.diag = torch.zeros(self.n, dtype=torch.float64, device=self.dev)
        on = ii[0] == ii[1]
        self.diag[ii[0][on]] = K.values()[on]
        if demag:
            self._boundary(xyz, X)

    def _sum(self, v):  # (t, 4, S) -> (n, S)
        out = torch.zeros((self.n, v.shape[2]), dtype=torch.float64, device=self.dev)
        return out.index_add(0, self.fel.reshape(-1), v.reshape(-1, v.shape[2]))

    def div(self, v):  # (3, n, S): sum_d tGrad_d v_d, the weak divergence with the element's mean of v
        mean = v[:, self.fel].sum(2)  # (3, t, S)
        return self._sum(torch.einsum("eid,des->eis", self.g, mean) * (self.vol / 4)[:, None, None])

    def grad(self, u):  # (n, S) -> (3, n, S), volume-weighted at nodes
        ge = torch.einsum("eid,eis->des", self.g, u[self.fel]) * (self.vol / 4)[None, :, None]
        return torch.stack([self._sum(x[:, None, :].expand(-1, 4, -1).contiguous()) for x in ge]) / self.node_vol[:, None]

    def curl_t(self, m):  # sum of e x m with the operator tGrad in place of the gradient
        t = [[self._sum((self.g[:, :, d] * (self.vol / 4)[:, None])[:, :, None] * m[c][self.fel].sum(1)[:, None, :])
              for c in range(3)] for d in range(3)]  # t[d][c] = tGrad_d m_c
        return torch.stack([t[1][2] - t[2][1], t[2][0] - t[0][2], t[0][1] - t[1][0]])

    def solve(self, b, fixed, value):
        """K x = b on the free nodes, x = value on the fixed ones."""
        free = (~fixed).to(torch.float64)[:, None]
        x = value * (1 - free)
        r = (b - self.K @ x) * free
        dinv = free / self.diag[:, None]
        z = dinv * r
        p, rz, bb = z, (r * z).sum(0), (r * r).sum(0)
        bb = torch.where(bb > 0, bb, torch.ones_like(bb))
        for it in range(20000):
            q = (self.K @ p) * free
            pq = (p * q).sum(0)
            a = torch.where(pq > 0, rz / pq, torch.zeros_like(pq))
            x, r = x + a * p, r - a * q
            z = dinv * r
            new = (r * z).sum(0)
            p = z + torch.where(rz > 0, new / rz, torch.zeros_like(rz)) * p
            rz = new
            if it % 20 == 19 and bool(((r * r).sum(0) / bb).max() < 1e-28):
                break
        return x

    def _angle(self, a, b, c):  # solid angle of the triangle a, b, c from the origin (Van Oosterom, Strackee)
        la, lb, lc = (torch.linalg.vector_norm(v, dim=-1) for v in (a, b, c))
        num = (a * torch.linalg.cross(b, c)).sum(-1).abs()
        den = la * lb * lc + (a * b).sum(-1) * lc + (b * c).sum(-1) * la + (c * a).sum(-1) * lb
        return 2 * torch.atan2(num, den)

    def _boundary(self, xyz, X):
        f = torch.cat([self.fel[:, [1, 2, 3]], self.fel[:, [0, 2, 3]], self.fel[:, [0, 1, 3]], self.fel[:, [0, 1, 2]]])
        opposite = torch.cat([self.fel[:, k] for k in range(4)])
        f = f.sort(1).values
        key = (f[:, 0] * self.n + f[:, 1]) * self.n + f[:, 2]
        _, at, count = torch.unique(key, return_inverse=True, return_counts=True)
        once = count[at] == 1
        f, opposite = f[once], opposite[once]
        nodes = f.unique()
        self.nodes, b = nodes, nodes.numel()
        index = torch.full((self.n,), -1, dtype=torch.int64, device=self.dev)
        index[nodes] = torch.arange(b, device=self.dev)
        self.on_surface = index >= 0
        # corners in the order in which the normal points outward
        p = xyz[f]
        normal = torch.linalg.cross(p[:, 1] - p[:, 0], p[:, 2] - p[:, 0])
        out = ((xyz[opposite] - p[:, 0]) * normal).sum(1) > 0
        f = torch.where(out[:, None], f[:, [0, 2, 1]], f)
        p, fb = xyz[f], index[f]
        normal = torch.linalg.cross(p[:, 1] - p[:, 0], p[:, 2] - p[:, 0])
        area = torch.linalg.vector_norm(normal, dim=1) / 2
        normal = normal / (2 * area)[:, None]
        weight = (normal * area[:, None] / 3)[:, None, :].expand(-1, 3, -1).reshape(-1, 3)
        # nodal surface: mean outward normal and a third of each face's area
        s = torch.zeros((self.n, 3), dtype=torch.float64, device=self.dev).index_add(0, f.reshape(-1), weight)
        a = torch.zeros(self.n, dtype=torch.float64, device=self.dev).index_add(
            0, f.reshape(-1), (area / 3).repeat_interleave(3))
        length = torch.linalg.vector_norm(s, dim=1, keepdim=True)
        self.surface = torch.where(length > 0, s / torch.where(length > 0, length, torch.ones_like(length)), s) * a[:, None]
        B = torch.zeros((b, b), dtype=torch.float64, device=self.dev)
        omega = torch.zeros(self.n, dtype=torch.float64, device=self.dev)
        for k in range(4):
            o = [X[:, (k + q) % 4] - X[:, k] for q in (1, 2, 3)]
            omega.index_add_(0, self.fel[:, k], self._angle(*o))
        B.diagonal().copy_(omega[nodes] / (4 * math.pi) - 1)
        e = p.roll(-1, 1) - p  # edges and their in-plane normals (D. A. Lindholm, IEEE Trans. Magn. 20 (1984) 2025)
        le = torch.linalg.vector_norm(e, dim=2)
        xi = e / le[:, :, None]
        eta = torch.linalg.cross(normal[:, None, :].expand(-1, 3, -1).contiguous(), xi)
        gamma = torch.einsum("fid,fjd->fij", xi.roll(-1, 1), xi)
        step = max(1, 6_000_000 // f.shape[0])
        for r0 in range(0, b, step):
            at = torch.arange(r0, min(b, r0 + step), device=self.dev)
            rho = p[None] - xyz[nodes[at]][:, None, None, :]
            l = torch.linalg.vector_norm(rho, dim=3)
            height = (rho[:, :, 0] * normal[None]).sum(2)
            eta0 = (rho * eta[None]).sum(3)
            l1 = l.roll(-1, 2)
            Pl = torch.log((l + l1 + le[None]) / (l + l1 - le[None]))
            om = self._angle(rho[:, :, 0], rho[:, :, 1], rho[:, :, 2]) * torch.where(height < 0, -1.0, 1.0)
            L = le.roll(-1, 1)[None] / (8 * math.pi * area[None, :, None]) * (
                eta0.roll(-1, 2) * om[:, :, None] - height[:, :, None] * torch.einsum("fij,rfj->rfi", gamma, Pl))
            L = torch.where((fb[None] == at[:, None, None]).any(2)[:, :, None], torch.zeros_like(L), L)
            for q in range(3):
                B[r0:r0 + at.numel()].index_add_(1, fb[:, q], L[:, :, q].contiguous())
        self.B = B

    def potential(self, m):
        prob = self.prob
        js = torch.from_numpy(prob.Js).to(self.dev)[None, :, None]
        b = self.div(js * m) / P.MU0
        pin = torch.zeros(self.n, dtype=torch.bool, device=self.dev)
        pin[self.n // 2] = True
        u1 = self.solve(b, pin, b)
        value = torch.zeros_like(b)
        value[self.nodes] = self.B @ u1[self.nodes]
        return u1 + self.solve(torch.zeros_like(b), self.on_surface, value)

    def local(self, m):
        """Exchange, anisotropy and DMI, J/m^3."""
        prob, to = self.prob, lambda a: torch.from_numpy(np.asarray(a)).to(self.dev)
        V = self.node_vol[:, None]
        hx = torch.stack([-2.0 * (to(prob.A)[:, None] / V) * (self.K @ m[c]) for c in range(3)])
        k = to(prob.kaxis).view(3, -1, 1)
        hu = 2.0 * to(prob.Ku)[:, None] * (k * m).sum(0) * k
        hd = torch.zeros_like(hx)
        if prob.use_dmi:
            s = self.surface.T[:, :, None].expand_as(m)
            hd = (torch.linalg.cross(m, s.contiguous(), dim=0) + 2.0 * self.curl_t(m)) * (to(prob.D)[:, None] / V)
        return hx, hu, hd

    def rhs(self, m, hext):
        hx, hu, hd = self.local(m)
        H = (hx + hu + hd) / torch.from_numpy(self.prob.Js).to(self.dev)[None, :, None]
        H = H + hext[:, None, :] - self.grad(self.potential(m))
        return self.llg(m, H), H

    def llg(self, m, H):
        t = torch.linalg.cross(m, H, dim=0)
        return -t - self.prob.alpha * torch.linalg.cross(m, t, dim=0)


def _charge(prob, m):
    """Right-hand side of the Neumann problem: the weak divergence of Js m / mu0."""
    f = _Fem(prob, demag=False)
    return f.div(torch.from_numpy(prob.Js).to(f.dev)[None, :, None] * m) / P.MU0


def exact(case, seed):
    prob, kind = _problem(case), case["kind"]
    if kind == "vjp" or kind == "ode" or (prob.n > 100000 and kind != "spmv"):
        return None  # a gradient or a step sequence of its own; or over 20 s
    if kind == "batch_rk4" and prob.n * case["samples"] * case["steps"] > 400000:
        return None
    if kind == "rk4" and prob.n * case["steps"] > 60000:
        return None
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    if kind == "spmv":
        f = _Fem(prob, demag=False)
        g = torch.Generator(device=dev).manual_seed(seed)
        x = torch.randn(prob.n, generator=g, dtype=torch.float64, device=dev)
        a = torch.from_numpy(prob.A).to(dev) / f.node_vol
        return -2.0 * a * (f.K @ x[:, None])[:, 0]
    if kind == "solve":
        f = _Fem(prob, demag=False)
        b = _charge(prob, _smooth(prob, 1, 7 * seed, dev))
        pin = torch.zeros(prob.n, dtype=torch.bool, device=dev)
        pin[prob.n // 2] = True
        return f.solve(b, pin, b)[:, 0]
    f = _Fem(prob)
    if kind == "classes":
        m = _smooth(prob, 1, 7 * seed, dev)
        hx, hu, hd = f.local(m)
        H = (hx + hu + hd) / prob.mat.Js
        t = torch.linalg.cross(m, H, dim=0)
        return {"exchange": hx[:, :, 0].T, "uniaxial": hu[:, :, 0].T, "dmi": hd[:, :, 0].T,
                "dmdt": f.llg(m, H)[:, :, 0].reshape(-1),
                "torque": float(torch.linalg.vector_norm(t, dim=0).max())}
    batch = kind.startswith("batch")
    m = _smooth(prob, case.get("samples", 1), seed, dev)
    hext = torch.from_numpy(_fields(case, prob) if batch else prob.hext[:, None]).to(dev)
    if kind in ("rk4", "batch_rk4"):
        dt = _tau(prob, case["fs"])
        for _ in range(case["steps"]):
            k1 = f.rhs(m, hext)[0]
            k2 = f.rhs(m + 0.5 * dt * k1, hext)[0]
            k3 = f.rhs(m + 0.5 * dt * k2, hext)[0]
            k4 = f.rhs(m + dt * k3, hext)[0]
            m = m + (dt / 6) * (k1 + 2 * k2 + 2 * k3 + k4)
            m = m / torch.linalg.vector_norm(m, dim=0, keepdim=True)
        return m if batch else m.reshape(-1)
    d, H = f.rhs(m, hext)
    if not batch:
        return {"dmdt": d.reshape(-1), "heff": H.reshape(-1)}
    return {"dmdt": d, "heff": H} if case.get("heff") else d
