"""The work users have this framework do, as timed cases.

A case is one call of a public entry point on a water cluster of the sizes,
bases and grids that the package's own configurations and tests use
(gauxc_amd.workloads): XCIntegrator's EXC/VXC, UKS, FXC contraction and
nuclear gradient, the batched device context and the SSF weights.

    listed()            the cases, each with its place in real use beside it
    draw(rng)           one more of the same ranges
    prepare(case, seed) molecule, grid, weights, integrator and densities
    run(state)          one call, whole outputs
    work(case)          bytes and operations the call cannot do without
    exact(case, seed)   the outputs in plain 64-bit torch

The geometry, the density and the trial density follow from the seed.  The
exact values take the quadrature points and their atomic weights as inputs,
as a user's program has them from the grid; partition weights, basis
functions, functional and contractions are formed here, without screening.
"""
import functools
import math

import numpy as np
import torch

import gauxc_amd as gx
from gauxc_amd import workloads

# (l, [contraction: (exponents, coefficients)]) per element, beside the
# uncontracted bases of the package: segmented contractions of the shape of
# a double-zeta set, and a set with g functions on oxygen.
_ET = lambda a0, beta, n: [a0 * beta ** k for k in range(n)][::-1]  # noqa: E731
_S6 = [0.01, 0.05, 0.15, 0.35, 0.40, 0.15]
BASIS_CONTRACTED = {
    8: [(0, _ET(0.9, 3.2, 6), _S6), (0, _ET(0.6, 2.5, 3), [-0.1, 0.4, 0.7]), (0, [0.3], [1.0]),
        (1, _ET(0.6, 2.8, 4), [0.05, 0.2, 0.45, 0.5]), (1, [0.25], [1.0]), (2, [1.1], [1.0])],
    1: [(0, _ET(0.4, 3.0, 4), [0.03, 0.15, 0.45, 0.5]), (0, [0.15], [1.0]), (1, [0.7], [1.0])],
}
BASIS_G = {
    8: [(0, [a], [1.0]) for a in _ET(0.2, 3.0, 4)] + [(1, [a], [1.0]) for a in _ET(0.3, 3.0, 3)]
    + [(2, [a], [1.0]) for a in (0.6, 1.8)] + [(3, [1.0], [1.0]), (4, [1.4], [1.0])],
    1: [(0, [a], [1.0]) for a in (0.15, 0.6)] + [(1, [0.7], [1.0])],
}
POINTS = {"GM3": 35 * 110, "FineGrid": 75 * 302, "UltraFineGrid": 99 * 590}


def listed():
    def case(name, kind, waters, box, basis, grid, func, precision="fp64", weights=True):
        return {"name": name, "kind": kind, "waters": waters, "box": box, "basis": basis,
                "grid": grid, "func": func, "precision": precision, "weight_derivs": weights}
    return [
        # A small molecule on a coarse grid: the first SCF cycles, where
        # launches and host work are most of the call.
        case("rks_3w_lda_coarse", "rks", 3, 6.0, "c0", "GM3", "SVWN5"),
        # An everyday SCF call: contracted double-zeta basis, hybrid
        # functional, fine grid.
        case("rks_5w_contracted", "rks", 5, 6.4, "contracted", "FineGrid", "PBE0"),
        # High angular momentum (correlation-consistent quadruple-zeta use).
        case("rks_4w_gfunctions", "rks", 4, 6.0, "g", "FineGrid", "PBE"),
        # The 1,248-function cluster, both precisions: SCF of a mid-size system.
        case("rks_24w", "rks", 24, 10.0, "c1", "UltraFineGrid", "PBE"),
        case("rks_24w_mixed", "rks", 24, 10.0, "c1", "UltraFineGrid", "PBE", "mixed"),
        # The headline system, 7,800 functions, both precisions.
        case("rks_150w", "rks", 150, 17.0, "c1", "UltraFineGrid", "PBE"),
        case("rks_150w_mixed", "rks", 150, 17.0, "c1", "UltraFineGrid", "PBE", "mixed"),
        # Open-shell SCF.
        case("uks_9w", "uks", 9, 7.4, "c1", "FineGrid", "PBE"),
        # Geometry optimisation and response properties.
        case("grad_13w", "grad", 13, 8.3, "c1", "FineGrid", "PBE"),
        case("fxc_24w", "fxc", 24, 10.0, "c1", "FineGrid", "PBE"),
        # Many molecules at once (conformers, training data).
        case("batch_2_to_12w_mixed", "batch", 12, 0.0, "c1", "FineGrid", "PBE", "mixed"),
        # Partition weights of a new geometry.
        case("ssf_24w", "ssf", 24, 10.0, "c1", "UltraFineGrid", "PBE"),
    ]


# Largest cluster drawn per kind; every drawn case stays below the listed
# 150-water call.
_MOST = {"rks": 60, "uks": 32, "fxc": 40, "uks_fxc": 16, "grad": 32, "uks_grad": 16,
         "density": 40, "batch": 14, "ssf": 60}


def draw(rng):
    kind = rng.choice(["rks", "rks", "rks", "uks", "fxc", "uks_fxc", "grad", "uks_grad",
                       "density", "batch", "ssf"])
    basis = rng.choice(["c1", "c1", "c1", "c0", "contracted", "g"])
    if kind == "batch":
        basis = "c1"
    most = min(_MOST[kind], 8 if basis == "g" else 99)
    least = 4 if kind == "batch" else 2 if kind == "ssf" else 1
    n = int(round(math.exp(rng.uniform(math.log(least), math.log(most)))))
    grid = rng.choice(["FineGrid", "FineGrid", "UltraFineGrid", "GM3"])
    if kind not in ("rks", "ssf") and grid == "UltraFineGrid" and n > 16:
        grid = "FineGrid"
    mixed = kind == "batch" or (kind == "rks" and rng.random() < 0.4)
    return {"kind": kind, "waters": n,
            "box": 0.0 if kind == "batch" else round(3.3 * n ** (1 / 3) + rng.uniform(0.6, 2.0), 2),
            "basis": basis, "grid": grid, "func": rng.choice(["PBE", "PBE", "PBE0", "SVWN5"]),
            "precision": "mixed" if mixed else "fp64",
            "weight_derivs": not (kind in ("grad", "uks_grad") and rng.random() < 0.3)}


# ---- inputs ------------------------------------------------------------------

def _shell_arrays(Z, xyz, basis):
    if basis in ("c0", "c1"):
        recipe = workloads.BASIS_C0 if basis == "c0" else workloads.BASIS_C1
        return workloads.even_tempered_basis(Z, xyz, recipe)
    recipe = BASIS_CONTRACTED if basis == "contracted" else BASIS_G
    l, pure, alpha, coeff, origin = [], [], [], [], []
    for z, r in zip(Z, xyz):
        for am, a, c in recipe[int(z)]:
            l.append(am)
            pure.append(am >= 2)
            alpha.append(list(a))
            coeff.append(list(c))
            origin.append(r)
    return l, pure, alpha, coeff, origin


def _clusters(case, seed):
    """[(waters, box, geometry seed)] of the case's molecules."""
    if case["kind"] != "batch":
        return [(case["waters"], case["box"], seed)]
    sizes = range(2, case["waters"] + 1, 2 if case["waters"] % 2 == 0 else 3)
    return [(n, 3.5 * n ** (1 / 3) + 1.0, 1000 * seed + n) for n in sizes]


def _geometry(waters, box, seed):
    return workloads.water_cluster(waters, box, seed)


def _matrices(nbf, waters, seed):
    """P_alpha, and P_beta of a system with fewer beta electrons, and
    symmetric trial matrices, on the host as an SCF program holds them."""
    rng = np.random.default_rng(seed + 17)
    width = max(2, min(nbf, 5 * waters))
    C, _ = np.linalg.qr(rng.normal(size=(nbf, width)))
    half = max(1, width - max(1, width // 8))
    return C, half, rng


def _density(nbf, waters, seed):
    C = _matrices(nbf, waters, seed)[0]
    return np.asfortranarray(2.0 * C @ C.T)


def _spin_densities(nbf, waters, seed):
    C, half, _ = _matrices(nbf, waters, seed)
    Pa, Pb = C @ C.T, C[:, :half] @ C[:, :half].T
    return np.asfortranarray(Pa + Pb), np.asfortranarray(Pa - Pb)


def _trial(nbf, waters, seed, scale):
    _, _, rng = _matrices(nbf, waters, seed)
    U, V = rng.normal(size=(2, nbf, 8)) * scale / math.sqrt(nbf)
    return np.asfortranarray(U @ V.T + V @ U.T)


def _molecule(case, waters, box, seed):
    Z, xyz = _geometry(waters, box, seed)
    mol = gx.Molecule(Z, xyz)
    l, pure, alpha, coeff, origin = _shell_arrays(Z, xyz, case["basis"])
    # Partition weights are wanted at every grid point, also at those whose
    # basis functions would all be screened.
    tol = 1e-200 if case.get("kind") == "ssf" else 1e-10
    bs = gx.BasisSet(l, pure, alpha, coeff, origin, normalize=True, shell_tolerance=tol)
    return xyz, mol, bs


def _tasks(case, mol, bs, ex="Host"):
    return workloads.build_tasks(mol, bs, grid=case["grid"], ex=ex)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        mols = []
        for n, box, s in _clusters(case, seed):
            xyz, mol, bs = _molecule(case, n, box, s)
            lb = _tasks(case, mol, bs, "Device")
            gx.MolecularWeightsFactory("Device", "Default").get_instance().modify_weights(lb)
            mols.append((bs, lb, _density(bs.nbf(), n, s)))
        ctx = gx.BatchedDeviceContext()
        ctx.upload_molecules([m[0].xcq_shells() for m in mols])
        ctx.upload_tasks([m[1].get_tasks() for m in mols])
        ctx.use_graph(True)
        return {"case": case, "ctx": ctx, "P": [m[2] for m in mols]}
    (n, box, s), = _clusters(case, seed)
    xyz, mol, bs = _molecule(case, n, box, s)
    if kind == "ssf":
        t = _tasks(case, mol, bs, "Device").get_tasks()
        return {"case": case, "xyz": xyz, "points": t["points"], "weights": t["weights"],
                "parent": np.repeat(t["iparent"], t["npts"]).astype(np.int32)}
    lb = _tasks(case, mol, bs, "Device")
    gx.MolecularWeightsFactory("Device", "Default").get_instance().modify_weights(lb)
    lwd = "Scheme1-MIXED" if case["precision"] == "mixed" else "Default"
    spin = kind.startswith("uks")
    integ = gx.XCIntegratorFactory("Device", "Replicated", "Default", lwd, "Default").get_instance(
        gx.Functional(case["func"], polarized=spin), lb)
    integ.device_context()  # task data on the device, as after a first call
    nbf = bs.nbf()
    state = {"case": case, "integ": integ}
    if spin:
        state["Ps"], state["Pz"] = _spin_densities(nbf, n, s)
    else:
        state["P"] = _density(nbf, n, s)
    if kind in ("fxc", "uks_fxc"):
        state["tP"] = _trial(nbf, n, s, 1.0)
    if kind == "uks_fxc":
        state["tPz"] = _trial(nbf, n, s + 1, 0.3)
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "batch":
        ctx = state["ctx"]
        for m, P in enumerate(state["P"]):
            ctx.upload_density(m, P)
        ctx.exc_vxc(case["func"], case["precision"])
        out = [ctx.results(m) for m in range(len(state["P"]))]
        return {"exc": [o[0] for o in out], "nel": [o[1] for o in out], "vxc": [o[2] for o in out]}
    if kind == "ssf":
        return {"weights": gx.ssf_weights_device(state["xyz"], state["points"], state["parent"],
                                                 state["weights"])}
    integ = state["integ"]
    if kind == "rks":
        exc, vxc = integ.eval_exc_vxc(state["P"])
        return {"exc": exc, "vxc": vxc}
    if kind == "uks":
        exc, vs, vz = integ.eval_exc_vxc(state["Ps"], state["Pz"])
        return {"exc": exc, "vxc_s": vs, "vxc_z": vz}
    if kind == "fxc":
        return {"fxc": integ.eval_fxc_contraction(state["P"], state["tP"])}
    if kind == "uks_fxc":
        fs, fz = integ.eval_fxc_contraction(state["Ps"], state["tP"], Pz=state["Pz"],
                                            tPz=state["tPz"])
        return {"fxc_s": fs, "fxc_z": fz}
    if kind == "grad":
        return {"grad": integ.eval_exc_grad(state["P"],
                                            include_weight_derivatives=case["weight_derivs"])}
    if kind == "uks_grad":
        return {"grad": integ.eval_exc_grad(state["Ps"], state["Pz"],
                                            include_weight_derivatives=case["weight_derivs"])}
    return {"nel": integ.integrate_den(state["P"])}


# ---- work --------------------------------------------------------------------

@functools.lru_cache(maxsize=64)
def _sizes(waters, box, seed, basis, grid):
    """(points, sum of npts nbe^2, nbf) of a cluster's task list."""
    _, mol, bs = _molecule({"basis": basis}, waters, box, seed)
    t = _tasks({"grid": grid}, mol, bs).get_tasks()
    npts, nbe = t["npts"].astype(np.float64), t["nbe"].astype(np.float64)
    return float(npts.sum()), float((npts * nbe * nbe).sum()), bs.nbf()


def work(case):
    """Operations: a product of the task's points with an nbe x nbe matrix is
    2 npts nbe^2; a symmetric result (V) or a density alone needs half of
    the two products that define it.  Bytes: points, weights and the
    matrices in and out."""
    kind = case["kind"]
    if kind == "ssf":
        pts = case["waters"] * 3 * POINTS[case["grid"]]
        return {"bytes": 44.0 * pts, "flops": 0.0}
    lda = case["func"] == "SVWN5"
    dens = 1 if lda else 2  # flops per npts nbe^2 of one density pass
    flops = {"rks": dens + 2, "batch": dens + 2, "uks": 2 * dens + 4, "fxc": 2 * dens + 2,
             "uks_fxc": 4 * dens + 4, "grad": 4, "uks_grad": 8, "density": 1}[kind]
    mats = {"rks": 2, "batch": 2, "uks": 4, "fxc": 3, "uks_fxc": 6, "grad": 1, "uks_grad": 2,
            "density": 1}[kind]
    total = {"bytes": 0.0, "flops": 0.0}
    for n, box, s in _clusters(case, 0):
        pts, pnn, nbf = _sizes(n, box, s, case["basis"], case["grid"])
        total["bytes"] += 32.0 * pts + mats * 8.0 * nbf * nbf
        total["flops"] += flops * pnn
    return total


# ---- exact values ------------------------------------------------------------

def _poly_mul(p, q):
    out = {}
    for (a, b, c), u in p.items():
        for (d, e, f), v in q.items():
            k = (a + d, b + e, c + f)
            out[k] = out.get(k, 0.0) + u * v
    return out


def _poly_pow(p, n):
    out = {(0, 0, 0): 1.0}
    for _ in range(n):
        out = _poly_mul(out, p)
    return out


@functools.lru_cache(maxsize=None)
def _harmonics(l, pure):
    """The angular polynomials of a shell, {exponents: coefficient} each:
    Cartesian in the order x^l, x^(l-1) y, ...; else the Racah-normalised
    real solid harmonics m = -l .. l, from the explicit sum of the associated
    Legendre polynomial and the real or imaginary part of (x + i y)^m."""
    if not pure:
        return [{(a, b, l - a - b): 1.0} for a in range(l, -1, -1) for b in range(l - a, -1, -1)]
    out = []
    r2 = {(2, 0, 0): 1.0, (0, 2, 0): 1.0, (0, 0, 2): 1.0}
    for m in range(-l, l + 1):
        am = abs(m)
        norm = math.sqrt((1 if m == 0 else 2) * math.factorial(l - am) / math.factorial(l + am))
        leg = {}
        for k in range((l - am) // 2 + 1):
            c = ((-1) ** k * 2.0 ** -l * math.comb(l, k) * math.comb(2 * l - 2 * k, l)
                 * math.factorial(l - 2 * k) / math.factorial(l - 2 * k - am))
            for e, v in _poly_mul(_poly_pow(r2, k), {(0, 0, l - 2 * k - am): c}).items():
                leg[e] = leg.get(e, 0.0) + v
        azi = {}
        for k in range(am + 1):  # (x + i y)^am = sum comb(am, k) x^(am-k) y^k i^k
            if k % 2 == (0 if m >= 0 else 1):
                azi[(am - k, k, 0)] = math.comb(am, k) * (-1.0) ** (k // 2)
        out.append({e: norm * v for e, v in _poly_mul(leg, azi).items() if v})
    return out


def _poly_d(p, d):
    out = {}
    for e, v in p.items():
        if e[d]:
            f = list(e)
            f[d] -= 1
            out[tuple(f)] = out.get(tuple(f), 0.0) + v * e[d]
    return out


def _poly_eval(p, pw, like):
    s = torch.zeros_like(like)
    for (a, b, c), v in p.items():
        t = None
        for k, e in enumerate((a, b, c)):
            if e:
                t = pw[k][e] if t is None else t * pw[k][e]
        s = s + (v if t is None else v * t)
    return s


class _Exact:
    """A molecule's quadrature in 64-bit torch."""

    def __init__(self, case, n, box, seed, dev):
        Z, xyz = _geometry(n, box, seed)
        l, pure, alpha, coeff, origin = _shell_arrays(Z, xyz, case["basis"])
        self.dev, self.func = dev, case["func"]
        self.R = torch.tensor(xyz, dtype=torch.float64, device=dev)
        xyz = np.asarray(xyz)
        groups, first = {}, 0
        for i in range(len(l)):
            a, c = np.array(alpha[i]), np.array(coeff[i], dtype=float)
            L = l[i]
            df = math.prod(range(2 * L - 1, 0, -2))
            c = c * np.sqrt(2.0 ** L * (2 * a) ** (L + 1.5) / (math.pi ** 1.5 * df))
            g = a[:, None] + a[None, :]
            c = c / math.sqrt((c[:, None] * c[None, :] * df * math.pi ** 1.5
                               / (2.0 ** L * g ** (L + 1.5))).sum())
            atom = int(np.argmin(((xyz - np.asarray(origin[i])) ** 2).sum(1)))
            groups.setdefault((L, bool(pure[i]), len(a)), []).append((first, atom, a, c))
            first += 2 * L + 1 if pure[i] else (L + 1) * (L + 2) // 2
        self.nbf = first
        t64 = lambda v: torch.tensor(np.array(v), dtype=torch.float64, device=dev)  # noqa: E731
        self.groups = [(k, torch.tensor([s[0] for s in v], device=dev),
                        torch.tensor([s[1] for s in v], device=dev),
                        t64([s[2] for s in v]), t64([s[3] for s in v])) for k, v in groups.items()]
        _, mol, bs = _molecule(case, n, box, seed)
        t = _tasks(case, mol, bs).get_tasks()
        self.parent = torch.tensor(np.repeat(t["iparent"], t["npts"]), device=dev).long()
        self.points = torch.tensor(t["points"], device=dev)
        self.w0 = torch.tensor(t["weights"], device=dev)
        self.npts = len(t["weights"])

    def ssf(self, pts, parent, w0, R):
        """SSF partition weights (Stratmann, Scuseria, Frisch 1996)."""
        if len(R) == 1:
            return w0
        a = 0.64
        eye = torch.eye(len(R), dtype=torch.bool, device=self.dev)
        rab = ((R[:, None] - R[None]) ** 2).sum(-1).masked_fill(eye, 1.0).sqrt()
        d = ((pts[:, None] - R[None]) ** 2).sum(-1).clamp_min(1e-60).sqrt()
        v = (d[:, :, None] - d[:, None, :]) / rab / a
        u = v.clamp(-1, 1)
        s = 0.5 * (1 - (35 * u - 35 * u ** 3 + 21 * u ** 5 - 5 * u ** 7) / 16)
        s = torch.where(v <= -1, 1.0, torch.where(v >= 1, 0.0, s)).masked_fill(eye, 1.0)
        P = s.prod(-1)
        near = rab.masked_fill(eye, math.inf).min(1).values
        dp = d.gather(1, parent[:, None])[:, 0]
        w = w0 * P.gather(1, parent[:, None])[:, 0] / P.sum(1)
        return torch.where(dp < 0.5 * (1 - a) * near[parent], w0, w)

    def basis(self, pts, R, grad):
        """Basis functions (and gradients): [1 or 4][npts, nbf]."""
        cols = [[] for _ in range(4 if grad else 1)]
        order = []
        for (l, pure, _), first, atom, alpha, coeff in self.groups:
            d = pts[:, None, :] - R[atom][None]
            r2 = (d * d).sum(-1)
            e = coeff * torch.exp(-alpha * r2[..., None])
            rad, drad = e.sum(-1), (-2 * alpha * e).sum(-1)
            pw = []
            for k in range(3):
                p = [None, d[..., k]]
                for _ in range(2, l + 1):
                    p.append(p[-1] * p[1])
                pw.append(p)
            for m, poly in enumerate(_harmonics(l, pure)):
                y = _poly_eval(poly, pw, r2)
                cols[0].append(y * rad)
                if grad:
                    for k in range(3):
                        cols[1 + k].append(_poly_eval(_poly_d(poly, k), pw, r2) * rad
                                           + y * drad * d[..., k])
                order.append(first + m)
        back = torch.argsort(torch.cat(order))
        return [torch.cat(c, 1)[:, back] for c in cols]

    # -- functional: energy density per volume from spin densities and gradients
    def energy(self, n, gn, m=None, gm=None):
        """n, m: total and spin density [npts]; gn, gm: gradients [3, npts]."""
        m = torch.zeros_like(n) if m is None else m
        gga = self.func != "SVWN5"
        xs = 0.75 if self.func == "PBE0" else 1.0
        na, nb = (n + m) / 2, (n - m) / 2
        saa = sbb = st = None
        if gga:
            gm = torch.zeros_like(gn) if gm is None else gm
            saa, sbb = (((gn + gm) / 2) ** 2).sum(0), (((gn - gm) / 2) ** 2).sum(0)
            st = (gn ** 2).sum(0)
        e = 0.0
        cx = -0.75 * (3 / math.pi) ** (1 / 3)
        for r, s in ((na, saa), (nb, sbb)):
            ok = 2 * r > 1e-15
            r2 = torch.where(ok, 2 * r, 1.0)
            ex = cx * r2 ** (4 / 3)
            if gga:
                s2 = 4 * s / (4 * (3 * math.pi ** 2) ** (2 / 3) * r2 ** (8 / 3))
                ex = ex * (1.804 - 0.804 / (1 + 0.2195149727645171 * s2 / 0.804))
            e = e + 0.5 * xs * torch.where(ok, ex, 0.0)
        ok = n > (1e-12 if gga else 1e-15)
        r = torch.where(ok, n, 1.0)
        z = torch.where(ok, m / r, 0.0).clamp(-1 + 1e-14, 1 - 1e-14)
        rs = (3 / (4 * math.pi * r)) ** (1 / 3)
        f = ((1 + z) ** (4 / 3) + (1 - z) ** (4 / 3) - 2) / (2 ** (4 / 3) - 2)
        if not gga:
            x = rs.sqrt()

            def vwn(A, b, c, x0):
                X = x * x + b * x + c
                Q = math.sqrt(4 * c - b * b)
                X0 = x0 * x0 + b * x0 + c
                at = torch.atan(Q / (2 * x + b))
                return A * (torch.log(x * x / X) + 2 * b / Q * at - b * x0 / X0
                            * (torch.log((x - x0) ** 2 / X) + 2 * (b + 2 * x0) / Q * at))
            ep = vwn(0.0310907, 13.0720, 42.7198, -0.409286)
            ef = vwn(0.01554535, 20.1231, 101.578, -0.743294)
            return e + torch.where(ok, r * (ep + (ef - ep) * f), 0.0)

        def pw92(a, a1, b1, b2, b3, b4):
            q = 2 * a * (b1 * rs.sqrt() + b2 * rs + b3 * rs ** 1.5 + b4 * rs * rs)
            return -2 * a * (1 + a1 * rs) * torch.log1p(1 / q)
        ep = pw92(0.0310907, 0.21370, 7.5957, 3.5876, 1.6382, 0.49294)
        ef = pw92(0.01554535, 0.20548, 14.1189, 6.1977, 3.3662, 0.62517)
        mac = pw92(0.0168869, 0.11125, 10.357, 3.6231, 0.88026, 0.49671)
        ec = ep - mac * f / 1.709920934161365617563962776245 * (1 - z ** 4) + (ef - ep) * f * z ** 4
        gamma, beta = (1 - math.log(2)) / math.pi ** 2, 0.06672455060314922
        phi = ((1 + z) ** (2 / 3) + (1 - z) ** (2 / 3)) / 2
        t2 = math.pi / (16 * (3 * math.pi ** 2) ** (1 / 3)) * st / (phi ** 2 * r ** (7 / 3))
        A = beta / gamma / torch.expm1(-ec / (gamma * phi ** 3))
        q = t2 * (1 + A * t2) / (1 + A * t2 + (A * t2) ** 2)
        h = gamma * phi ** 3 * torch.log1p(beta / gamma * q)
        return e + torch.where(ok, r * (ec + h), 0.0)

    def chunks(self, step):
        for a in range(0, self.npts, step):
            yield slice(a, min(self.npts, a + step))

    def rho(self, B, P, fac):
        X = fac * (B[0] @ P)
        return torch.stack([(B[0] * X).sum(1)] + [2 * (b * X).sum(1) for b in B[1:]])

    def potentials(self, mats, fac, trial=None):
        """EXC, NEL and the potential of each density matrix; with trial
        matrices the potentials' derivatives along them."""
        gga = self.func != "SVWN5"
        exc = nel = 0.0
        V = [torch.zeros(self.nbf, self.nbf, dtype=torch.float64, device=self.dev) for _ in mats]
        for c in self.chunks(max(256, int(4e8) // (self.nbf * 8 * 8))):
            pts = self.points[c]
            w = self.ssf(pts, self.parent[c], self.w0[c], self.R)
            B = self.basis(pts, self.R, gga)
            rho = [self.rho(B, P, fac).detach().requires_grad_() for P in mats]
            args = []
            for r in rho:
                args += [r[0], r[1:] if gga else None]
            e = (w * self.energy(*args)).sum()
            exc, nel = exc + float(e.detach()), nel + float((w * rho[0][0]).sum().detach())
            g = torch.autograd.grad(e, rho, create_graph=trial is not None)
            if trial is not None:
                t = [self.rho(B, T, fac) for T in trial]
                g = torch.autograd.grad(sum((x * y).sum() for x, y in zip(g, t)), rho)
            for x, v in zip(g, V):
                Zm = 0.5 * x[0][:, None] * B[0]
                for k in range(1, len(B)):
                    Zm = Zm + x[k][:, None] * B[k]
                W = B[0].T @ Zm
                v += W + W.T
        return exc, nel, V

    def gradient(self, mats, fac, weights):
        gga = self.func != "SVWN5"
        R = self.R.clone().requires_grad_()
        G = torch.zeros_like(R)
        terms = 60 * self.nbf * (4 if gga else 1) + 30 * len(R) ** 2
        for c in self.chunks(max(64, int(2e10) // (8 * terms))):
            par = self.parent[c]
            u = self.points[c] - self.R[par]
            pts = R[par] + u if weights else self.points[c]
            Rw = R if weights else self.R
            w = self.ssf(pts, par, self.w0[c], Rw)
            B = self.basis(pts, R, gga)
            args = []
            for P in mats:
                r = self.rho(B, P, fac)
                args += [r[0], r[1:] if gga else None]
            e = (w * self.energy(*args)).sum()
            G += torch.autograd.grad(e, R)[0]
        return G


def exact(case, seed):
    kind = case["kind"]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    cost = 0.0  # about the operations of the dense evaluation below
    for n, box, s in _clusters(case, seed):
        nat = 3 * n
        per = sum(2 * l + 1 if l > 1 else (l + 1) * (l + 2) // 2
                  for l in _shell_arrays(*workloads.water_cluster(1, 5.0, 0), case["basis"])[0])
        pts = nat * POINTS[case["grid"]]
        passes = {"ssf": 0, "uks": 8, "fxc": 8, "uks_fxc": 14, "uks_grad": 24, "grad": 14}.get(kind, 4)
        if case["basis"] == "g" or kind in ("grad", "uks_grad"):
            cost += pts * n * per * 9000.0
        cost += pts * (passes * (n * per) ** 2 + 2000.0 * n * per * (kind != "ssf") + 150.0 * nat * nat)
    if cost > (2e14 if dev == "cuda" else 2e12):
        return None
    outs = []
    for n, box, s in _clusters(case, seed):
        E = _Exact(case, n, box, s, dev)
        if kind == "ssf":
            w = [E.ssf(E.points[c], E.parent[c], E.w0[c], E.R)
                 for c in E.chunks(max(256, int(2e9) // (8 * 9 * n * n * 8)))]
            return {"weights": torch.cat(w).cpu().numpy()}
        put = lambda a: torch.tensor(np.ascontiguousarray(a), device=dev)  # noqa: E731
        nbf, uks = E.nbf, kind.startswith("uks")
        mats = [put(m) for m in (_spin_densities(nbf, n, s) if uks else (_density(nbf, n, s),))]
        fac = 1.0 if uks else 2.0
        if kind in ("grad", "uks_grad"):
            return {"grad": E.gradient(mats, fac, case["weight_derivs"]).cpu().numpy()}
        trial = None
        if kind == "fxc":
            trial = [put(_trial(nbf, n, s, 1.0))]
        elif kind == "uks_fxc":
            trial = [put(_trial(nbf, n, s, 1.0)), put(_trial(nbf, n, s + 1, 0.3))]
        exc, nel, V = E.potentials(mats, 1.0 if kind == "density" else fac, trial)
        outs.append((exc, nel, [v.cpu().numpy() for v in V]))
    exc, nel, V = outs[0]
    if kind == "batch":
        return {"exc": [o[0] for o in outs], "nel": [o[1] for o in outs],
                "vxc": [o[2][0] for o in outs]}
    if kind == "rks":
        return {"exc": exc, "vxc": V[0]}
    if kind == "uks":
        return {"exc": exc, "vxc_s": V[0], "vxc_z": V[1]}
    if kind == "fxc":
        return {"fxc": V[0]}
    if kind == "uks_fxc":
        return {"fxc_s": V[0], "fxc_z": V[1]}
    return {"nel": nel}
