"""The work that a user of this framework has it do, as cases to be timed.

Each case is one pass through the public entry points of the Python binding on
a Kuhn-subdivided sphere with n subcubes a side (n = 2: 72 unknowns, n = 5:
1,350, n = 12: 19,872), the mesh family of the repository's configurations:

- scatter: one frequency of the scattering loop -- matrix, incident fields,
  factorisation, solve, absorbed and scattered powers -- in the forms that the
  library offers: "fp64" (complex128 LU), "mixed" (complex64 LU with FP64
  refinement) and "fast" (block-local pivoting, split-FP16 updates, FP64
  refinement), the last two with the precision form's far field;
- assemble: the matrix alone, for programs that bring their own solver, also
  with a compiled permittivity expression and a complex frequency;
- batch: uneven spheres swept over frequencies in one call;
- rytov: buff-neq's dressed Rytov matrix and the power from it;
- fields: total fields at points around and inside the object;
- cold: what a new mesh costs before its first frequency.

The learned surrogate is not here: its tables depend on how a network was
trained, and the scattering loop does not use it by default.
"""
import importlib.util
import math
import os

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_spec = importlib.util.spec_from_file_location("buffem_amd", os.path.join(_ROOT, "buff-em_amd", "__init__.py"))
bfa = importlib.util.module_from_spec(_spec)
_spec.loader.exec_module(bfa)

ZVAC = 376.73031346177
TD_ORDER = 10        # the order that bench.py and the batch workload use
TOL, MAXIT = 1e-10, 30
DEV = "cuda"


# ---------------------------------------------------------------------------
# the cases

def listed():
    return [
        # the smallest problem of a convergence study: launches and latency
        dict(name="scatter_fp64_n3", kind="scatter", form="fp64", n=3, radius=1.0, omega=1.0, mat="iso", nrhs=1),
        # the plain method on the repository's small configuration
        dict(name="scatter_fp64_n5", kind="scatter", form="fp64", n=5, radius=1.0, omega=1.0, mat="iso", nrhs=1),
        # the precision form: inhomogeneous material, many incidence directions
        dict(name="scatter_mixed_n5", kind="scatter", form="mixed", n=5, radius=1.0, omega=1.0, mat="sincos", nrhs=32),
        # the fast form at an ordinary size, the Janus sphere of the sweep
        dict(name="scatter_fast_n8", kind="scatter", form="fast", n=8, radius=0.9, omega=2.0, mat="janus", nrhs=1),
        # the plain method at a size that fills the chip
        dict(name="scatter_fp64_n10", kind="scatter", form="fp64", n=10, radius=1.2, omega=0.7, mat="janus", nrhs=1),
        # the headline configuration: 19,872 unknowns, anisotropic, two polarisations
        dict(name="scatter_fast_n12", kind="scatter", form="fast", n=12, radius=1.0, omega=1.0, mat="diag", nrhs=2),
        # the matrix of the headline configuration alone
        dict(name="assemble_n12", kind="assemble", n=12, radius=1.0, omega=1.0, omega_im=0.0, mat="diag"),
        # a permittivity file's expression at a complex frequency (Casimir-like use), odd size
        dict(name="assemble_expr_n7", kind="assemble", n=7, radius=0.8, omega=1.3, omega_im=0.4, mat="expr"),
        # a sweep over uneven particles
        dict(name="batch_10", kind="batch", count=10, nlo=4, nhi=8, nfreq=2, wlo=0.3, whi=4.0, nrhs=1),
        # thermal emission: one frequency of buff-neq
        dict(name="rytov_n6", kind="rytov", n=6, radius=1.0, omega=1.0, mat="sincos"),
        # a field map
        dict(name="fields_n8", kind="fields", n=8, radius=1.0, omega=1.5, npts=1000, nrhs=1),
        # a new mesh
        dict(name="cold_n8", kind="cold", n=8, radius=1.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["scatter"] * 5 + ["assemble"] * 2 + ["batch", "rytov", "fields", "cold"])
    radius, omega = round(rng.uniform(0.5, 1.5), 3), round(math.exp(rng.uniform(math.log(0.3), math.log(3.0))), 3)
    mat = rng.choice(["iso", "diag", "sincos", "janus"])
    if kind == "scatter":
        form = rng.choice(["fp64", "mixed", "fast"])
        n = rng.randint(2, 9) if form != "fast" else rng.randint(4, 11)
        nrhs = rng.choice([1, 2, 3, 8, 32]) if n < 10 else 2
        return dict(kind=kind, form=form, n=n, radius=radius, omega=omega, mat=mat, nrhs=nrhs)
    if kind == "assemble":
        return dict(kind=kind, n=rng.randint(3, 11), radius=radius, omega=omega,
                    omega_im=rng.choice([0.0, round(rng.uniform(0.05, 0.6), 3)]), mat=rng.choice([mat, "expr"]))
    if kind == "batch":
        nlo = rng.randint(3, 5)
        return dict(kind=kind, count=rng.randint(2, 10), nlo=nlo, nhi=rng.randint(nlo, 8), nfreq=rng.randint(1, 2),
                    wlo=0.3, whi=round(rng.uniform(1.0, 4.0), 2), nrhs=rng.randint(1, 3))
    if kind == "rytov":
        return dict(kind=kind, n=rng.randint(3, 6), radius=radius, omega=omega, mat=rng.choice(["iso", "sincos"]))
    if kind == "fields":
        return dict(kind=kind, n=rng.randint(3, 9), radius=radius, omega=omega, npts=_log_int(rng, 30, 1500),
                    nrhs=rng.randint(1, 2))
    return dict(kind=kind, n=rng.randint(3, 9), radius=radius)


# ---------------------------------------------------------------------------
# inputs

def _material(name):
    if name == "iso":
        return bfa.material("iso", eps=4 + 0.1j)
    if name == "diag":
        return bfa.material("diag", eps=(4 + 0.05j, 5 + 0.05j, 6 + 0.05j))
    if name == "sincos":
        return bfa.material("sincos", base=4.0, amp=2.0, imag=0.1)
    if name == "janus":
        return bfa.material("janus", up=4 + 0.1j, down=12 + 1j)
    return bfa.material_expr("4+0.5*sin(2*x)*cos(y)+0.3*z*z+0.1*i")


def _planewaves(count, rng):
    """The two polarisations along +z, then random directions with a transverse field."""
    spec = [((1, 0, 0), (0, 0, 1)), ((0, 1, 0), (0, 0, 1))][:count]
    while len(spec) < count:
        d = rng.standard_normal(3)
        d /= np.linalg.norm(d)
        e = np.cross(d, rng.standard_normal(3))
        spec.append((tuple(e / np.linalg.norm(e)), tuple(d)))
    return spec


def _mesh(n, radius, seed):
    return bfa.kuhn_sphere(n, radius, 0.05, seed)


def _geometry(V, T):
    g = bfa.Geometry(V, T)
    g.upload()
    g.build_static(TD_ORDER)
    return g


def _batch_meshes(case, seed):
    rng = np.random.default_rng(12345)      # sizes belong to the case, the meshes to the seed
    out = []
    for i in range(case["count"]):
        n, R = int(rng.integers(case["nlo"], case["nhi"] + 1)), float(rng.uniform(0.5, 1.5))
        out.append(_mesh(n, R, seed * 100 + i) + ("janus" if i % 2 else "iso",))
    return out


def _omegas(case):
    return np.geomspace(case["wlo"], case["whi"], case["nfreq"])


def _field_inputs(case, N, seed):
    rng = np.random.default_rng(seed)
    X = rng.uniform(-2.0, 2.0, (case["npts"], 3)) * case["radius"]
    J = (rng.standard_normal(N) + 1j * rng.standard_normal(N)) * 1e-3
    return X, J


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    s = dict(case=case)
    if kind == "batch":
        meshes = _batch_meshes(case, seed)
        geoms = [_geometry(V, T) for V, T, _ in meshes]
        s["batch"] = bfa.Batch(geoms, [_material(m) for _, _, m in meshes], bfa.planewaves(_planewaves(case["nrhs"], rng)))
        s["batch"].set_tiles([2] * 16)      # a stored tuning: the variant that the tuner picks
        s["omegas"] = _omegas(case)
        return s
    V, T = _mesh(case["n"], case["radius"], seed)
    if kind == "cold":
        s["V"], s["T"] = V, T
        return s
    s["g"] = g = _geometry(V, T)
    N = g.N
    if kind == "fields":
        s["X"], J = _field_inputs(case, N, seed)
        s["J"] = torch.from_numpy(J).to(DEV)
        s["pws"] = bfa.planewaves(_planewaves(case["nrhs"], rng))
        return s
    s["mat"] = _material(case["mat"])
    s["M"] = torch.zeros((N, N), dtype=torch.complex128, device=DEV)
    if kind == "scatter":
        s["pws"] = bfa.planewaves(_planewaves(case["nrhs"], rng))
        s["B"] = torch.zeros((case["nrhs"], N), dtype=torch.complex128, device=DEV)
        s["piv"] = torch.zeros(N, dtype=torch.int32, device=DEV)
        if case["form"] != "fp64":
            s["M32"] = torch.zeros((N, N), dtype=torch.complex64, device=DEV)
    if kind == "rytov":
        s["Sinv"] = torch.zeros((N, N), dtype=torch.complex128, device=DEV)
        g.gram_inverse(s["Sinv"])
        s["work"] = torch.zeros(g.dressed_rytov_work_bytes(), dtype=torch.uint8, device=DEV)
    return s


# ---------------------------------------------------------------------------
# one pass

def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind == "scatter":
        g, w, N, nrhs, M, B = s["g"], case["omega"], s["g"].N, case["nrhs"], s["M"], s["B"]
        form = case["form"]
        g.assemble_vie(w, s["mat"], M, far32=form != "fp64")
        g.assemble_rhs(w, s["pws"], B)
        if form == "fp64":
            bfa.lu_factor(M, N, s["piv"])
            bfa.lu_solve(M, N, s["piv"], B, nrhs)
        else:
            bfa.convert_z2c(M, N, N, s["M32"])
            (bfa.lu_factor_c if form == "mixed" else bfa.lu_factor_c_local)(s["M32"], N, s["piv"])
            bfa.solve_refine(M, s["M32"], s["piv"], N, B, nrhs, tol=TOL, maxit=MAXIT)
        return {"J": B, "power": g.emt_power(w, s["pws"], B)}
    if kind == "assemble":
        s["g"].assemble_vie(complex(case["omega"], case["omega_im"]), s["mat"], s["M"])
        return {"M": s["M"]}
    if kind == "batch":
        r = s["batch"].run(s["omegas"], use_graph=True, tol=TOL, maxit=6)
        return {"power": r["power"], "info": r["info"], "J": [s["batch"].solution(i) for i in range(case["count"])]}
    if kind == "rytov":
        s["g"].dressed_rytov(case["omega"], s["mat"], s["Sinv"], s["M"], s["work"])
        return {"DR": s["M"], "power": s["g"].emt_power_dr(case["omega"], s["M"])}
    if kind == "fields":
        E, H = s["g"].get_fields(case["omega"], s["X"], s["J"], s["pws"])
        return {"E": E, "H": H}
    g = _geometry(s["V"], s["T"])
    out = {"table": g.static_table()}
    g.close()
    return out


# ---------------------------------------------------------------------------
# what a pass cannot do without

def _sizes(n):
    """Tetrahedra and interior faces of the Kuhn sphere; touching pairs are about 84 a face at n = 12."""
    nt, nbf = 6 * n ** 3, 12 * n ** 3 - 6 * n ** 2
    return nt, nbf


def _assembly_flops(n):
    """16 point pairs a tetrahedron pair (a distance, a complex exponential, 16 moments: about 100
    operations), then 4 combinations of 4 moments a matrix entry of one triangle (about 160); 64 point
    pairs of about 60 operations for each of some 60 touching pairs a row."""
    nt, nbf = _sizes(n)
    return nt * nt / 2 * 16 * 100 + nbf * nbf / 2 * 160 + 60.0 * nbf * 64 * 60


def _power_flops(n, nrhs):
    """The same point pairs with the real kernel, 8 moments, and a form in the currents a tetrahedron pair."""
    nt, nbf = _sizes(n)
    return nt * nt / 2 * (16 * 60 + nrhs * 60.0) + 60.0 * nbf * 1024 * 30


def work(case):
    kind = case["kind"]
    if kind == "batch":
        rng = np.random.default_rng(12345)
        f = b = 0.0
        for _ in range(case["count"]):
            n = int(rng.integers(case["nlo"], case["nhi"] + 1))
            rng.uniform(0.5, 1.5)
            one = work(dict(kind="scatter", form="fast", n=n, nrhs=case["nrhs"]))
            f += one["flops"] * case["nfreq"]
            b += one["bytes"] * case["nfreq"]
        return {"bytes": b, "flops": f}
    nt, nbf = _sizes(case["n"])
    geom = nt * 16 * 8.0 + nbf * 100.0                 # points and basis functions
    static = 60.0 * nbf * 48                           # static records
    if kind == "scatter":
        r = case["nrhs"]
        f = _assembly_flops(case["n"]) + _power_flops(case["n"], r) + 8.0 / 3.0 * nbf ** 3 + 8.0 * nbf * nbf * r
        return {"bytes": geom + static + 32.0 * nbf * r, "flops": f}
    if kind == "assemble":
        return {"bytes": geom + static + 16.0 * nbf * nbf, "flops": _assembly_flops(case["n"])}
    if kind == "rytov":                                # three products, one LU, one solve of N columns
        return {"bytes": geom + static + 32.0 * nbf * nbf,
                "flops": _assembly_flops(case["n"]) + _power_flops(case["n"], 1) + (24.0 + 8.0 / 3.0 + 8.0) * nbf ** 3}
    if kind == "fields":                               # 8 source points a basis function and point, far rule
        return {"bytes": geom + 16.0 * nbf + 120.0 * case["npts"], "flops": 8.0 * nbf * case["npts"] * 120}
    # cold: 256 point pairs of the static kernel, four tetrahedron pairs a touching pair, and the singular pairs' cubature
    return {"bytes": geom + 2 * static, "flops": 60.0 * nbf * 4 * 256 * 20 + nt * 40.0 * 20 * 1e4 * 60}


def tolerance(case):
    """About four times what the listed cases and drawn ones show against exact()."""
    kind = case["kind"]
    if kind == "scatter" and case["form"] != "fp64" or kind == "batch":
        return {"rel": 4e-8, "max": 4e-6}      # the far field's FP32 remainder, a residual of 1e-10 in the refinement
    if kind == "scatter":
        return {"rel": 2e-10, "max": 2e-8}
    if kind == "assemble":                     # the desingularised kernel's series ends at 1e-8 of its own value
        return {"rel": 1.3e-9, "max": 1e-6}
    if kind == "rytov":
        return {"rel": 5e-11, "max": 5e-9}
    return {"rel": 1e-12, "max": 1e-9}


# ---------------------------------------------------------------------------
# the same results in 64 bits, from torch alone

def _orbit(bary):
    """Distinct permutations of barycentric coordinates, (u1, u2, u3) of each."""
    import itertools
    seen = []
    for p in itertools.permutations(bary):
        if p[1:] not in seen:
            seen.append(p[1:])
    return seen


def _rule(npts):
    """The reference's symmetric tetrahedron rules of 4, 16 and 33 points: (u [n, 3], w [n]), sum w = 1/6."""
    a = 0.13819660112501051
    orbits = {
        4: [((1 - 3 * a, a, a, a), 0.041666666666666666)],
        16: [((0.771642902067237,) + (0.076119032644254315,) * 3, 8.3956323500204695e-3),
             ((0.07183164526766925, 0.11970052779780202, 0.40423391346726440, 0.40423391346726440), 0.011090344772215399)],
        33: [((0.25,) * 4, 0.017783308938202055),
             ((0.05777714911165610,) + (0.31407428362944793,) * 3, -0.019099406118263309),
             ((0.81235958507558810,) + (0.06254680497480394,) * 3, 3.8252276536630236e-3),
             ((0.61738099120939840, 0.04120213879937276, 0.04120213879937276, 0.30021473119185615), 0.0035475499144103266),
             ((0.44311853122966216, 0.05292032110257111, 0.25198057383388334, 0.25198057383388334), 0.013950789384495153)],
    }[npts]
    u, w = [], []
    for bary, wt in orbits:
        pts = _orbit(bary)
        u += pts
        w += [wt] * len(pts)
    return torch.tensor(u, dtype=torch.float64, device=DEV), torch.tensor(w, dtype=torch.float64, device=DEV)


class _Exact:
    """Topology and cubature of one mesh, and the method's integrals over it."""

    def __init__(self, V, T):
        self.V = torch.from_numpy(np.asarray(V)).to(DEV)
        nt = len(T)
        # interior faces, numbered at the second visit; face i is opposite vertex i
        opp = np.array([[1, 2, 3], [0, 2, 3], [0, 1, 3], [0, 1, 2]])
        key = np.sort(T[:, opp].reshape(-1, 3), axis=1).astype(np.int64)
        nv = len(V)
        code = (key[:, 0] * nv + key[:, 1]) * nv + key[:, 2]
        order = np.argsort(code, kind="stable")
        same = np.flatnonzero(code[order][1:] == code[order][:-1])
        first, second = order[same], order[same + 1]
        by = np.argsort(second)
        first, second = first[by], second[by]
        self.N, self.nt = len(first), nt
        sides = np.stack([first, second], 1)
        tet, loc = sides // 4, sides % 4
        self.tet = torch.from_numpy(tet).to(DEV)
        self.qv = torch.from_numpy(T[tet, loc].astype(np.int64)).to(DEV)
        fv = torch.from_numpy(key[first]).to(DEV)
        self.Q = self.V[self.qv]
        P = self.V[fv]
        area = 0.5 * torch.linalg.norm(torch.cross(P[:, 1] - P[:, 0], P[:, 2] - P[:, 0], dim=1), dim=1)
        tv = self.V[torch.from_numpy(T.astype(np.int64)).to(DEV)]
        self.L = tv[:, 1:] - tv[:, :1]
        self.P0 = tv[:, 0]
        self.vol = torch.linalg.det(self.L) / 6.0
        sign = torch.tensor([1.0, -1.0], dtype=torch.float64, device=DEV)
        self.pf = sign * area[:, None] / (3.0 * self.vol[self.tet])
        verts = torch.cat([fv, self.qv], 1)
        self.cen = P.mean(1)
        self.rad = torch.linalg.norm(self.V[verts] - self.cen[:, None], dim=2).amax(1)
        inc = torch.zeros((self.N, nv), dtype=torch.float32, device=DEV)
        inc.scatter_(1, verts, 1.0)
        self.touch = torch.cat([torch.nonzero(torch.triu(inc[a:a + 2048] @ inc.T > 0.5, a)) +
                                torch.tensor([a, 0], device=DEV) for a in range(0, self.N, 2048)])
        self.facebf = torch.full((nt * 4,), -1, dtype=torch.int64, device=DEV)
        for c in range(2):
            self.facebf[torch.from_numpy(sides[:, c]).to(DEV)] = 2 * torch.arange(self.N, device=DEV) + c
        self.facebf = self.facebf.view(nt, 4)
        self._pts = {}

    def points(self, npts):
        if npts not in self._pts:
            u, w = _rule(npts)
            x = self.P0[:, None] + torch.einsum("pk,tkd->tpd", u, self.L)
            self._pts[npts] = (x, 6.0 * self.vol[:, None] * w)
        return self._pts[npts]

    def bf_points(self, a, npts):
        """Points of basis functions a and w b (3 components) and w div b there: [n, 2 npts, ...]."""
        x, w = self.points(npts)
        t = self.tet[a]
        xs, ws = x[t], w[t]
        pf = self.pf[a][:, :, None]
        b = torch.cat([(pf * ws)[..., None] * (xs - self.Q[a][:, :, None]), (3.0 * pf * ws)[..., None]], -1)
        return xs.flatten(1, 2), b.flatten(1, 2)

    def far(self, kernel, k2, dtype):
        """The 4-point rule on every pair: sum over both points of (b.b' - div div'/k^2) kernel(r)."""
        x, _ = self.points(4)
        cols = x.reshape(-1, 3)
        idx = (self.tet[:, :, None] * 4 + torch.arange(4, device=DEV)).reshape(-1)
        M = torch.empty((self.N, self.N), dtype=dtype, device=DEV)
        _, ball = self.bf_points(torch.arange(self.N, device=DEV), 4)
        wcol = [ball[:, :, c].reshape(-1) * (1.0 if c < 3 else -1.0) for c in range(4)]
        step = max(1, int(1.2e7 // len(cols)) // 8)
        for a in range(0, self.N, step):
            xa, ba = self.bf_points(torch.arange(a, min(a + step, self.N), device=DEV), 4)
            r = torch.zeros((len(xa) * 8, len(cols)), dtype=torch.float64, device=DEV)
            for d in range(3):
                r += (xa.reshape(-1, 3)[:, d, None] - cols[None, :, d]) ** 2
            g = kernel(r.sqrt_()).view(len(xa), 8, -1)
            acc = 0
            for c in range(4):
                f = torch.zeros((len(xa), len(cols)), dtype=dtype, device=DEV)
                for i in range(8):
                    f += ba[:, i, c, None] * g[:, i]
                s = (f[:, idx] * wcol[c]).view(len(xa), self.N, 8).sum(2)
                acc = acc + (s if c < 3 else s / k2)
            M[a:a + len(xa)] = acc
        return M

    def pairs(self, npts, kernel, k2):
        """The npts-point rule on the touching pairs."""
        out = []
        step = max(1, 16_000_000 // (4 * npts * npts))
        for p in self.touch.split(step):
            xa, ba = self.bf_points(p[:, 0], npts)
            xb, bb = self.bf_points(p[:, 1], npts)
            r = torch.cdist(xa, xb, compute_mode="donot_use_mm_for_euclid_dist")
            dot = ba[:, :, :3] @ bb[:, :, :3].transpose(1, 2).contiguous()
            dd = ba[:, :, 3, None] * bb[:, None, :, 3]
            out.append(((dot - dd / k2) * kernel(r)).sum((1, 2)))
        return torch.cat(out)

    def faces(self, weight):
        """Sum over tetrahedra of w F_i . weight(x) . F_j for their interior faces: (rows, cols, values)."""
        x, w = self.points(33)
        bf = self.facebf.clamp(min=0)
        a, side = bf // 2, bf % 2
        F = self.pf[a, side][:, :, None, None] * (x[:, None] - self.Q[a, side][:, :, None])
        val = torch.einsum("tp,tipd,tpd,tjpd->tij", w.to(torch.complex128), F.to(torch.complex128), weight(x),
                           F.to(torch.complex128))
        ok = (self.facebf[:, :, None] >= 0) & (self.facebf[:, None, :] >= 0)
        rows, cols = a[:, :, None].expand_as(val), a[:, None, :].expand_as(val)
        return rows[ok], cols[ok], val[ok]

    def vie(self, omega, table, chi):
        k = complex(omega)
        k2, ik = k * k, 1j * k
        def helm(r):
            v = torch.exp(ik * r) / (4 * math.pi * r)
            return torch.where(r < 1e-12, torch.zeros_like(v), v)
        M = self.far(helm, k2, torch.complex128)

        def exprel(r):
            x = ik * r
            s = torch.zeros_like(x)
            for n in range(30, 2, -1):
                s = (s + 1.0 / math.factorial(n)) * x if n > 3 else s + 1.0 / 6.0
            small = s * x ** 3
            big = torch.exp(x) - 1 - x - x * x / 2
            v = torch.where(x.abs() < 2.0, small, big) / (4 * math.pi * r)
            return torch.where(r < 1e-12, torch.zeros_like(v), v)
        G = table
        near = self.pairs(4, exprel, k2) + (G[:, 0] - G[:, 1] / k2) + ik * (G[:, 2] - G[:, 3] / k2) + \
            ik * ik * (G[:, 4] - G[:, 5] / k2)
        a, b = self.touch[:, 0], self.touch[:, 1]
        M[a, b] = near
        M[b, a] = near
        if chi is not None:
            r, c, v = self.faces(lambda x: 1.0 / chi(x))
            M.index_put_((r, c), -v / (omega.real if isinstance(omega, complex) else omega) ** 2, accumulate=True)
        return M

    def rhs(self, omega, spec):
        """<b, E> of each plane wave: [nrhs, N]."""
        out = []
        for e0, d in spec:
            e = torch.tensor(np.asarray(e0, complex), device=DEV)
            dd = torch.tensor(np.asarray(d, float), device=DEV)
            x, b = self.bf_points(torch.arange(self.N, device=DEV), 33)
            ph = torch.exp(1j * omega * (x @ dd))
            out.append(((b[..., :3].to(torch.complex128) @ e) * ph).sum(1))
        return torch.stack(out)

    def emt(self, omega):
        """k Im of the scattered-power integrals, 16-point rule on touching pairs (k radius <= 5)."""
        k = float(omega)
        if float(self.rad.max()) * k > 5.0:
            return None

        def sine(r):
            kr = k * r
            return k * torch.where(kr < 2e-2, (1 - kr * kr / 6) * k / (4 * math.pi), torch.sin(kr) / (4 * math.pi * r))
        Q = self.far(sine, k * k, torch.float64)
        near = self.pairs(16, sine, k * k)
        a, b = self.touch[:, 0], self.touch[:, 1]
        Q[a, b] = near
        Q[b, a] = near
        return Q

    def power(self, omega, spec, J):
        Q = self.emt(omega)
        if Q is None:
            return None
        b = self.rhs(omega, spec)
        out = []
        for j in range(len(spec)):
            y = torch.complex(Q @ J[j].real, Q @ J[j].imag)
            scat = 0.5 * ZVAC * ((J[j].conj() * y).real.sum() + (J[j].abs() ** 2 * Q.diagonal()).sum())
            ext = 0.5 * (J[j].conj() * b[j]).real.sum()
            out.append([float(ext - scat), float(scat)])
        return np.array(out)


def _chi(name):
    """eps - 1 at points [..., 3], its three diagonal values."""
    def f(x):
        one = torch.ones(x.shape[:-1] + (3,), dtype=torch.complex128, device=x.device)
        if name == "iso":
            return one * (3 + 0.1j)
        if name == "diag":
            return one * torch.tensor([3 + 0.05j, 4 + 0.05j, 5 + 0.05j], device=x.device)
        if name == "sincos":
            return one * (3 + 0.1j + 2 * torch.sin(math.pi * x[..., 0]) * torch.cos(math.pi * x[..., 1]))[..., None]
        if name == "janus":
            return torch.where((x[..., 2] > 0)[..., None], one * (3 + 0.1j), one * (11 + 1j))
        v = 3 + 0.1j + 0.5 * torch.sin(2 * x[..., 0]) * torch.cos(x[..., 1]) + 0.3 * x[..., 2] ** 2
        return one * v[..., None]
    return f


def _exact_scatter(V, T, omega, mat, spec, table):
    e = _Exact(V, T)
    M = e.vie(omega, table, _chi(mat))
    B = e.rhs(omega, spec) * (1j / (omega * ZVAC))
    J = torch.linalg.solve(M, B.T.contiguous()).T.contiguous()
    del M
    return J, e.power(omega, spec, J)


def _static_table(V, T):
    """The static records, which a program has before its first frequency, are an input here."""
    return torch.from_numpy(_geometry(V, T).static_table()).to(DEV)


def exact(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    if kind == "cold":
        return None      # singular integrals: the cubature's own error, not rounding, is what a formula would show
    if kind == "batch":
        meshes = _batch_meshes(case, seed)
        spec = _planewaves(case["nrhs"], rng)
        om = _omegas(case)
        power = np.zeros((len(om), len(meshes), len(spec), 2))
        Js = []
        for i, (V, T, m) in enumerate(meshes):
            table = _static_table(V, T)
            for f, w in enumerate(om):
                J, p = _exact_scatter(V, T, float(w), m, spec, table)
                power[f, i] = p
            Js.append(J.cpu().numpy().T)
        return {"power": power, "info": None, "J": Js}
    V, T = _mesh(case["n"], case["radius"], seed)
    if kind == "fields":
        e = _Exact(V, T)
        X, J = _field_inputs(case, e.N, seed)
        return _exact_fields(e, case, X, J, _planewaves(case["nrhs"], rng))
    table = _static_table(V, T)
    if kind == "scatter":
        J, p = _exact_scatter(V, T, case["omega"], case["mat"], _planewaves(case["nrhs"], rng), table)
        return {"J": J, "power": p}
    e = _Exact(V, T)
    if kind == "assemble":
        w = complex(case["omega"], case["omega_im"])
        return {"M": e.vie(w if case["omega_im"] else case["omega"], table, _chi(case["mat"]))}
    # rytov: DR = (1 + S^-1 V S^-1 G)^-1 (S^-1 R S^-1)^H
    w, chi = case["omega"], _chi(case["mat"])

    def dense(weight):
        A = torch.zeros((e.N, e.N), dtype=torch.complex128, device=DEV)
        r, c, v = e.faces(weight)
        return A.index_put_((r, c), v, accumulate=True)
    S = dense(lambda x: torch.ones_like(chi(x)))
    Vb = dense(lambda x: -w * w * chi(x))
    R = dense(lambda x: (4 * w / (math.pi * ZVAC)) * chi(x).imag.to(torch.complex128))
    G = e.vie(w, table, None)
    Si = torch.linalg.inv(S)
    A = torch.eye(e.N, dtype=torch.complex128, device=DEV) + Si @ (Vb @ (Si @ G))
    DR = torch.linalg.solve(A, ((Si @ R) @ Si).conj().T.contiguous())
    Q = e.emt(w)
    s = ZVAC * float((torch.tril(DR).real * Q).sum()) if Q is not None else None
    return {"DR": DR.T.contiguous(), "power": None if s is None else np.array([-s, s])}


def _exact_fields(e, case, X, J, spec):
    k = case["omega"]
    Jd = torch.from_numpy(J).to(DEV)
    Xd = torch.from_numpy(X).to(DEV)
    E = torch.zeros((len(X), 3), dtype=torch.complex128, device=DEV)
    H = torch.zeros_like(E)
    allb = torch.arange(e.N, device=DEV)
    far_x, far_b = e.bf_points(allb, 4)
    near_x, near_b = e.bf_points(allb, 16)

    def add(p, xs, b, j):
        R = Xd[p] - xs
        r = torch.linalg.norm(R, dim=-1, keepdim=True)
        u, b = R / r, b[..., :3]
        kr = k * r
        g = torch.exp(1j * kr) / (4 * math.pi * r)
        ub = (u * b).sum(-1, keepdim=True)
        e_ = g * ((1 + 1j / kr - 1 / kr ** 2) * b + (-1 - 3j / kr + 3 / kr ** 2) * u * ub)
        h_ = -(1 + 1j / kr) * g * torch.cross(u, b, dim=-1)
        E[p] += 1j * k * ZVAC * (j[:, None, None] * e_).sum((0, 1))
        H[p] += -1j * k * (j[:, None, None] * h_).sum((0, 1))
    for p in range(len(X)):
        far = torch.linalg.norm(Xd[p] - e.cen, dim=1) > 10.0 * e.rad
        add(p, far_x[far], far_b[far], Jd[far])
        add(p, near_x[~far], near_b[~far], Jd[~far])
    for e0, d in spec:
        e0 = torch.tensor(np.asarray(e0, complex), device=DEV)
        dd = torch.tensor(np.asarray(d, float), device=DEV)
        Ei = torch.exp(1j * k * (Xd @ dd))[:, None] * e0
        E += Ei
        H += torch.cross(dd.to(torch.complex128).expand_as(Ei), Ei, dim=1) / ZVAC
    return {"E": E.cpu().numpy(), "H": H.cpu().numpy()}
