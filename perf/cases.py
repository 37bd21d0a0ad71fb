"""Performance cases of the dense PMCHWT framework, each through its public
Python entry points (bem_amd.Context).

Kinds of work and what they stand for:

  pipeline   one parameter point of a size or refractive-index scan: assemble,
             plane waves, LU, multi-RHS solve (refined for FP32 factors), far
             field and Mueller matrices of all orientations
  more       further orientations of a particle whose factors are kept
  gradient   one step of a fit: the pipeline and the adjoint gradient
  dense      the LU drop-in on a caller's own host matrix
  assemble   the assembly drop-in: Z on the host
  farfield   the far-field drop-in on a caller's coefficients
  precond    block-Jacobi preconditioned GMRES on the dense operator

The meshes are the generators' (icosphere, hexagonal prism) and a
latitude-longitude ellipsoid whose size is any multiple of 6.  A state is a
context with its mesh set; every input depends on the seed.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bem-cpp_amd"))
import bem_amd  # noqa: E402


def _case(name, kind, mesh="sphere", ref=0, nlat=0, nlon=0, aspect=1.0, quad=7, ka=1.0, m_re=1.3116, m_im=0.0,
          na=1, nb=1, ng=1, ntheta=181, precision="fp32", mirror=False, n=0, nrhs=0, block=0):
    c = dict(kind=kind, mesh=mesh, ref=ref, nlat=nlat, nlon=nlon, aspect=aspect, quad=quad, ka=ka, m_re=m_re,
             m_im=m_im, na=na, nb=nb, ng=ng, ntheta=ntheta, precision=precision, mirror=mirror, n=n, nrhs=nrhs,
             block=block)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # a small sphere in the lab frame: launches, copies and latency
        _case("pipe sphere 240", "pipeline", ref=1, ka=1.0, m_im=0.01),
        # FP64 factors, 13-point quadrature
        _case("pipe sphere 960 fp64 q13", "pipeline", ref=2, ka=1.0, quad=13, precision="fp64"),
        # the single-orientation run of an absorbing sphere (2N = 3840)
        _case("pipe sphere 3840", "pipeline", ref=3, ka=5.0, m_im=0.01),
        # an orientation average of a hexagonal column (2N = 4608, 128 RHS)
        _case("pipe hex 4608 x64", "pipeline", mesh="hex", ref=3, aspect=1.4286, ka=5.0, na=8, nb=8),
        # a mesh of no round size, 4-point quadrature, 15 orientations, mirror averaging (2N = 6042)
        _case("pipe ellipsoid 6042 x15", "pipeline", mesh="ellipsoid", nlat=20, nlon=53, aspect=1.6, quad=4, ka=4.0,
              m_re=1.5, m_im=0.002, na=5, nb=3, ntheta=91, mirror=True),
        # the largest: a hexagonal plate, 2N = 18432, 64 orientations
        _case("pipe hex 18432 x64", "pipeline", mesh="hex", ref=4, aspect=0.7, ka=10.0, na=8, nb=8),
        # 33 more orientations on the plate's kept factors
        _case("more hex 18432 x33", "more", mesh="hex", ref=4, aspect=0.7, ka=10.0, na=11, nb=3),
        # a refractive-index fit: Mueller loss and its gradient (2N = 3840)
        _case("gradient sphere 3840", "gradient", ref=3, ka=3.0, m_re=1.33, m_im=0.005),
        # a caller's own matrix through the FP64 LU drop-in
        _case("dense 1999 x33 fp64", "dense", n=1999, nrhs=33, precision="fp64"),
        # Z of a small particle handed to the caller
        _case("assemble ellipsoid 918", "assemble", mesh="ellipsoid", nlat=10, nlon=17, aspect=0.8, ka=2.0, m_im=0.02),
        # far field of 12 coefficient sets over 721 directions each
        _case("farfield hex 2304", "farfield", mesh="hex", ref=3, aspect=1.0, ka=4.0, na=6, ntheta=721),
        # iterative solution without a full factorisation (2N = 4608)
        _case("precond hex 4608", "precond", mesh="hex", ref=3, aspect=1.0, ka=3.0, na=2, block=120),
    ]


def draw(rng):
    kind = rng.choice(["pipeline", "pipeline", "pipeline", "more", "gradient", "dense", "assemble", "farfield",
                       "precond"])
    c = _case(None, kind)
    top = {"pipeline": 8000, "more": 5000, "gradient": 2500, "assemble": 900, "farfield": 5000, "precond": 2400,
           "dense": 3000}[kind]
    if kind == "dense":
        c["n"] = int(round(math.exp(rng.uniform(math.log(60), math.log(top)))))
        c["nrhs"] = rng.choice([1, 2, 5, 33, 70])
        c["precision"] = rng.choice(["fp32", "fp64"])
        return c
    N = math.exp(rng.uniform(math.log(100), math.log(top)))
    c["aspect"] = round(rng.uniform(0.6, 1.7), 3)
    c["mesh"] = rng.choice(["sphere", "hex", "ellipsoid", "ellipsoid"])
    if c["mesh"] == "ellipsoid":  # N = 3 nlon (nlat - 1)
        c["nlat"] = max(4, int(round(math.sqrt(N / 7.5))))
        c["nlon"] = max(5, int(round(N / (3 * (c["nlat"] - 1)))))
        N = 3 * c["nlon"] * (c["nlat"] - 1)
    else:
        base = 30 if c["mesh"] == "sphere" else 36
        c["ref"] = max(1, int(math.log(N / base, 4)))
        N = base * 4 ** c["ref"]
    c["quad"] = rng.choice([4, 7, 7, 13])
    c["ka"] = round(rng.uniform(0.03, 0.1) * math.sqrt(N), 4)
    c["m_re"] = round(rng.uniform(1.2, 1.6), 4)
    c["m_im"] = rng.choice([0.0, round(rng.uniform(0.001, 0.05), 4)])
    c["na"], c["nb"], c["ng"] = rng.choice([(1, 1, 1), (2, 1, 1), (5, 1, 1), (3, 5, 1), (4, 2, 3), (8, 8, 1)])
    c["ntheta"] = rng.choice([19, 91, 181, 361])
    c["mirror"] = rng.random() < 0.3
    c["precision"] = rng.choice(["fp32", "fp32", "fp64"]) if N < 4000 else "fp32"
    if kind in ("gradient", "precond"):
        c["na"], c["nb"], c["ng"] = rng.choice([(1, 1, 1), (2, 1, 1), (3, 2, 1)])
    if kind == "precond":
        c["block"] = rng.randint(40, 130)
    return c


# -- inputs ------------------------------------------------------------------


def _split(v, t, project):
    """Every triangle into four; new vertices at the edge midpoints."""
    e = np.sort(np.concatenate([t[:, [0, 1]], t[:, [1, 2]], t[:, [2, 0]]]), axis=1)
    u, inv = np.unique(e, axis=0, return_inverse=True)
    mid = 0.5 * (v[u[:, 0]] + v[u[:, 1]])
    if project:
        mid /= np.linalg.norm(mid, axis=1, keepdims=True)
    ab, bc, ca = (len(v) + inv.reshape(3, -1)).astype(np.int32)
    a, b, c = t.T
    out = np.stack([a, ab, ca, b, bc, ab, c, ca, bc, ab, bc, ca], axis=1)
    return np.concatenate([v, mid]), out.reshape(-1, 3)


def _mesh(case, rng):
    """Vertices and outward triangles, stretched along each axis by up to 2 %
    as the seed says."""
    kind = case["mesh"]
    if kind == "sphere":
        g = 0.5 * (1 + math.sqrt(5))
        v = np.array([(-1, g, 0), (1, g, 0), (-1, -g, 0), (1, -g, 0), (0, -1, g), (0, 1, g), (0, -1, -g), (0, 1, -g),
                      (g, 0, -1), (g, 0, 1), (-g, 0, -1), (-g, 0, 1)], float)
        v /= np.linalg.norm(v[0])
        t = np.array([(0, 11, 5), (0, 5, 1), (0, 1, 7), (0, 7, 10), (0, 10, 11), (1, 5, 9), (5, 11, 4), (11, 10, 2),
                      (10, 7, 6), (7, 1, 8), (3, 9, 4), (3, 4, 2), (3, 2, 6), (3, 6, 8), (3, 8, 9), (4, 9, 5),
                      (2, 4, 11), (6, 2, 10), (8, 6, 7), (9, 8, 1)], np.int32)
        for _ in range(case["ref"]):
            v, t = _split(v, t, True)
    elif kind == "hex":
        a = (8 * math.pi / (27 * case["aspect"])) ** (1 / 3)
        h = case["aspect"] * a * math.sqrt(3)
        ring = [(a * math.cos(math.pi * i / 3), a * math.sin(math.pi * i / 3)) for i in range(6)]
        v = np.array([(0, 0, h / 2)] + [(x, y, h / 2) for x, y in ring] + [(0, 0, -h / 2)]
                     + [(x, y, -h / 2) for x, y in ring], float)
        f = []
        for i in range(6):
            t1, t2, b1, b2 = 1 + i, 1 + (i + 1) % 6, 8 + i, 8 + (i + 1) % 6
            f += [(0, t1, t2), (7, b2, b1), (t1, b1, b2), (t1, b2, t2)]
        t = np.array(f, np.int32)
        for _ in range(case["ref"]):
            v, t = _split(v, t, False)
    else:
        nlat, nlon = case["nlat"], case["nlon"]
        th = math.pi * np.arange(1, nlat) / nlat
        ph = 2 * math.pi * np.arange(nlon) / nlon
        s, z = np.sin(th)[:, None], np.cos(th)[:, None]
        body = np.stack([s * np.cos(ph), s * np.sin(ph), z + 0 * ph], axis=2).reshape(-1, 3)
        v = np.concatenate([[(0.0, 0.0, 1.0)], body, [(0.0, 0.0, -1.0)]])
        v[:, 2] *= case["aspect"]
        f, last = [], len(v) - 1
        for j in range(nlon):
            k = (j + 1) % nlon
            f += [(0, 1 + j, 1 + k), (last, 1 + (nlat - 2) * nlon + k, 1 + (nlat - 2) * nlon + j)]
            for i in range(nlat - 2):
                p, q = 1 + i * nlon, 1 + (i + 1) * nlon
                f += [(p + j, q + j, q + k), (p + j, q + k, p + k)]
        t = np.array(f, np.int32)
    v = v * rng.uniform(0.98, 1.02, 3)
    return np.ascontiguousarray(v), np.ascontiguousarray(t)


def _inputs(case, seed):
    """Everything of a case that depends on the seed, as numpy arrays."""
    rng = np.random.default_rng([seed, 77])
    d = {}
    if case["kind"] == "dense":
        n = case["n"]
        z = (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))) * (0.35 / math.sqrt(n))
        z[np.arange(n), np.arange(n)] += 1.0
        d["Z"] = np.ascontiguousarray(z[rng.permutation(n)])
        d["B"] = rng.standard_normal((n, case["nrhs"])) + 1j * rng.standard_normal((n, case["nrhs"]))
        return d
    d["verts"], d["tris"] = _mesh(case, rng)
    d["ka"] = case["ka"] * (1 + 0.02 * rng.uniform(-1, 1))
    d["m"] = complex(case["m_re"] * (1 + 0.01 * rng.uniform(-1, 1)), case["m_im"] * (1 + 0.1 * rng.uniform(-1, 1)))
    d["theta"] = np.linspace(0.0, np.pi, case["ntheta"])
    na, nb, ng = case["na"], case["nb"], case["ng"]
    if na * nb * ng == 1:
        d["RT"], d["w"] = np.eye(3)[None], np.ones(1)
    else:  # Euler angles: uniform in alpha and gamma, Gauss-Legendre in cos beta
        x, wx = np.polynomial.legendre.leggauss(nb)
        al = 2 * np.pi * (np.arange(na) + rng.uniform()) / na
        ga = 2 * np.pi * (np.arange(ng) + rng.uniform()) / ng
        rt, w = [], []
        for a in al:
            for xb, wb in zip(x, wx):
                for g in ga:
                    ca, sa, cg, sg, cb, sb = np.cos(a), np.sin(a), np.cos(g), np.sin(g), xb, math.sqrt(1 - xb * xb)
                    rz1 = np.array([[ca, -sa, 0], [sa, ca, 0], [0, 0, 1]])
                    ry = np.array([[cb, 0, sb], [0, 1, 0], [-sb, 0, cb]])
                    rz2 = np.array([[cg, -sg, 0], [sg, cg, 0], [0, 0, 1]])
                    rt.append((rz1 @ ry @ rz2).T)
                    w.append(wb / 2 / (na * ng))
        d["RT"], d["w"] = np.ascontiguousarray(np.array(rt)), np.array(w)
    if case["kind"] == "farfield":
        N, calls = 3 * len(d["tris"]) // 2, 2 * len(d["w"])
        for f in ("cJ", "cM"):
            d[f] = (rng.standard_normal((calls, N)) + 1j * rng.standard_normal((calls, N))) / N
        r = rng.standard_normal((len(d["w"]), case["ntheta"], 3))
        d["rhat"] = r / np.linalg.norm(r, axis=2, keepdims=True)
        d["k"] = complex(d["ka"], case["m_im"] * d["ka"])
    if case["kind"] == "gradient":
        d["weight"] = np.sin(d["theta"]) * (1 + 0.1 * rng.uniform(size=len(d["theta"])))
    return d


def _tol(case):
    return 1e-12 if case["kind"] in ("gradient", "dense") else 1e-10


def _assemble(s):
    s["ctx"].assemble(complex(s["ka"]), s["ka"] * s["m"], 1.0, 1.0 / abs(s["m"]))


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    s["ctx"] = bem_amd.Context(0)
    if case["kind"] == "dense":
        return s
    s["ctx"].set_mesh(s["verts"], s["tris"], case["quad"])
    s["kh"], s["e0"] = bem_amd.planewave_orient_rhs(s["RT"])
    if case["kind"] in ("more", "precond"):
        _assemble(s)
    if case["kind"] == "more":
        s["ctx"].factor(case["precision"])
    if case["kind"] == "precond":
        s["ctx"].rhs_planewave(s["ka"], 1.0, s["kh"], s["e0"])
    return s


# -- one pass ----------------------------------------------------------------


def _solve_and_scatter(s):
    ctx, case = s["ctx"], s["case"]
    ctx.solve(None, ir_tol=_tol(case), ir_max=10, return_X=False, nrhs=len(s["kh"]))
    return ctx.orient_mueller(s["ka"], 1.0, s["RT"], s["w"], s["theta"], gamma_mirror=case["mirror"])


def run(s):
    ctx, case = s["ctx"], s["case"]
    kind = case["kind"]
    if kind == "dense":
        ctx.set_Z(s["Z"])
        ctx.factor(case["precision"])
        return ctx.solve(s["B"], ir_tol=_tol(case), ir_max=10 if case["precision"] == "fp32" else 0)[0]
    if kind == "assemble":
        _assemble(s)
        return ctx.get_Z()
    if kind == "farfield":
        return ctx.farfield(s["cJ"], s["cM"], s["rhat"], s["k"], 1.0, len(s["cJ"]), len(s["w"]))
    if kind == "precond":
        ctx.block_jacobi(radius_mult=2.0, max_block_rwg=case["block"], overlap_layers=1)
        return ctx.solve_gmres(None, tol=1e-10, restart=60, max_iter=600, nrhs=len(s["kh"]),
                               precond="block")[0]
    if kind == "more":
        ctx.rhs_planewave(s["ka"], 1.0, s["kh"], s["e0"])
        return _solve_and_scatter(s)
    _assemble(s)
    ctx.rhs_planewave(s["ka"], 1.0, s["kh"], s["e0"])
    ctx.factor(case["precision"])
    M = _solve_and_scatter(s)
    if kind == "pipeline":
        return M
    dL = np.zeros_like(M)  # L = sum_t weight_t log M11(theta_t)
    dL[0, 0] = s["weight"] / M[0, 0]
    return {"M": M, "grad": ctx.mueller_grad(dL)}


def _num_rwg(case):
    if case["mesh"] == "ellipsoid":
        return 3 * case["nlon"] * (case["nlat"] - 1)
    return (30 if case["mesh"] == "sphere" else 36) * 4 ** case["ref"]


def work(case):
    """Inputs read once and outputs written once; the arithmetic of one
    assembly (both wavenumbers, symmetry used), one LU, the solves and the far
    field, in real operations."""
    kind = case["kind"]
    if kind == "dense":
        n, r = case["n"], case["nrhs"]
        return {"bytes": 16.0 * n * n + 32.0 * n * r, "flops": 8 / 3 * n ** 3 + 8.0 * n * n * r}
    N, o = _num_rwg(case), case["na"] * case["nb"] * case["ng"]
    n, q, r = 2 * N, {4: 4, 13: 13}.get(case["quad"], 7), 2 * o
    geom = 8.0 * 3 * (2 * N / 3) * 4
    asm = 74.0 * (2 * N / 3 * q) ** 2 / 2 * 2
    solve = 8.0 * n * n * r
    ff = 100.0 * (2 * N / 3 * q) * o * case["ntheta"]
    out = 8.0 * 16 * case["ntheta"]
    zb = 16.0 * n * n
    if kind == "farfield":
        return {"bytes": geom + 32.0 * N * r + 48.0 * r * case["ntheta"], "flops": ff}
    if kind == "assemble":
        return {"bytes": geom + zb, "flops": asm}
    if kind == "more":
        return {"bytes": geom + zb + out, "flops": 2 * solve + ff}
    if kind == "precond":
        return {"bytes": zb, "flops": 10 * solve}
    flops = asm + 8 / 3 * n ** 3 + solve + ff
    if kind == "gradient":
        return {"bytes": geom + 3 * zb + out, "flops": flops + 2 * solve + asm}
    return {"bytes": geom + zb + out, "flops": flops}


# -- the same in 64 bits, plain torch ------------------------------------------

_R, _S, _U = 0.260345966079038, 0.479308067841923, 0.065130102902216
_V, _E, _F, _G = 0.869739794195568, 0.048690315425316, 0.312865496004875, 0.638444188569809
_RULES = {
    4: ([(1 / 3, 1 / 3), (0.6, 0.2), (0.2, 0.6), (0.2, 0.2)], [-27 / 48] + 3 * [25 / 48]),
    7: ([(1 / 3, 1 / 3), (0.059715871789770, 0.470142064105115), (0.470142064105115, 0.059715871789770),
         (0.470142064105115, 0.470142064105115), (0.797426985353087, 0.101286507323456),
         (0.101286507323456, 0.797426985353087), (0.101286507323456, 0.101286507323456)],
        [0.225] + 3 * [0.13239415278851] + 3 * [0.12593918054483]),
    13: ([(1 / 3, 1 / 3), (_R, _R), (_R, _S), (_S, _R), (_U, _U), (_U, _V), (_V, _U), (_E, _F), (_F, _E), (_G, _F),
          (_F, _G), (_E, _G), (_G, _E)],
         [-0.149570044467670] + 3 * [0.175615257433204] + 3 * [0.053347235608839] + 6 * [0.077113760890257]),
}


def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


class _Basis:
    """Quadrature points and RWG halves of a closed mesh (edges in sorted order)."""

    def __init__(self, verts, tris, order):
        pts, wts = _RULES[order]
        p = verts[tris]  # T, 3, 3
        cross = np.cross(p[:, 1] - p[:, 0], p[:, 2] - p[:, 0])
        area = 0.5 * np.linalg.norm(cross, axis=1)
        l1, l2 = np.array(pts).T
        x = np.einsum("kq,tkd->tqd", np.stack([1 - l1 - l2, l1, l2]), p)
        e = np.stack([tris, np.roll(tris, -1, axis=1)], axis=2).reshape(-1, 2)
        e = np.sort(e, axis=1)
        _, first, rwg = np.unique(e, axis=0, return_index=True, return_inverse=True)
        length = np.linalg.norm(verts[e[:, 0]] - verts[e[:, 1]], axis=1)
        sign = -np.ones(len(e))
        sign[first] = 1.0  # the edge's first triangle is the plus one
        half_area = np.repeat(area, 3)
        t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(_dev())  # noqa: E731
        self.T, self.nq, self.N = len(tris), len(pts), len(e) // 2
        self.x, self.jw = t(x), t(area[:, None] * np.array(wts))
        self.wq, self.area, self.corner = t(np.array(wts)), t(area), t(p)
        self.c = t((sign * length / (2 * half_area)).reshape(-1, 3))
        self.free = t(np.roll(p, -2, axis=1))  # half j: edge (j, j + 1), free vertex j + 2
        self.rwg = t(rwg.reshape(-1).astype(np.int64))
        # f[t, a, q] = c (x - p) jw and its divergence 2 c jw
        self.f = self.c[:, :, None, None] * (self.x[:, None] - self.free[:, :, None]) * self.jw[:, None, :, None]
        self.div = 2 * self.c[:, :, None] * self.jw[:, None, :]

    def to_rwg(self, h):
        """Sums the halves (first axis, 3 T) of each RWG."""
        out = torch.zeros((self.N,) + h.shape[1:], dtype=h.dtype, device=h.device)
        return out.index_add(0, self.rwg, h)


def _static(b):
    """int 1/|r - r'| and int (r - r')-weighted terms over a point's own
    triangle: P(r) in closed form and V(r) = r P - grad sum_q A w_q |r_q - r|."""
    T, q = b.T, b.nq
    r = b.x
    normal = torch.linalg.cross(b.corner[:, 1] - b.corner[:, 0], b.corner[:, 2] - b.corner[:, 0])
    normal = normal / normal.norm(dim=1, keepdim=True)
    P = torch.zeros(T, q, dtype=torch.float64, device=r.device)
    for i in range(3):
        a, c = b.corner[:, i], b.corner[:, (i + 1) % 3]
        t = (c - a) / (c - a).norm(dim=1, keepdim=True)
        m = torch.linalg.cross(normal, t)
        d = ((r - a[:, None]) * m[:, None]).sum(2)
        sp, sm = ((c[:, None] - r) * t[:, None]).sum(2), ((a[:, None] - r) * t[:, None]).sum(2)
        Rp, Rm = (c[:, None] - r).norm(dim=2), (a[:, None] - r).norm(dim=2)
        P = P + d * torch.log((Rp + sp) / (Rm + sm))
    diff = r[:, :, None] - r[:, None]  # point, source
    dist = diff.norm(dim=3)
    unit = torch.where(dist[..., None] > 0, diff / dist.clamp_min(1e-300)[..., None], torch.zeros_like(diff))
    grad = b.area[:, None, None] * (b.wq[None, None, :, None] * unit).sum(2)
    return P, r * P[..., None] - grad


def _L_K(b, kr, ki):
    """L and K of one wavenumber k = kr + i ki (0-dim tensors), N x N."""
    T, q = b.T, b.nq
    i4pi = 1 / (4 * math.pi)
    k = torch.complex(kr, ki)
    c128 = torch.complex128
    x = b.x.reshape(-1, 3)
    f = b.f  # T, 3, q, 3
    src_cross = torch.linalg.cross(b.x[:, None].expand_as(f), f)  # r x f at the source point
    tst_cross = torch.linalg.cross(f, b.x[:, None].expand_as(f))  # f x r at the test point
    test_G = torch.cat([f, b.div[..., None]], 3).permute(0, 1, 3, 2).reshape(T, 12, q)  # (half, component)
    test_g = torch.cat([tst_cross, f], 3).permute(0, 1, 3, 2).reshape(T, 18, q)
    src_G = torch.cat([f, b.div[..., None]], 3).permute(0, 3, 2, 1).reshape(T, 4, q, 3)
    src_g = torch.cat([f, -src_cross], 3).permute(0, 3, 2, 1).reshape(T, 6, q, 3)
    step = max(1, int(2.5e7 // (q * q * T)))
    Lh, Kh = [], []
    for t0 in range(0, T, step):
        t1 = min(T, t0 + step)
        n = t1 - t0
        d = x[t0 * q:t1 * q, None] - x[None]
        r2 = (d * d).sum(2)
        zero = r2 < 1e-24
        R = torch.where(zero, torch.ones_like(r2), r2).sqrt()
        amp = torch.exp(-ki * R) * i4pi / R
        G = torch.complex(amp * torch.cos(kr * R), amp * torch.sin(kr * R))
        g = G * (1j * k - 1 / R) / R
        own = torch.zeros(n, q, T, q, dtype=torch.bool, device=x.device)
        own[torch.arange(n), :, torch.arange(t0, t1), :] = True
        own = own.reshape(n * q, T * q)
        G = torch.where(own, G - (i4pi / R).to(c128), G)
        G = torch.where(zero, torch.complex(torch.zeros_like(kr), kr * i4pi), G)
        g = torch.where(own, torch.zeros_like(g), g)
        for kern, test, srcs, comp, out in ((G, test_G, src_G, 4, Lh), (g, test_g, src_g, 6, Kh)):
            a = torch.bmm(test[t0:t1].to(c128), kern.reshape(n, q, T * q))  # n, 3 comp, T q
            a = a.reshape(n, 3, comp, T, q).permute(3, 0, 1, 2, 4)  # T, n, 3, comp, q
            if comp == 4:
                v = torch.bmm(a[:, :, :, :3].reshape(T, n * 3, 3 * q), srcs[:, :3].reshape(T, 3 * q, 3).to(c128))
                w = torch.bmm(a[:, :, :, 3:].reshape(T, n * 3, q), srcs[:, 3].to(c128))
                v = 1j * k * v - 1j / k * w
            else:
                v = torch.bmm(a.reshape(T, n * 3, 6 * q), srcs.reshape(T, 6 * q, 3).to(c128))
            v = v.reshape(T, n, 3, 3).permute(1, 2, 0, 3).reshape(n * 3, T * 3)
            out.append(b.to_rwg(v.T).T)  # sources summed to their RWGs
    L, K = torch.cat(Lh), torch.cat(Kh)
    # the singular part on a triangle with itself
    P, V = _static(b)
    SP, SPr = (b.jw * P).sum(1), (b.jw[..., None] * P[..., None] * b.x).sum(1)
    SV, SrV = (b.jw[..., None] * V).sum(1), (b.jw * (b.x * V).sum(2)).sum(1)
    sym = (b.free[:, :, None] + b.free[:, None]) @ (SPr + SV)[:, None, :, None]
    papb = b.free @ b.free.transpose(1, 2)
    vec = SrV[:, None, None] - 0.5 * sym[..., 0] + papb * SP[:, None, None]
    cc = b.c[:, :, None] * b.c[:, None] * i4pi
    corr = cc * (1j * k * vec - 4j / k * SP[:, None, None])  # T, 3, 3
    rows = torch.arange(3 * T, device=x.device).reshape(T, 3, 1).expand(T, 3, 3)
    cols = b.rwg.reshape(T, 1, 3).expand(T, 3, 3)
    L = L.index_put((rows, cols), corr, accumulate=True)
    L, K = b.to_rwg(L), b.to_rwg(K)
    return 0.5 * (L + L.T), 0.5 * (K + K.T)


def _system(b, ka, mr, mi):
    eta = 1 / torch.sqrt(mr * mr + mi * mi)
    L, K = _L_K(b, ka, torch.zeros_like(ka))
    Li, Ki = _L_K(b, ka * mr, ka * mi)
    K = K + Ki
    return torch.cat([torch.cat([L + eta * Li, -K], 1), torch.cat([K, L + Li / eta], 1)])


def _plane_waves(b, ka, kh, e0):
    ph = ka * (b.x @ kh.T)  # T, q, rhs
    wave = torch.complex(torch.cos(ph), torch.sin(ph))
    out = []
    for e in (e0, torch.linalg.cross(kh, e0)):
        amp = torch.einsum("taqd,jd->taqj", b.f, e)
        out.append(b.to_rwg((amp * wave[:, None]).sum(2).reshape(3 * b.T, -1)))
    return torch.cat(out)


def _far(b, cJ, cM, rhat, k):
    """F of coefficient columns cJ, cM (N x 2 o) in directions rhat (o, d, 3)."""
    out = []
    for o in range(rhat.shape[0]):
        pair = []
        for c in (cJ, cM):
            h = c[b.rwg][:, 2 * o:2 * o + 2].reshape(b.T, 3, -1)
            pair.append(torch.einsum("taqd,tac->tqdc", b.f.to(h.dtype), h).reshape(b.T * b.nq, -1))
        J, M = [], []
        for r in rhat[o].split(max(1, int(4e7 // (b.T * b.nq)))):
            ph = b.x.reshape(-1, 3) @ r.T
            wave = torch.exp(-1j * k * ph).T
            J.append(wave @ pair[0])
            M.append(wave @ pair[1])
        nd = rhat.shape[1]
        J, M = (torch.cat(v).reshape(nd, 3, -1).permute(2, 0, 1) for v in (J, M))
        r = rhat[o].to(J.dtype)
        F = J - r * (J * r).sum(2, keepdim=True) - torch.linalg.cross(r.expand_as(M), M)
        out.append(-1j * k / (4 * math.pi) * F)
    return torch.cat(out)


def _mueller(b, X, s, mirror, ka):
    dev = b.x.device
    th = torch.from_numpy(s["theta"]).to(dev)
    RT = torch.from_numpy(s["RT"]).to(dev)
    z = torch.zeros_like(th)
    lab = torch.stack([torch.stack([th.sin(), z, th.cos()], 1), torch.stack([th.cos(), z, -th.sin()], 1)])
    rhat, par = torch.einsum("oij,ntj->noti", RT, lab)
    perp = RT[:, :, 1]
    F = _far(b, X[:b.N], X[b.N:], rhat, torch.complex(ka, torch.zeros_like(ka)))
    F = F.reshape(len(RT), 2, len(th), 3)
    sp = -1j * ka * (F * par[:, None]).sum(3)
    sq = -1j * ka * (F * perp[:, None, None]).sum(3)
    S2, S4, S3, S1 = sp[:, 0], sq[:, 0], sp[:, 1], sq[:, 1]
    a1, a2, a3, a4 = (v.abs() ** 2 for v in (S1, S2, S3, S4))
    p = lambda u, v: u * v.conj()  # noqa: E731
    m = [(a1 + a2 + a3 + a4) / 2, (a2 - a1 + a4 - a3) / 2, (p(S2, S3) + p(S1, S4)).real, (p(S2, S3) - p(S1, S4)).imag,
         (a2 - a1 - a4 + a3) / 2, (a2 + a1 - a4 - a3) / 2, (p(S2, S3) - p(S1, S4)).real, (p(S2, S3) + p(S1, S4)).imag,
         (p(S2, S4) + p(S1, S3)).real, (p(S2, S4) - p(S1, S3)).real, (p(S1, S2) + p(S3, S4)).real,
         (p(S2, S1) + p(S4, S3)).imag, (p(S4, S2) + p(S1, S3)).imag, (p(S4, S2) - p(S1, S3)).imag,
         (p(S1, S2) - p(S3, S4)).imag, (p(S1, S2) - p(S3, S4)).real]
    M = torch.stack(m, 1) / ka ** 2
    w = torch.from_numpy(s["w"]).to(dev)
    M = (w[:, None, None] * M).sum(0)
    if mirror:
        keep = torch.ones(16, 1, dtype=M.dtype, device=dev)
        keep[[2, 3, 6, 7, 8, 9, 12, 13]] = 0
        M = M * keep
    return M.reshape(4, 4, -1)


def exact(case, seed):
    s = _inputs(case, seed)
    dev = _dev()
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    if case["kind"] == "dense":
        return torch.linalg.solve(t(s["Z"]), t(s["B"])).cpu().numpy()
    N = _num_rwg(case)
    # without a GPU the larger ones take longer than a check may
    if (N > 500 and dev.type == "cpu") or (case["kind"] == "gradient" and N > 500):
        return None
    b = _Basis(s["verts"], s["tris"], case["quad"])
    if case["kind"] == "farfield":
        F = _far(b, t(s["cJ"]).T, t(s["cM"]).T, t(s["rhat"]), torch.tensor(s["k"], dtype=torch.complex128, device=dev))
        return F.cpu().numpy()
    p = [torch.tensor(v, dtype=torch.float64, device=dev, requires_grad=case["kind"] == "gradient")
         for v in (s["m"].real, s["m"].imag, s["ka"])]
    Z = _system(b, p[2], p[0], p[1])
    if case["kind"] == "assemble":
        return Z.cpu().numpy()
    kh, e0 = bem_amd.planewave_orient_rhs(s["RT"])
    B = _plane_waves(b, p[2], t(kh), t(e0))
    X = torch.linalg.solve(Z, B)
    if case["kind"] == "precond":
        return X.cpu().numpy()
    M = _mueller(b, X, s, case["mirror"], p[2])
    if case["kind"] != "gradient":
        return M.cpu().numpy()
    L = (t(s["weight"]) * torch.log(M[0, 0])).sum()
    grad = torch.autograd.grad(L, p)
    return {"M": M.detach().cpu().numpy(), "grad": np.array([float(g) for g in grad])}
