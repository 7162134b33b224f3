"""The work that a program using this framework has it do, as timed cases.

A 2.5-D full-waveform inversion calls, per frequency batch and model update:
the batched operator product S(omega, ky) x (matrix-free solvers and
Gauss-Newton products), the assembled operator handed to a direct solver, the
adjoint-state gradient, the Jacobian rows J = G^T F of the Gauss-Newton path
with their contraction J^H J p, and new models during a line search.  Meshes,
frequencies and wavenumbers follow the repository's own configurations
(fem25_amd.configs, bench.py, the tests).

The mesh handle (numbering, pattern, device copies) belongs to the program,
not to one call: it is built once per mesh and shared by the states of a case.
The numbering is the caller's own, handed over as the Fortran drop-ins do.
"""
from __future__ import annotations

import ctypes as C
import functools
import math

import numpy as np
import torch

from fem25_amd import _lib
from fem25_amd import configs as cf
from fem25_amd.api import Graph, MeshInfo

FMIN, FMAX, VS_MIN = 0.02, 0.1, 6300.0 / math.sqrt(3.0)
PML_PAR = dict(rcoeff=1e-3, kappa=1.0, fcent=0.05)
QP, QS, FREQ0 = 300.0, 150.0, 1.0


# --------------------------------------------------------------------------
# Cases
def listed():
    return [
        # the smallest call: one (omega, ky) pair of the 40 x 20 element mesh, as inside a Krylov solver
        dict(name="product_one_pair", kind="product", nx=40, nz=20, p=4, nfreq=1, nky=1, dtype="f64", pml=0),
        # the 200 x 100 order-4 configuration, 128 pairs
        dict(name="product_p4", kind="product", nx=200, nz=100, p=4, nfreq=8, nky=16, dtype="f64", pml=0),
        # the order-6 Gauss-Newton batch of 192 pairs, on a mesh whose state fits the card three times
        dict(name="product_p6", kind="product", nx=160, nz=80, p=6, nfreq=6, nky=32, dtype="f64", pml=0),
        # a ragged mesh and batch in single precision
        dict(name="product_f32_p5", kind="product", nx=97, nz=61, p=5, nfreq=5, nky=15, dtype="f32", pml=0),
        # two absorbing rings and a Bielak ring, 240 pairs: the meshes forward modelling really uses
        dict(name="product_pml_p4", kind="product", nx=200, nz=100, p=4, nfreq=10, nky=24, dtype="f64", pml=2),
        # ASMBLE_DRIVER's COMPLEX*8 operator of one (omega, ky) on the absorbing mesh, and its product
        dict(name="assemble_pml_p4", kind="assemble", nx=200, nz=100, p=4, dtype="c64", pml=2, disp=False),
        # the same in a dispersive medium (every element depends on the frequency), double precision
        dict(name="assemble_disp_p4", kind="assemble", nx=64, nz=33, p=4, dtype="c128", pml=2, disp=True),
        # the adjoint gradient over the 128 wavefield pairs of the order-4 configuration
        dict(name="gradient_p4", kind="gradient", nx=200, nz=100, p=4, nfreq=8, nky=16, dtype="f64"),
        # the order-6 gradient on a ragged mesh and batch
        dict(name="gradient_p6", kind="gradient", nx=121, nz=59, p=6, nfreq=3, nky=15, dtype="f64"),
        # Jacobian rows of 60 receivers x 3 components
        dict(name="jacobian_p4", kind="jacobian", nx=200, nz=100, p=4, nrhs=180),
        # J^H J p over 10 frequencies x 12 sources of 20..120 receivers
        dict(name="gauss_newton_p4", kind="gauss_newton", nx=200, nz=100, p=4, njac=120),
        # two trial models of a line search, each applied to a frequency's 16 pairs
        dict(name="line_search_p4", kind="line_search", nx=120, nz=61, p=4, nfreq=1, nky=16),
    ]


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(["product", "product", "product", "assemble", "gradient", "gradient", "jacobian",
                           "gauss_newton", "line_search"])
        p = rng.choice([2, 3, 4, 4, 5, 6, 6])
        nx = int(round(math.exp(rng.uniform(math.log(12), math.log(200)))))
        nz = max(9, int(round(nx * rng.uniform(0.4, 0.8))))
        c = dict(kind=kind, nx=nx, nz=nz, p=p)
        if kind in ("product", "gradient"):
            c.update(nfreq=rng.randint(1, 10), nky=int(round(math.exp(rng.uniform(0.0, math.log(32))))),
                     dtype=rng.choice(["f64", "f64", "f32"]))
            if kind == "product":
                c.update(pml=rng.choice([0, 0, 2]))
        elif kind == "assemble":
            c.update(dtype=rng.choice(["c64", "c128"]), pml=rng.choice([0, 2]), disp=rng.random() < 0.3)
        elif kind == "jacobian":
            c.update(nrhs=3 * int(round(math.exp(rng.uniform(math.log(4), math.log(80))))))
        elif kind == "gauss_newton":
            c.update(njac=rng.randint(2, 120))
        else:
            c.update(nfreq=1, nky=rng.randint(1, 24))
        # no dearer than the dearest listed case; dispersive meshes and CSR patterns of listed sizes
        if _cost(c) > most or _nee(c) ** 2 * nx * nz > 2.0e8 or (c.get("disp") and nx * nz > 64 * 33):
            continue
        if kind == "gauss_newton" and (nx + 1) * (nz + 1) * c["njac"] > 201 * 101 * 120:
            continue
        return c


def _nee(c):
    return 3 * (c["p"] + 1) ** 2


def _ndof(c):
    return 3 * (c["nx"] * c["p"] + 1) * (c["nz"] * c["p"] + 1)


def _cost(c):
    w = work(c)
    return max(w["bytes"] / 4e12, w["flops"] / 4e13)


def work(case):
    """Each input read and each output written once; multiplications by sum
    factorisation with order + 2 points per direction."""
    n1, ne, ndof = case["p"] + 1, case["nx"] * case["nz"], _ndof(case)
    q = n1 + 1
    field = 12.0 * (2 * n1 * n1 * q + 3 * n1 * q * q)      # one element field to the points, or back
    kind = case["kind"]
    if kind in ("product", "line_search"):
        nb = case["nfreq"] * case["nky"] * (2 if kind == "line_search" else 1)
        size = 8 if case.get("dtype") == "f32" else 16
        return {"bytes": 2.0 * size * ndof * nb, "flops": (2 * field + 200.0 * q * q) * ne * nb}
    if kind == "assemble":
        size = 8 if case["dtype"] == "c64" else 16
        nz = float(_nee(case)) ** 2 * ne * 0.92
        return {"bytes": nz * (2 * size + 4) + 3.0 * size * ndof, "flops": 8.0 * nz}
    if kind == "gradient":
        nb = case["nfreq"] * case["nky"]
        size = 8 if case["dtype"] == "f32" else 16
        return {"bytes": 2.0 * size * ndof * nb, "flops": (2 * field + 100.0 * q * q) * ne * nb}
    if kind == "jacobian":
        cols = (case["nx"] + 1) * (case["nz"] + 1)
        return {"bytes": 8.0 * ndof * case["nrhs"] + 8.0 * cols * case["nrhs"] + 12.0 * cols * _nee(case),
                "flops": 8.0 * cols * _nee(case) * case["nrhs"]}
    jac = float(_nobs(case).sum()) * (case["nx"] + 1) * (case["nz"] + 1)
    return {"bytes": 8.0 * jac, "flops": 8.0 * jac}


# --------------------------------------------------------------------------
# What the program holds before the call
@functools.lru_cache(maxsize=2)
def _numbering(nx, nz, p, npml):
    """LM (element, node, component), 1-based in order of first touch, zero on
    the fixed outer sides of the absorbing rings; number of DOFs."""
    nl = p + 1
    e = np.arange(nx * nz)
    jz, jx = np.divmod(np.arange(nl * nl), nl)
    ix = (e % nx * p)[:, None] + jx
    iz = (e // nx * p)[:, None] + jz
    node = (iz * (nx * p + 1) + ix).ravel()
    free = np.ones((nx * p + 1) * (nz * p + 1), bool)
    if npml:
        side = free.reshape(nz * p + 1, nx * p + 1)
        side[:, 0] = side[:, -1] = side[0, :] = False
    seen, at = np.unique(node, return_index=True)
    seen = seen[np.argsort(at, kind="stable")]
    seen = seen[free[seen]]
    number = np.zeros(free.size, np.int64)
    number[seen] = np.arange(seen.size) + 1
    k = number[node].reshape(nx * nz, nl * nl, 1)
    lm = np.where(k > 0, 3 * (k - 1) + 1 + np.arange(3), 0).astype(np.int32)
    return lm, 3 * seen.size


def _keys(lm, ndof):
    """row * ndof + column of every element coupling, sorted and unique."""
    d = torch.from_numpy(lm.reshape(lm.shape[0], -1)).cuda().long() - 1
    parts, step = [], max(1, 40_000_000 // d.shape[1] ** 2)
    for s in range(0, d.shape[0], step):
        r, c = d[s:s + step, :, None], d[s:s + step, None, :]
        parts.append(torch.unique((r * ndof + c)[(r >= 0) & (c >= 0)]))
    return torch.unique(torch.cat(parts))


def _pml(case):
    return cf.PML(**PML_PAR) if case.get("pml") else cf.PML()


def _mesh(case):
    return cf.structured_mesh(case["nx"], case["nz"], case["p"], npml=case.get("pml", 0),
                              nbielak=1 if case.get("pml") else 0)


def _model(mesh, case, seed=2):
    model = cf.layered_model(mesh, seed=seed)
    return cf.with_attenuation(model, QP, QS, FREQ0) if case.get("disp") else model


@functools.lru_cache(maxsize=1)
def _handle(kind, nx, nz, p, npml, disp):
    case = dict(nx=nx, nz=nz, p=p, pml=npml, disp=disp)
    mesh = _mesh(case)
    lm, ndof = _numbering(nx, nz, p, npml)
    keys = _keys(lm, ndof)
    irptr = torch.searchsorted(keys, torch.arange(ndof + 1, device="cuda") * ndof).int().cpu().numpy() + 1
    jcptr = (keys % ndof).int().cpu().numpy() + 1
    del keys
    torch.cuda.empty_cache()
    mi = MeshInfo(mesh, _pml(case), graph=Graph(0, ndof, jcptr.size, None, lm, irptr, jcptr, b""))
    mi.set_model(_model(mesh, case))
    return mi


def _get(case):
    return _handle(case["kind"], case["nx"], case["nz"], case["p"], case.get("pml", 0), case.get("disp", False))


def _batch(case):
    om, ky, f, py = cf.freq_ky_batch(case["nfreq"], case["nky"], FMIN, FMAX, VS_MIN)
    return om, ky


def _gen(seed, salt):
    return torch.Generator(device="cuda").manual_seed(1000 * int(seed) + salt)


def _vec(shape, seed, salt, dtype=torch.complex128):
    return torch.randn(*shape, dtype=dtype, device="cuda", generator=_gen(seed, salt))


def _nobs(case):
    return 3 * np.random.default_rng(8).integers(20, 121, size=case["njac"])


def _one_pair(seed):
    """A frequency and slowness of the batch's range."""
    r = np.random.default_rng(seed)
    f = float(r.uniform(FMIN, FMAX))
    return f, float(r.uniform(0.0, 0.5) / VS_MIN)


def _trial_models(case, seed):
    mesh = _mesh(case)
    return [_model(mesh, case, seed=1000 + 2 * int(seed) + k) for k in range(2)]


def _virtual_forces(case, seed):
    """F in CSC order: a column per anchor over the DOFs of its elements, the
    rows of its last element filled (CFMAT_DIST's columns); offsets, rows."""
    lm, ndof = _numbering(case["nx"], case["nz"], case["p"], 0)
    nx, nz = case["nx"], case["nz"]
    e = np.arange(nx * nz)
    a1 = e // nx * (nx + 1) + e % nx
    corners = np.stack([a1, a1 + 1, a1 + nx + 2, a1 + nx + 1], 1)
    d = torch.from_numpy(lm.reshape(nx * nz, -1)).cuda().long() - 1
    an = torch.from_numpy(corners).cuda()
    keys = torch.unique((an[:, :, None] * ndof + d[:, None, :]).reshape(-1))
    ncol = (nx + 1) * (nz + 1)
    off = torch.searchsorted(keys, torch.arange(ncol + 1, device="cuda") * ndof)
    last = torch.zeros(ncol, dtype=torch.long, device="cuda")
    for k in range(4):
        last[an[:, k]] = torch.maximum(last[an[:, k]], torch.from_numpy(e).cuda())
    mine = torch.searchsorted(keys, (torch.arange(ncol, device="cuda")[:, None] * ndof + d[last]).reshape(-1))
    val = torch.zeros(keys.numel(), dtype=torch.complex64, device="cuda")
    val[mine] = _vec((mine.numel(),), seed, 3, torch.complex64)
    return val, keys // ndof, keys % ndof, off


def prepare(case, seed):
    kind, mi = case["kind"], _get(case)
    s = dict(kind=kind, mi=mi)
    if kind == "product":
        dt = torch.complex64 if case["dtype"] == "f32" else torch.complex128
        om, ky = _batch(case)
        s.update(om=om, ky=ky, x=_vec((mi.ndof, om.size), seed, 1, dt),
                 mode=_lib.F25_APPLY_F32 if case["dtype"] == "f32" else _lib.F25_APPLY_F64)
        s["y"] = torch.empty_like(s["x"])
    elif kind == "line_search":
        om, ky = _batch(case)
        s.update(om=om, ky=ky, x=_vec((mi.ndof, om.size), seed, 1), models=_trial_models(case, seed))
        s["y"] = [torch.empty_like(s["x"]) for _ in range(2)]
    elif kind == "assemble":
        dt = torch.complex64 if case["dtype"] == "c64" else torch.complex128
        s.update(pair=_one_pair(seed), x=_vec((mi.ndof,), seed, 1, dt),
                 s=torch.empty(mi.nz, dtype=dt, device="cuda"))
        s["y"] = torch.empty_like(s["x"])
    elif kind == "gradient":
        dt = torch.complex64 if case["dtype"] == "f32" else torch.complex128
        om, ky = _batch(case)
        s.update(om=om, ky=ky, u=_vec((om.size, mi.ndof), seed, 1, dt), lam=_vec((om.size, mi.ndof), seed, 2, dt),
                 g=torch.zeros(mi.mesh.nnpg, 3, dtype=torch.float64, device="cuda"),
                 call=mi.gradient32_dev if case["dtype"] == "f32" else mi.gradient_dev)
    else:
        inv = mi.inv or mi.inv_setup(b"PP")
        if kind == "jacobian":
            n = case["nrhs"]
            s.update(nrhs=n, gt=_vec((mi.ndof, n), seed, 1, torch.complex64), f=_virtual_forces(case, seed)[0],
                     jac=torch.empty(inv.nnpgl, n, dtype=torch.complex64, device="cuda"),
                     hd=torch.zeros(inv.na35, dtype=torch.float32, device="cuda"))
        else:
            nobs = _nobs(case).astype(np.int32)
            s.update(nobs=nobs, alpha=np.ones(nobs.size),
                     jac=_vec((int(nobs.sum()) * inv.nnpgl,), seed, 1, torch.complex64),
                     p=_vec((inv.na35,), seed, 2, torch.float64),
                     z=torch.zeros(inv.na35, dtype=torch.float64, device="cuda"))
    return s


def _dev(t):
    return C.c_void_p(t.data_ptr())


def run(s):
    kind, mi = s["kind"], s["mi"]
    if kind == "product":
        mi.apply_batch_dev(s["om"], s["ky"], s["x"], s["y"], s["mode"])
        return s["y"]
    if kind == "line_search":
        for model, y in zip(s["models"], s["y"]):
            mi.set_model(model)
            mi.apply_batch_dev(s["om"], s["ky"], s["x"], y)
        return s["y"]
    if kind == "assemble":
        mi.asmble_dev(b"B", *s["pair"], s["s"])
        mi.csr_apply_dev(s["s"], s["x"], s["y"])
        return s["s"], s["y"]
    if kind == "gradient":
        s["g"].zero_()
        s["call"](s["om"], s["ky"], s["u"], s["lam"], s["g"])
        return s["g"]
    # the C entry points take device arrays produced on PyTorch's stream
    if kind == "jacobian":
        s["hd"].zero_()
        torch.cuda.current_stream().synchronize()
        _lib.check(_lib.load().f25_pchadj_jac_dev(mi.h, s["nrhs"], _dev(s["gt"]), _dev(s["f"]), _dev(s["jac"]),
                                                  _dev(s["hd"])), "f25_pchadj_jac_dev")
        return s["jac"], s["hd"]
    s["z"].zero_()
    torch.cuda.current_stream().synchronize()
    _lib.check(_lib.load().f25_gnmfree_dev(mi.h, s["nobs"].size, s["nobs"].ctypes.data_as(_lib.ip),
                                           s["alpha"].ctypes.data_as(_lib.dp), _dev(s["jac"]), _dev(s["p"]),
                                           _dev(s["z"])), "f25_gnmfree_dev")
    return s["z"]


# --------------------------------------------------------------------------
# The same in plain torch, 64 bits: fields at the quadrature points, fluxes,
# and their projection on the test functions
def _gll(n):
    """Gauss-Lobatto-Legendre nodes and weights."""
    c = np.zeros(n)
    c[-1] = 1.0
    d1 = np.polynomial.legendre.legder(c)
    x = np.sort(np.real(np.polynomial.legendre.legroots(d1)))
    for _ in range(3):
        x -= np.polynomial.legendre.legval(x, d1) / np.polynomial.legendre.legval(x, np.polynomial.legendre.legder(d1))
    x = np.concatenate([[-1.0], x, [1.0]])
    return x, 2.0 / (n * (n - 1) * np.polynomial.legendre.legval(x, c) ** 2)


def _cardinal(nodes, pts):
    """Values and derivatives [point, node] of the Lagrange polynomials."""
    n = nodes.size
    v, d = np.ones((pts.size, n)), np.zeros((pts.size, n))
    for j in range(n):
        others = [k for k in range(n) if k != j]
        for k in others:
            v[:, j] *= (pts - nodes[k]) / (nodes[j] - nodes[k])
        for m in others:
            t = np.full(pts.size, 1.0 / (nodes[j] - nodes[m]))
            for k in others:
                if k != m:
                    t *= (pts - nodes[k]) / (nodes[j] - nodes[k])
            d[:, j] += t
    return v, d


class _Plain:
    """A structured mesh's elements at the reference's 2 p + 5 points per direction."""

    def __init__(self, case):
        self.case, self.mesh = case, _mesh(case)
        p, n1, nq = case["p"], case["p"] + 1, 2 * case["p"] + 5
        xq, wq = _gll(nq)
        v, d = _cardinal(_gll(n1)[0], xq)
        hx, hz = 80e3 / case["nx"], 40e3 / case["nz"]
        dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()   # noqa: E731
        outer = lambda a, b: dev(np.einsum("ye,xi->yxei", a, b).reshape(nq * nq, n1 * n1))   # noqa: E731
        self.n, self.nx, self.nz = outer(v, v), outer(v, d) * (2 / hx), outer(d, v) * (2 / hz)
        self.w = dev(np.outer(wq, wq).ravel()) * (hx * hz / 4)
        lo, hi = (1 - xq) / 2, (1 + xq) / 2
        self.hat = dev(np.stack([np.outer(z, x).ravel() for z, x in ((lo, lo), (lo, hi), (hi, hi), (hi, lo))]))
        self.corner = dev(self.mesh.ieng.astype(np.int64) - 1)
        lm, self.ndof = _numbering(case["nx"], case["nz"], p, case.get("pml", 0))
        self.dof = dev(lm.astype(np.int64)).reshape(lm.shape[0], -1) - 1
        self.absorbing = dev(np.frombuffer(self.mesh.cdomain, np.uint8) == ord("A"))

    def at_points(self, anchors, el):
        return torch.from_numpy(np.ascontiguousarray(anchors)).cuda()[self.corner[el]] @ self.hat

    def coefficients(self, model, el, omega):
        """w lambda, w mu, w rho and the stretch factors 1/e_x, 1/e_z (None without)."""
        rho, lam, mu = model.dens, model.ecoeff[:, 0], model.ecoeff[:, 1]
        vp, vs = np.sqrt((lam + 2 * mu) / rho), np.sqrt(mu / rho)
        if model.qp is not None:
            lg = math.log(omega / (2 * math.pi) / model.freq0)
            zp, zs = ((v * (1 + lg / (math.pi * q)) - 0.5j * v / q) for v, q in (
                (self.at_points(v, el), self.at_points(q, el)) for v, q in ((vp, model.qp), (vs, model.qs))))
            L, M, R = zp ** 2 - 2 * zs ** 2, zs ** 2, torch.ones_like(zp.real)
        else:
            L, M, R = (self.at_points(a, el) for a in (lam, mu, rho))
        ex = ez = None
        if self.case.get("pml"):
            par, vel = _pml(self.case), self.at_points(vp, el)

            def stretch(depth, width):
                r = self.at_points(depth, el) / width
                damp = -3.0 * vel * math.log(par.rcoeff) / (2.0 * width) * r * r
                e = 1.0 / (par.kappa + damp.abs() / torch.complex(math.pi * par.fcent * (1 - r), torch.full_like(r, omega)))
                return torch.where(self.absorbing[el][:, None] & (r > 1e-14), e, torch.ones_like(e))

            ex, ez = stretch(self.mesh.xd, self.mesh.xwidth), stretch(self.mesh.zd, self.mesh.zwidth)
        return self.w * L, self.w * M, self.w * R, ex, ez

    @staticmethod
    def _real(mat, x):
        """mat @ x over the nodes or points (axis 1) of a complex [element, node, ...] tensor."""
        s = torch.view_as_real(x.contiguous())
        y = torch.matmul(mat, s.reshape(s.shape[0], s.shape[1], -1))
        return torch.view_as_complex(y.reshape(s.shape[0], mat.shape[0], *s.shape[2:]).contiguous())

    def apply(self, xe, coef, om, ky):
        """Element products: xe [element, node, 3, pair], om and ky per pair."""
        L, M, R, ex, ez = (None if c is None else c[:, :, None] for c in coef)
        U, X, Z = self._real(self.n, xe), self._real(self.nx, xe), self._real(self.nz, xe)
        if ex is not None:
            X, Z = ex[..., None] * X, ez[..., None] * Z
        U, X, Z = (a.unbind(2) for a in (U, X, Z))
        ik, k2, w2, P = 1j * ky, ky * ky, om * om, L + 2 * M
        FN = [ik * M * X[1] + (k2 * M - w2 * R) * U[0],
              ik * L * (X[0] + Z[2]) + (k2 * P - w2 * R) * U[1],
              ik * M * Z[1] + (k2 * M - w2 * R) * U[2]]
        FX = [P * X[0] + L * Z[2] - ik * L * U[1], M * X[1] - ik * M * U[0], M * (Z[0] + X[2])]
        FZ = [M * (Z[0] + X[2]), M * Z[1] - ik * M * U[2], L * X[0] + P * Z[2] - ik * L * U[1]]
        FN, FX, FZ = (torch.stack(f, 2) for f in (FN, FX, FZ))
        if ex is not None:
            FX, FZ = ex[..., None] * FX, ez[..., None] * FZ
        return self._real(self.n.T, FN) + self._real(self.nx.T, FX) + self._real(self.nz.T, FZ)

    def chunks(self, pairs):
        step = max(1, int(4e7 / (self.n.shape[0] * pairs)))
        for s in range(0, self.dof.shape[0], step):
            yield torch.arange(s, min(s + step, self.dof.shape[0]), device="cuda")

    def product(self, model, om, ky, x):
        """S(om_b, ky_b) x_b for x [dof, pair]."""
        y = torch.zeros(self.ndof, x.shape[1], dtype=torch.complex128, device="cuda")
        groups = [np.nonzero(om == w)[0] for w in np.unique(om)] if self.case.get("pml") else [np.arange(om.size)]
        for idx in groups:
            i = torch.from_numpy(idx).cuda()
            xi = torch.cat([x[:, i].to(torch.complex128), torch.zeros(1, idx.size, dtype=torch.complex128, device="cuda")])
            yi = torch.zeros_like(xi)
            o, k = (torch.from_numpy(a[idx]).cuda() for a in (om, ky))
            for el in self.chunks(idx.size):
                d = self.dof[el]
                xe = xi[d].reshape(el.numel(), -1, 3, idx.size)
                ye = self.apply(xe, self.coefficients(model, el, float(om[idx[0]])), o, k)
                yi.index_add_(0, torch.where(d < 0, self.ndof, d).reshape(-1), ye.reshape(-1, idx.size))
            y[:, i] = yi[:-1]
        return y

    def assembled(self, model, om, ky, x):
        """The operator's values in CSR order, and its product with x."""
        lm, _ = _numbering(self.case["nx"], self.case["nz"], self.case["p"], self.case.get("pml", 0))
        keys = _keys(lm, self.ndof)
        val = torch.zeros(keys.numel(), dtype=torch.complex128, device="cuda")
        nee = self.dof.shape[1]
        eye = torch.eye(nee, dtype=torch.complex128, device="cuda").reshape(1, nee // 3, 3, nee)
        o, k = (torch.full((nee,), v, dtype=torch.float64, device="cuda") for v in (om, ky))
        for el in self.chunks(nee):
            m = self.apply(eye.expand(el.numel(), -1, -1, -1), self.coefficients(model, el, om), o, k)
            d = self.dof[el]
            r, c = d[:, :, None].expand(-1, -1, nee), d[:, None, :].expand(-1, nee, -1)
            ok = (r >= 0) & (c >= 0)
            val.index_add_(0, torch.searchsorted(keys, (r * self.ndof + c)[ok]), m.reshape(el.numel(), nee, nee)[ok])
        y = torch.zeros(self.ndof, dtype=torch.complex128, device="cuda")
        y.index_add_(0, keys // self.ndof, val * x.to(torch.complex128)[keys % self.ndof])
        return val, y

    def gradient(self, model, om, ky, u, lam):
        """sum_t Re(lam_t^H dS_t/dm u_t) for (Vp, Vs, rho) at the anchors."""
        o, k = torch.from_numpy(om).cuda(), torch.from_numpy(ky).cuda()
        g = torch.zeros(self.mesh.nnpg, 3, dtype=torch.float64, device="cuda")

        def fields(a, el):
            xe = a[:, self.dof[el]].permute(1, 2, 0).to(torch.complex128).reshape(el.numel(), -1, 3, om.size)
            U, X, Z = self._real(self.n, xe), self._real(self.nx, xe), self._real(self.nz, xe)
            return U, [X, -1j * k * U, Z]      # G[j][:, :, i] = d_j u_i

        dot = lambda a, b: (a.real * b.real + a.imag * b.imag).sum(-1)   # noqa: E731
        for el in self.chunks(2 * om.size):
            U, G = fields(u, el)
            V, H = fields(lam, el)
            div = [sum(f[i][:, :, i] for i in range(3)) for f in (G, H)]
            dl = dot(div[1], div[0])
            dm = sum(dot(H[j][:, :, i], G[j][:, :, i] + G[i][:, :, j]) for i in range(3) for j in range(3))
            dr = -((o * o) * (V.real * U.real + V.imag * U.imag).sum(2)).sum(-1)
            for c in range(4):
                part = torch.stack([((self.w * self.hat[c]) * t).sum(1) for t in (dl, dm, dr)], 1)
                g.index_add_(0, self.corner[el][:, c], part)
        rho, la, mu = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (
            model.dens, model.ecoeff[:, 0], model.ecoeff[:, 1]))
        vp, vs = torch.sqrt((la + 2 * mu) / rho), torch.sqrt(mu / rho)
        return torch.stack([g[:, 0] * 2 * rho * vp, -4 * rho * vs * g[:, 0] + 2 * rho * vs * g[:, 1],
                            g[:, 0] * (vp ** 2 - 2 * vs ** 2) + g[:, 1] * vs ** 2 + g[:, 2]], 1)


def exact(case, seed):
    kind, n = case["kind"], _ndof(case)
    if kind in ("product", "line_search", "assemble", "gradient"):
        pl = _Plain(case)
        n = pl.ndof
        if kind == "assemble":
            f, py = _one_pair(seed)
            x = _vec((n,), seed, 1, torch.complex64 if case["dtype"] == "c64" else torch.complex128)
            return pl.assembled(_model(pl.mesh, case), 2 * math.pi * f, 2 * math.pi * f * py, x)
        om, ky = _batch(case)
        dt = torch.complex64 if case.get("dtype") == "f32" else torch.complex128
        if kind == "gradient":
            u, lam = (_vec((om.size, n), seed, salt, dt) for salt in (1, 2))
            return pl.gradient(_model(pl.mesh, case), om, ky, u, lam)
        x = _vec((n, om.size), seed, 1, dt)
        if kind == "product":
            return pl.product(_model(pl.mesh, case), om, ky, x)
        return [pl.product(m, om, ky, x) for m in _trial_models(case, seed)]
    ncol = (case["nx"] + 1) * (case["nz"] + 1)
    if kind == "jacobian":
        gt = _vec((n, case["nrhs"]), seed, 1, torch.complex64)
        val, col, row, _ = _virtual_forces(case, seed)
        jac = torch.zeros(ncol, case["nrhs"], dtype=torch.complex128, device="cuda")
        keep = torch.nonzero(val != 0)[:, 0]
        for at in torch.split(keep, max(1, 200_000_000 // case["nrhs"] // 16)):
            jac.index_add_(0, col[at], val[at].to(torch.complex128)[:, None] * gt[row[at]].to(torch.complex128))
        return jac, (jac.real ** 2 + jac.imag ** 2).sum(1)
    nobs = _nobs(case)
    jac = _vec((int(nobs.sum()) * ncol,), seed, 1, torch.complex64)
    p = _vec((ncol,), seed, 2, torch.float64)
    z, at = torch.zeros(ncol, dtype=torch.float64, device="cuda"), 0
    for m in nobs.tolist():
        J = jac[at:at + m * ncol].reshape(ncol, m)
        at += m * ncol
        for part in (J.real.double(), J.imag.double()):
            z += part @ (p @ part)
    return z
