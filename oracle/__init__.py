"""Python access to the parity checkers (TEST INFRASTRUCTURE ONLY).

`liboracle.so` is the C restatement in oracle.c; `_ref/libfem25ref.so` is the
reference's own Fortran compiled in place by oracle/Makefile.  Only tests/,
__graft_entry__.smoke() and bench.py's CPU-baseline leg import this package.
"""
from __future__ import annotations

import ctypes as C
import dataclasses
import json
import os
import subprocess
import sys
import tempfile

import numpy as np

_HERE = os.path.dirname(os.path.abspath(__file__))
_ORC = None
_REF = None

dp = C.POINTER(C.c_double)
ip = C.POINTER(C.c_int)
fp = C.POINTER(C.c_float)


def _p(a, t):
    return a.ctypes.data_as(t)


def build(ref: bool = True) -> None:
    subprocess.run(["make", "-s", "liboracle.so"], cwd=_HERE, check=True)
    src = os.environ.get("FEM25_REFERENCE", "/root/reference")
    if ref and os.path.exists(os.path.join(src, "fwd_struc.h")):   # the sources, not an empty folder
        subprocess.run(["make", "-s", "-j8", "ref", "REF=" + src], cwd=_HERE, check=True)


def lib():
    global _ORC
    if _ORC is None:
        path = os.path.join(_HERE, "liboracle.so")
        if not os.path.exists(path):
            build(ref=False)
        _ORC = C.CDLL(path)
    return _ORC


def ref_available() -> bool:
    return os.path.exists(os.path.join(_HERE, "_ref", "libfem25ref.so"))


def ref():
    global _REF
    if _REF is None:
        _REF = C.CDLL(os.path.join(_HERE, "_ref", "libfem25ref.so"))
    return _REF


def _child_call(name, scalars, arrays):
    """Runs oracle.<name>(**scalars, **arrays, reference=True) in a fresh
    interpreter that has not loaded torch; returns its outputs (npz)."""
    with tempfile.TemporaryDirectory(prefix="orcref") as d:
        np.savez(os.path.join(d, "in.npz"), **arrays)
        with open(os.path.join(d, "in.json"), "w") as f:
            json.dump({"name": name, "scalars": scalars}, f)
        env = dict(os.environ, PYTHONPATH=os.pathsep.join([os.path.dirname(_HERE), os.environ.get("PYTHONPATH", "")]))
        subprocess.run([sys.executable, "-m", "oracle._child", d], check=True, env=env, cwd=os.path.dirname(_HERE))
        with np.load(os.path.join(d, "out.npz"), allow_pickle=False) as z:
            return {k: z[k] for k in z.files}


class _Asm(C.Structure):
    _fields_ = [("nord", C.c_int), ("nelem", C.c_int), ("nnpg", C.c_int), ("ndof", C.c_int),
                ("ieng", ip), ("lm", ip), ("irptr", ip), ("jcptr", ip),
                ("xlocs", dp), ("zlocs", dp), ("dens", dp), ("ecoeff", dp), ("xd", dp),
                ("zd", dp), ("cdomain", C.c_char_p), ("xwidth", C.c_double),
                ("zwidth", C.c_double), ("rcoeff", C.c_double), ("dmax", C.c_double),
                ("kappa", C.c_double), ("fcent", C.c_double), ("ldisp", C.c_int), ("qp", dp),
                ("qs", dp), ("freq0", C.c_double)]


class _Mesh(C.Structure):
    _fields_ = [("nord", C.c_int), ("nelem", C.c_int), ("nnpg", C.c_int), ("ieng", ip),
                ("xlocs", dp), ("zlocs", dp), ("cdomain", C.c_char_p), ("cnnpg", C.c_char_p)]


class _Inv(C.Structure):
    _fields_ = [("nnpinv", C.c_int), ("na35", C.c_int), ("nvinv", C.c_int), ("ncon", C.c_int),
                ("nnpgl", C.c_int), ("nz_fdist", C.c_int), ("mbufrhs", C.c_int),
                ("mconn", ip), ("maskg", ip), ("mygrad", ip), ("jcsc", ip), ("icsc", ip),
                ("elem_wts", dp)]


@dataclasses.dataclass
class Graph:
    nnp: int
    ndof: int
    nz: int
    ien: np.ndarray     # (nelem, nen) 1-based
    lm: np.ndarray      # (nelem, nen, 3) 1-based, 0 fixed
    irptr: np.ndarray   # (ndof+1,) 1-based
    jcptr: np.ndarray   # (nz,) 1-based
    cnp: bytes


@dataclasses.dataclass
class Inv:
    nnpinv: int
    ncon: int
    nnpgl: int
    nz_fdist: int
    mbufrhs: int
    na35: int
    maskg: np.ndarray
    mconn: np.ndarray   # (ncon, nnpg) i.e. Fortran MCONN(NNPG,NCON) memory
    mygrad: np.ndarray
    jcsc: np.ndarray
    icsc: np.ndarray
    elem_wts: np.ndarray


def _mesh_struct(mesh):
    keep = (np.ascontiguousarray(mesh.ieng, np.int32), np.ascontiguousarray(mesh.xlocs),
            np.ascontiguousarray(mesh.zlocs))
    s = _Mesh(mesh.nord, mesh.nelem, mesh.nnpg, _p(keep[0], ip), _p(keep[1], dp),
              _p(keep[2], dp), mesh.cdomain, mesh.cnnpg)
    return s, keep


def graph(mesh) -> Graph:
    """GENIEN, CONNECT, GENID, GENLM, GENCRS_QUICK, CNMESH restated in C."""
    L = lib()
    ms, keep = _mesh_struct(mesh)
    nl = mesh.nord + 1
    nen = nl * nl
    xipts = np.zeros(nl)
    xq = np.zeros(2 * mesh.nord + 5)
    wq = np.zeros_like(xq)
    shl = np.zeros(3 * nen * xq.size * xq.size)
    L.orc_dshl(nl, xq.size, _p(xipts, dp), _p(xq, dp), _p(wq, dp), _p(shl, dp))
    ien = np.zeros((mesh.nelem, nen), np.int32)
    L.orc_genien.restype = C.c_int
    nnp = L.orc_genien(C.byref(ms), _p(xipts, dp), _p(ien, ip))
    if nnp < 0:
        raise RuntimeError("genien failed %d" % nnp)
    ident = np.zeros((nnp, 3), np.int32)
    ndof = L.orc_genid(C.byref(ms), _p(xipts, dp), _p(ien, ip), nnp, _p(ident, ip))
    if ndof < 0:
        raise RuntimeError("genid failed")
    lm = np.zeros((mesh.nelem, nen, 3), np.int32)
    L.orc_genlm(nen, mesh.nelem, _p(ident, ip), _p(ien, ip), _p(lm, ip))
    ncon = L.orc_icmcon(nen, nnp, mesh.nelem, _p(ien, ip))
    mconn = np.zeros((ncon, nnp), np.int32)
    L.orc_connect(nen, nnp, mesh.nelem, ncon, _p(ien, ip), _p(mconn, ip))
    cap = ndof * 3 * ncon * nen
    irptr = np.zeros(ndof + 1, np.int32)
    jc = np.zeros(cap, np.int32)
    L.orc_gencrs.restype = C.c_long
    nz = L.orc_gencrs(nen, nnp, mesh.nelem, ndof, ncon, _p(mconn, ip), _p(ien, ip), _p(lm, ip),
                      _p(irptr, ip), _p(jc, ip), C.c_long(cap))
    if nz < 0:
        raise RuntimeError("gencrs failed")
    cnp = C.create_string_buffer(ndof)
    L.orc_cnmesh(nen, ndof, mesh.nelem, mesh.cdomain, _p(lm, ip), cnp)
    return Graph(nnp, ndof, int(nz), ien, lm, irptr, jc[:nz].copy(), cnp.raw[:ndof])


def ref_graph(mesh) -> Graph:
    """The reference's GENIEN..GENCRS_QUICK and CNMESH, compiled."""
    R = ref()
    sizes = np.zeros(3, np.int32)
    ierr = C.c_int(0)
    ieng = np.ascontiguousarray(mesh.ieng, np.int32)
    R.ref_graph(mesh.nord, mesh.nelem, mesh.nnpg, _p(ieng, ip), _p(mesh.xlocs, dp),
                _p(mesh.zlocs, dp), mesh.cdomain, mesh.cnnpg, _p(sizes, ip), C.byref(ierr))
    if ierr.value:
        raise RuntimeError("reference graph failed %d" % ierr.value)
    nnp, ndof, nz = (int(v) for v in sizes)
    nen = (mesh.nord + 1) ** 2
    ien = np.zeros((mesh.nelem, nen), np.int32)
    lm = np.zeros((mesh.nelem, nen, 3), np.int32)
    irptr = np.zeros(ndof + 1, np.int32)
    jcptr = np.zeros(nz, np.int32)
    cnp = C.create_string_buffer(ndof)
    R.ref_graph_get(_p(ien, ip), _p(lm, ip), _p(irptr, ip), _p(jcptr, ip), cnp)
    return Graph(nnp, ndof, nz, ien, lm, irptr, jcptr, cnp.raw[:ndof])


def _asm_struct(mesh, model, g: Graph, pml):
    keep = dict(ieng=np.ascontiguousarray(mesh.ieng, np.int32),
                lm=np.ascontiguousarray(g.lm, np.int32), irptr=g.irptr, jcptr=g.jcptr,
                xlocs=mesh.xlocs, zlocs=mesh.zlocs, dens=model.dens,
                ecoeff=np.asfortranarray(model.ecoeff), xd=mesh.xd, zd=mesh.zd)
    pa = pml.as_array(mesh)
    disp = getattr(model, "qp", None) is not None
    if disp:
        keep["qp"] = np.ascontiguousarray(model.qp, np.float64)
        keep["qs"] = np.ascontiguousarray(model.qs, np.float64)
    s = _Asm(mesh.nord, mesh.nelem, mesh.nnpg, g.ndof, _p(keep["ieng"], ip), _p(keep["lm"], ip),
             _p(keep["irptr"], ip), _p(keep["jcptr"], ip), _p(keep["xlocs"], dp),
             _p(keep["zlocs"], dp), _p(keep["dens"], dp), _p(keep["ecoeff"], dp),
             _p(keep["xd"], dp), _p(keep["zd"], dp), mesh.cdomain, pa[0], pa[1], pa[2],
             pa[3], pa[4], pa[5], int(disp), _p(keep["qp"], dp) if disp else None,
             _p(keep["qs"], dp) if disp else None, float(model.freq0) if disp else 0.0)
    return s, keep


def asmble_z(mesh, model, g, freq, py, pml) -> np.ndarray:
    """FP64 element sums ME+KE in CSR order (ASM_DISP-style accumulation)."""
    s, keep = _asm_struct(mesh, model, g, pml)
    out = np.zeros(g.nz, np.complex128)
    if lib().orc_asmble_z(C.byref(s), C.c_double(freq), C.c_double(py), _p(out, dp)):
        raise RuntimeError("orc_asmble_z failed")
    return out


def asmble_cdist(mesh, model, g, freq, py, pml) -> np.ndarray:
    """COMPLEX*8 CDIST with per-contribution rounding (asmble.f90:302-305)."""
    s, keep = _asm_struct(mesh, model, g, pml)
    out = np.zeros(g.nz, np.complex64)
    if lib().orc_asmble_cdist(C.byref(s), C.c_double(freq), C.c_double(py), _p(out, fp)):
        raise RuntimeError("orc_asmble_cdist failed")
    return out


def ref_asmble(mesh, model, g, freq, py, pml, cftype=b"B") -> np.ndarray:
    """The reference's ASMBLE_DRIVER (COMPLEX*8 CDIST)."""
    out = np.zeros(g.nz, np.complex64)
    ierr = C.c_int(0)
    ieng = np.ascontiguousarray(mesh.ieng, np.int32)
    lm = np.ascontiguousarray(g.lm, np.int32)
    ec = np.asfortranarray(model.ecoeff)
    pa = pml.as_array(mesh)
    if getattr(model, "qp", None) is not None:
        qp = np.ascontiguousarray(model.qp, np.float64)
        qs = np.ascontiguousarray(model.qs, np.float64)
        ref().ref_asmble_q(mesh.nord, mesh.nelem, mesh.nnpg, g.ndof, g.nz, _p(ieng, ip),
                           _p(mesh.xlocs, dp), _p(mesh.zlocs, dp), _p(model.dens, dp), _p(ec, dp),
                           _p(mesh.xd, dp), _p(mesh.zd, dp), mesh.cdomain, _p(lm, ip),
                           _p(g.irptr, ip), _p(g.jcptr, ip), _p(pa, dp), _p(qp, dp), _p(qs, dp),
                           C.c_double(model.freq0), C.c_char(cftype), C.c_double(freq),
                           C.c_double(py), _p(out, fp), C.byref(ierr))
    else:
        ref().ref_asmble(mesh.nord, mesh.nelem, mesh.nnpg, g.ndof, g.nz, _p(ieng, ip),
                         _p(mesh.xlocs, dp), _p(mesh.zlocs, dp), _p(model.dens, dp), _p(ec, dp),
                         _p(mesh.xd, dp), _p(mesh.zd, dp), mesh.cdomain, _p(lm, ip),
                         _p(g.irptr, ip), _p(g.jcptr, ip), _p(pa, dp), C.c_char(cftype),
                         C.c_double(freq), C.c_double(py), _p(out, fp), C.byref(ierr))
    if ierr.value:
        raise RuntimeError("reference ASMBLE_DRIVER failed")
    return out


def spmv_z(g: Graph, s: np.ndarray, x: np.ndarray) -> np.ndarray:
    y = np.zeros(g.ndof, np.complex128)
    x = np.ascontiguousarray(x, np.complex128)
    lib().orc_spmv_z(g.ndof, _p(g.irptr, ip), _p(g.jcptr, ip), _p(s, dp), _p(x, dp), _p(y, dp))
    return y


def spmv_c(g: Graph, s: np.ndarray, x: np.ndarray) -> np.ndarray:
    y = np.zeros(g.ndof, np.complex64)
    x = np.ascontiguousarray(x, np.complex64)
    lib().orc_spmv_c(g.ndof, _p(g.irptr, ip), _p(g.jcptr, ip), _p(s, fp), _p(x, fp), _p(y, fp))
    return y


def asmb_peff(g: Graph, cdist, ue) -> np.ndarray:
    out = np.zeros(g.ndof, np.complex64)
    ue = np.ascontiguousarray(ue, np.complex64)
    lib().orc_asmb_peff(g.ndof, g.cnp, _p(g.irptr, ip), _p(g.jcptr, ip), _p(cdist, fp),
                        _p(ue, fp), _p(out, fp))
    return out


def ref_asmb_peff(g: Graph, cdist, ue) -> np.ndarray:
    """The reference's ASMB_PEFF (asmble.f90:318-377), one rank."""
    out = np.zeros(g.ndof, np.complex64)
    cdist = np.ascontiguousarray(cdist, np.complex64)
    ue = np.ascontiguousarray(ue, np.complex64)
    irptr = np.ascontiguousarray(g.irptr, np.int32)
    jcptr = np.ascontiguousarray(g.jcptr, np.int32)
    ref().ref_asmb_peff(g.ndof, g.nz, g.cnp, _p(irptr, ip), _p(jcptr, ip), _p(cdist, fp), _p(ue, fp),
                        _p(out, fp))
    return out


def inv_setup(mesh, model, g, pml, nvinv=1, linrec=True, lkbdry=True) -> Inv:
    """GENGMASK + GRADPTRS + ELEM_WTS restated (one rank, no .mask file)."""
    s, keep = _asm_struct(mesh, model, g, pml)
    inv = _Inv()
    L = lib()
    if L.orc_gengmask(C.byref(s), mesh.cnnpg, nvinv, int(linrec), int(lkbdry), 0, None,
                      C.byref(inv)):
        raise RuntimeError("gengmask failed")
    if L.orc_gradptrs(C.byref(s), C.byref(inv)) or L.orc_elem_wts(C.byref(s), C.byref(inv)):
        raise RuntimeError("gradptrs/elem_wts failed")
    n = mesh.nnpg
    out = Inv(inv.nnpinv, inv.ncon, inv.nnpgl, inv.nz_fdist, inv.mbufrhs, inv.na35,
              np.ctypeslib.as_array(inv.maskg, (n,)).copy(),
              np.ctypeslib.as_array(inv.mconn, (inv.ncon * n,)).copy().reshape(inv.ncon, n),
              np.ctypeslib.as_array(inv.mygrad, (inv.nnpgl,)).copy(),
              np.ctypeslib.as_array(inv.jcsc, (inv.nnpgl + 1,)).copy(),
              np.ctypeslib.as_array(inv.icsc, (inv.nz_fdist,)).copy(),
              np.ctypeslib.as_array(inv.elem_wts, (mesh.nelem,)).copy())
    L.orc_inv_free(C.byref(inv))
    return out


def ref_inv_setup(mesh, model, g, cinvtype=b"PP", vpvs=3 ** 0.5) -> Inv:
    """The reference's GENGMASK, ELEM_WTS and GRADPTRS, compiled."""
    R = ref()
    sizes = np.zeros(6, np.int32)
    ierr = C.c_int(0)
    ieng = np.ascontiguousarray(mesh.ieng, np.int32)
    lm = np.ascontiguousarray(g.lm, np.int32)
    ec = np.asfortranarray(model.ecoeff)
    R.ref_inv_setup(mesh.nord, mesh.nelem, mesh.nnpg, g.ndof, g.nz, _p(ieng, ip),
                    _p(mesh.xlocs, dp), _p(mesh.zlocs, dp), _p(model.dens, dp), _p(ec, dp),
                    mesh.cdomain, mesh.cnnpg, _p(lm, ip), cinvtype, C.c_double(vpvs),
                    _p(sizes, ip), C.byref(ierr))
    if ierr.value:
        raise RuntimeError("reference inversion setup failed")
    nnpinv, ncon, nnpgl, nzf, mbuf, na35 = (int(v) for v in sizes)
    n = mesh.nnpg
    maskg = np.zeros(n, np.int32)
    mconn = np.zeros(n * ncon, np.int32)
    mygrad = np.zeros(nnpgl, np.int32)
    jcsc = np.zeros(nnpgl + 1, np.int32)
    icsc = np.zeros(nzf, np.int32)
    ew = np.zeros(mesh.nelem)
    R.ref_inv_get(_p(maskg, ip), _p(mconn, ip), _p(mygrad, ip), _p(jcsc, ip), _p(icsc, ip),
                  _p(ew, dp))
    return Inv(nnpinv, ncon, nnpgl, nzf, mbuf, na35, maskg, mconn.reshape(ncon, n), mygrad,
               jcsc, icsc, ew)


def _inv_struct(inv: Inv):
    keep = dict(mconn=np.ascontiguousarray(inv.mconn.ravel(), np.int32), maskg=inv.maskg,
                mygrad=inv.mygrad, jcsc=inv.jcsc, icsc=inv.icsc, ew=inv.elem_wts)
    s = _Inv(inv.nnpinv, inv.na35, inv.na35 // max(inv.nnpinv, 1), inv.ncon, inv.nnpgl, inv.nz_fdist, inv.mbufrhs,
             _p(keep["mconn"], ip), _p(keep["maskg"], ip), _p(keep["mygrad"], ip),
             _p(keep["jcsc"], ip), _p(keep["icsc"], ip), _p(keep["ew"], dp))
    return s, keep


def cfmat_dist(mesh, model, g, inv: Inv, freq, py, wave, cinvtype=b"PP", vpvs=3 ** 0.5,
               pml=None):
    from fem25_amd.configs import PML
    s, keep = _asm_struct(mesh, model, g, pml or PML())
    si, keep2 = _inv_struct(inv)
    wave = np.ascontiguousarray(wave, np.complex64)
    out = np.zeros(inv.nz_fdist, np.complex64)
    if lib().orc_cfmat_dist(C.byref(s), C.byref(si), cinvtype, C.c_double(vpvs),
                            C.c_double(freq), C.c_double(py), _p(wave, fp), _p(out, fp)):
        raise RuntimeError("orc_cfmat_dist failed")
    return out


def ref_cfmat(freq, py, wave, nz_fdist):
    """Reference CFMAT_DIST on the structures of the last ref_inv_setup call."""
    wave = np.ascontiguousarray(wave, np.complex64)
    out = np.zeros(nz_fdist, np.complex64)
    ierr = C.c_int(0)
    ref().ref_cfmat(C.c_double(freq), C.c_double(py), _p(wave, fp), _p(out, fp), C.byref(ierr))
    if ierr.value:
        raise RuntimeError("reference CFMAT_DIST failed")
    return out


def qp_nu_alpha(mesh, model, g, inv: Inv, freq, py, v, adjlam, wave, cinvtype=b"PP", pml=None):
    """CADJ_NU_ALPHA's element loops: (RHSBNU, RHSALP, P3) before the solves."""
    from fem25_amd.configs import PML
    s, keep = _asm_struct(mesh, model, g, pml or PML())
    si, keep2 = _inv_struct(inv)
    v = np.ascontiguousarray(v, np.float32)
    adjlam = np.ascontiguousarray(adjlam, np.complex64)
    wave = np.ascontiguousarray(wave, np.complex64)
    bnu = np.zeros(g.ndof, np.complex64)
    alp = np.zeros(g.ndof, np.complex64)
    p3 = np.zeros(inv.na35, np.float32)
    if lib().orc_qp_nu_alpha(C.byref(s), C.byref(si), cinvtype, C.c_double(freq), C.c_double(py),
                             _p(v, fp), _p(adjlam, fp), _p(wave, fp), _p(bnu, fp), _p(alp, fp),
                             _p(p3, fp)):
        raise RuntimeError("orc_qp_nu_alpha failed")
    return bnu, alp, p3


def met225(mesh, model, g, inv: Inv, freq, py, adjlam, nu, alpha, wave, cinvtype=b"PP", pml=None):
    """MET225_MOD's element loops: (P1, P2) before the reductions."""
    from fem25_amd.configs import PML
    s, keep = _asm_struct(mesh, model, g, pml or PML())
    si, keep2 = _inv_struct(inv)
    vecs = [np.ascontiguousarray(x, np.complex64) for x in (adjlam, nu, alpha, wave)]
    p1 = np.zeros(inv.na35, np.float32)
    p2 = np.zeros(inv.na35, np.float32)
    if lib().orc_met225(C.byref(s), C.byref(si), cinvtype, C.c_double(freq), C.c_double(py),
                        *[_p(x, fp) for x in vecs], _p(p1, fp), _p(p2, fp)):
        raise RuntimeError("orc_met225 failed")
    return p1, p2


# ---- adjoint-source pipeline ----
def _c8(a):
    return np.ascontiguousarray(a, np.complex64)


def exresp25d(ndof, freq, py, yrec, sol, mrdof, recv, reference=False):
    """EXRESP25D: est (nsrc, nrec, 3) from sol (nsrc*ndof,), mrdof/recv (nrec, 3)."""
    py = np.ascontiguousarray(py, np.float64)
    yrec = np.ascontiguousarray(yrec, np.float64)
    sol, recv = _c8(sol), _c8(recv)
    mrdof = np.ascontiguousarray(mrdof, np.int32)
    nsrc, nrec = py.size, yrec.size
    est = np.zeros((nsrc, nrec, 3), np.complex64)
    if reference:
        i = lambda v: C.byref(C.c_int(v))   # noqa: E731
        ref().exresp25d_(i(3), i(nrec), i(ndof), i(nsrc), i(nrec), i(3), C.byref(C.c_double(freq)),
                         _p(py, dp), _p(yrec, dp), _p(sol, fp), _p(mrdof, ip), _p(recv, fp), _p(est, fp))
    else:
        lib().orc_exresp25d(ndof, nsrc, nrec, C.c_double(freq), _p(py, dp), _p(yrec, dp), _p(sol, fp),
                            _p(mrdof, ip), _p(recv, fp), _p(est, fp))
    return est


def bpresid4(norm, irestp, epss, freq, dtmax, swght, obs, est, reference=False):
    """BPRESID4 on (nrec, 3) arrays; returns RESID (nrec, 3) COMPLEX*8."""
    swght = np.ascontiguousarray(swght, np.float32)
    obs, est = _c8(obs), _c8(est)
    nrec = obs.shape[0]
    out = np.zeros((nrec, 3), np.complex64)
    if reference:
        i = lambda v: C.byref(C.c_int(v))   # noqa: E731
        ref().bpresid4_(i(3), i(nrec), i(3), i(norm), i(irestp), C.byref(C.c_float(epss)),
                        C.byref(C.c_double(freq)), C.byref(C.c_float(dtmax)), _p(swght, fp), _p(obs, fp),
                        _p(est, fp), _p(out, fp))
    else:
        lib().orc_bpresid4(nrec, norm, irestp, C.c_float(epss), C.c_double(freq), C.c_float(dtmax),
                           _p(swght, fp), _p(obs, fp), _p(est, fp), _p(out, fp))
    return out


def cresid(irestp, obs, est, reference=False):
    obs, est = _c8(obs).ravel(), _c8(est).ravel()
    out = np.zeros(obs.size, np.complex64)
    f = ref().ref_cresid_n if reference else lib().orc_cresid_n
    f(obs.size, irestp, _p(obs, fp), _p(est, fp), _p(out, fp))
    return out


def cphm2cm(xmag, ph, reference=False):
    xmag = np.ascontiguousarray(xmag, np.float32).ravel()
    ph = np.ascontiguousarray(ph, np.float32).ravel()
    out = np.zeros(xmag.size, np.complex64)
    f = ref().ref_cphm2cm_n if reference else lib().orc_cphm2cm_n
    f(xmag.size, _p(xmag, fp), _p(ph, fp), _p(out, fp))
    return out


def crotate(theta, q1, q2, reference=False):
    q1, q2 = _c8(q1).ravel(), _c8(q2).ravel()
    r1, r2 = np.zeros_like(q1), np.zeros_like(q2)
    f = ref().ref_crotate_n if reference else lib().orc_crotate_n
    f(q1.size, C.c_float(theta), _p(q1, fp), _p(q2, fp), _p(r1, fp), _p(r2, fp))
    return r1, r2


def hdiffer(ibphase, freq):
    out = np.zeros(2, np.float32)
    lib().orc_hdiffer_v(ibphase, C.c_double(freq), _p(out, fp))
    return np.complex64(complex(out[0], out[1]))


def resid_drhs(ndof, ibphase, freq, mrdof, resid):
    mrdof = np.ascontiguousarray(mrdof, np.int32)
    resid = _c8(resid)
    rhs = np.zeros(ndof, np.complex64)
    iw = C.c_int(0)
    lib().orc_resid_drhs(ndof, mrdof.shape[0], ibphase, C.c_double(freq), _p(mrdof, ip), _p(resid, fp),
                         _p(rhs, fp), C.byref(iw))
    return rhs, iw.value


def cadjlam_rhs(ndof, ifreq, isrc, freq, py, azmod, norm, irestp, epss, dtmax, ibphase, lunwrap, yrec,
                mrdof, est, obs, wghts):
    """CADJLAM's right-hand side (before the solve) for (ifreq, isrc), 1-based;
    est/obs COMPLEX*8 and wghts REAL*4 in the reference's (3, nfreq, nrec,
    nsrc) layout, passed as numpy arrays of shape (nsrc, nrec, nfreq, 3)."""
    est, obs = _c8(est), _c8(obs)
    wghts = np.ascontiguousarray(wghts, np.float32)
    nsrc, nrec, nfreq, _ = est.shape
    yrec = np.ascontiguousarray(yrec, np.float64)
    mrdof = np.ascontiguousarray(mrdof, np.int32)
    rhs = np.zeros(ndof, np.complex64)
    iw = C.c_int(0)
    lib().orc_cadjlam_rhs(ndof, nfreq, nrec, ifreq, isrc, C.c_double(freq), C.c_double(py), C.c_double(azmod),
                          norm, irestp, C.c_float(epss), C.c_float(dtmax), ibphase, int(lunwrap), _p(yrec, dp),
                          _p(mrdof, ip), _p(est, fp), _p(obs, fp), _p(wghts, fp), _p(rhs, fp), C.byref(iw))
    return rhs, iw.value


def rec_space1d(xrec, reference=False):
    """REC_SPACE1D: normalised receiver spacings (nrec - 1) and the error flag."""
    xrec = np.ascontiguousarray(xrec, np.float64)
    n = xrec.size
    dx = np.zeros(max(n - 1, 1), np.float64)
    if reference:
        ierr = C.c_int(0)
        ref().ref_rec_space1d(n, _p(xrec, dp), _p(dx, dp), C.byref(ierr))
        ierr = ierr.value
    else:
        ierr = lib().orc_rec_space1d(n, _p(xrec, dp), _p(dx, dp))
    return dx[:n - 1], ierr


def covd_resid(nrec, irestp, ldwght, dtmax, freq, dx, obsraw, obs, est, swght, reference=False):
    """LAPLACE_1DV2 + PERM_OBS on obsraw, BPRESID_COVD4 on (obs, est, swght),
    all (nrec, 3).  Returns (resid (nrec, 3), COVD8 (6 nrec, 6 nrec),
    iperm (nrec, 3), ierr)."""
    obsraw, obs, est = _c8(obsraw), _c8(obs), _c8(est)
    swght = np.ascontiguousarray(swght, np.float32)
    dx = np.ascontiguousarray(np.resize(np.asarray(dx, np.float64), max(nrec - 1, 1)))
    resid = np.zeros((nrec, 3), np.complex64)
    covd = np.zeros((6 * nrec, 6 * nrec), np.float64)      # column-major: covd[col, row]
    iperm = np.zeros((nrec, 3), np.int32)
    if reference and "torch" in sys.modules:
        # libtorch_cpu carries a static MKL whose exported entry points take
        # the place of the MKL the compiled reference links (its SGEMV then
        # returns wrong values): run the compiled routine in a fresh process
        out = _child_call("covd_resid", dict(nrec=nrec, irestp=irestp, ldwght=int(ldwght), dtmax=float(dtmax),
                                             freq=float(freq)),
                          dict(dx=dx, obsraw=obsraw, obs=obs, est=est, swght=swght))
        return out["resid"], out["covd"], out["iperm"], int(out["ierr"])
    if reference:
        ierr = C.c_int(0)
        ref().ref_covd_resid(nrec, irestp, int(ldwght), C.c_float(dtmax), C.c_double(freq), _p(dx, dp),
                             _p(obsraw, fp), _p(obs, fp), _p(est, fp), _p(swght, fp), _p(resid, fp),
                             _p(covd, dp), _p(iperm, ip), C.byref(ierr))
        ierr = ierr.value
    else:
        L = lib()
        ierr = L.orc_laplace_1dv2(nrec, int(ldwght), _p(dx, dp), _p(obsraw, fp), _p(covd, dp))
        if not ierr:
            ierr = L.orc_perm_obs(nrec, _p(obsraw, fp), _p(iperm, ip))
        if not ierr:
            L.orc_bpresid_covd4(nrec, _p(iperm, ip), irestp, C.c_float(dtmax), C.c_double(freq), _p(covd, dp),
                                _p(swght, fp), _p(obs, fp), _p(est, fp), _p(resid, fp))
    return resid, covd.T.copy(), iperm, ierr


def cadjlam_rhs_covd(ndof, ifreq, isrc, freq, py, azmod, irestp, dtmax, ibphase, lunwrap, ldwght, dx, yrec,
                     mrdof, est, obs, wghts):
    """CADJLAM's right-hand side with the data covariance (LCOVD); arguments
    as cadjlam_rhs with ldwght and dx (REC_SPACE1D) in place of norm and
    epss.  Returns (rhs, iwarn, ierr)."""
    est, obs = _c8(est), _c8(obs)
    wghts = np.ascontiguousarray(wghts, np.float32)
    nsrc, nrec, nfreq, _ = est.shape
    yrec = np.ascontiguousarray(yrec, np.float64)
    mrdof = np.ascontiguousarray(mrdof, np.int32)
    dx = np.ascontiguousarray(np.resize(np.asarray(dx, np.float64), max(nrec - 1, 1)))
    rhs = np.zeros(ndof, np.complex64)
    iw = C.c_int(0)
    ierr = lib().orc_cadjlam_rhs_covd(ndof, nfreq, nrec, ifreq, isrc, C.c_double(freq), C.c_double(py),
                                      C.c_double(azmod), irestp, C.c_float(dtmax), ibphase, int(lunwrap),
                                      int(ldwght), _p(dx, dp), _p(yrec, dp), _p(mrdof, ip), _p(est, fp),
                                      _p(obs, fp), _p(wghts, fp), _p(rhs, fp), C.byref(iw))
    return rhs, iw.value, ierr

def fill_uwave(mesh, g, kappax, kappaz, baz, aoi, reference=False, model=None, pml=None):
    """FILL_UWAVE_QMESH's plane wave at every DOF, complex128 (ndof,)."""
    ue = np.zeros(g.ndof, np.complex128)
    if reference:
        ierr = C.c_int(0)
        ieng = np.ascontiguousarray(mesh.ieng, np.int32)
        lm = np.ascontiguousarray(g.lm, np.int32)
        ref().ref_fill_uwave(mesh.nord, mesh.nelem, mesh.nnpg, g.ndof, _p(ieng, ip),
                             _p(np.ascontiguousarray(mesh.xlocs), dp), _p(np.ascontiguousarray(mesh.zlocs), dp),
                             _p(lm, ip), C.c_double(kappax), C.c_double(kappaz), C.c_double(baz),
                             C.c_double(aoi), _p(ue, dp), C.byref(ierr))
        ierr = ierr.value
    else:
        from fem25_amd.configs import PML, homogeneous_model
        s, keep = _asm_struct(mesh, model if model is not None else homogeneous_model(mesh), g, pml or PML())
        ierr = lib().orc_fill_uwave(C.byref(s), C.c_double(kappax), C.c_double(kappaz), C.c_double(baz),
                                    C.c_double(aoi), _p(ue, dp))
    if ierr:
        raise RuntimeError("fill_uwave failed")
    return ue

def _elem_inputs(nord, xlocs, zlocs, dens, ecoeff):
    xlocs = np.ascontiguousarray(xlocs, np.float64)
    zlocs = np.ascontiguousarray(zlocs, np.float64)
    dens = np.ascontiguousarray(dens, np.float64)
    ecoeff = np.asfortranarray(np.asarray(ecoeff, np.float64).reshape(-1, 2))
    return xlocs, zlocs, dens, ecoeff


def djacab2(nord, inpg, xlocs, zlocs, dens, ecoeff, tables=None):
    """DJACAB2 on the element with anchors 1..4 (1-based inpg); returns
    det (nq,), dab (2, nq), dab2 (2, nq), shg (nq, nen, 3), q = ix + nint*iz.
    tables = (abscissae, shl) replaces the oracle's own DSHL tables."""
    nint, nen = 2 * nord + 5, (nord + 1) ** 2
    if tables is None:
        _, xq, _, shl = dshl(nord)
    else:
        xq, shl = (np.ascontiguousarray(t, np.float64) for t in tables)
    xlocs, zlocs, dens, ecoeff = _elem_inputs(nord, xlocs, zlocs, dens, ecoeff)
    ieng = np.arange(1, 5, dtype=np.int32)
    nq = nint * nint
    det, dab, dab2 = np.zeros(nq), np.zeros(2 * nq), np.zeros(2 * nq)
    shg = np.zeros(3 * nen * nq)
    shl = np.ascontiguousarray(shl.ravel())
    if lib().orc_djacab2(nen, nint, inpg, _p(ieng, ip), _p(xq, dp), _p(xlocs, dp), _p(zlocs, dp),
                         _p(dens, dp), _p(ecoeff.ravel(order="F"), dp), len(dens), _p(shl, dp),
                         _p(det, dp), _p(dab, dp), _p(dab2, dp), _p(shg, dp)):
        raise RuntimeError("orc_djacab2 failed")
    return det, dab.reshape(2, nq), dab2.reshape(2, nq), shg.reshape(nq, nen, 3)


def ref_djacab2(nord, inpg, xlocs, zlocs, dens, ecoeff):
    """The reference's DJACAB2 (compiled), same layout as djacab2()."""
    nint, nen = 2 * nord + 5, (nord + 1) ** 2
    xg, _, shl = ref_dshl(nord)
    xlocs, zlocs, dens, ecoeff = _elem_inputs(nord, xlocs, zlocs, dens, ecoeff)
    ieng = np.arange(1, 5, dtype=np.int32)
    nq = nint * nint
    det, dab, dab2 = np.zeros(nq), np.zeros(2 * nq), np.zeros(2 * nq)
    shg = np.zeros(3 * nen * nq)
    shl = np.ascontiguousarray(shl.ravel())
    ierr = C.c_int(0)
    i = lambda v: C.byref(C.c_int(v))   # noqa: E731
    ec = np.ascontiguousarray(ecoeff.ravel(order="F"))
    xg = np.ascontiguousarray(xg)
    ref().djacab2_(i(nen), i(nint), i(nint), i(len(dens)), i(1), i(nint), i(nint), i(nen), i(4),
                   i(len(dens)), i(inpg), _p(ieng, ip), _p(xg, dp), _p(xg, dp), _p(xlocs, dp),
                   _p(zlocs, dp), _p(dens, dp), _p(ec, dp), _p(shl, dp), _p(det, dp), _p(dab, dp),
                   _p(dab2, dp), _p(shg, dp), C.byref(ierr))
    if ierr.value:
        raise RuntimeError("reference DJACAB2 failed")
    return det, dab.reshape(2, nq), dab2.reshape(2, nq), shg.reshape(nq, nen, 3)


def _dab_out(nee):
    return [np.zeros(nee * nee), np.zeros(nee * nee), np.zeros(nee * nee, np.complex128),
            np.zeros(nee * nee, np.complex128)]


def dabmkisob25(nord, lisp, liss, omega, py, det, dab, shg, reference=False, dab2=None, wq=None):
    """DABMKISOB25 (or, with dab2, DABM2KISOB25) from DJACAB(2) outputs; the
    oracle's restatement or, with reference=True, the compiled routine.
    Returns the NEE x NEE matrices (Fortran order) DMDA, DMDB, DKDA, DKDB
    (+ the four second-derivative ones with dab2)."""
    nint, nen = 2 * nord + 5, (nord + 1) ** 2
    nee = 3 * nen
    if wq is None:
        wq = ref_dshl(nord)[1] if reference else dshl(nord)[2]
    wq = np.ascontiguousarray(wq, np.float64)
    det = np.ascontiguousarray(det, np.float64)
    dab = np.ascontiguousarray(dab, np.float64).ravel()
    shg = np.ascontiguousarray(shg, np.float64).ravel()
    out = _dab_out(nee) + (_dab_out(nee) if dab2 is not None else [])
    ptrs = [_p(o, dp) for o in out]
    if reference:
        i = lambda v: C.byref(C.c_int(v))   # noqa: E731
        head = [i(nen), i(nee), i(nint), i(nint), i(nen), i(nint), i(nint), i(int(lisp)), i(int(liss)),
                C.byref(C.c_double(omega)), C.byref(C.c_double(py)), _p(wq, dp), _p(wq, dp), _p(det, dp),
                _p(dab, dp)]
        if dab2 is None:
            ref().dabmkisob25_(*head, _p(shg, dp), *ptrs)
        else:
            d2 = np.ascontiguousarray(dab2, np.float64).ravel()
            ref().dabm2kisob25_(*head, _p(d2, dp), _p(shg, dp), *ptrs)
    else:
        args = [nen, nint, int(lisp), int(liss), C.c_double(omega), C.c_double(py), _p(wq, dp),
                _p(det, dp), _p(dab, dp)]
        if dab2 is None:
            lib().orc_dabmkisob25(*args, _p(shg, dp), *ptrs)
        else:
            d2 = np.ascontiguousarray(dab2, np.float64).ravel()
            lib().orc_dabm2kisob25(*args, _p(d2, dp), _p(shg, dp), *ptrs)
    return [o.reshape(nee, nee, order="F") for o in out]


def adjflam_dist(inv: Inv, fmat, adjlam) -> np.ndarray:
    out = np.zeros(inv.na35, np.float32)
    fmat = np.ascontiguousarray(fmat, np.complex64)
    adjlam = np.ascontiguousarray(adjlam, np.complex64)
    lib().orc_adjflam_dist(inv.nnpgl, inv.na35, _p(inv.mygrad, ip), _p(inv.jcsc, ip),
                           _p(inv.icsc, ip), _p(fmat, fp), _p(adjlam, fp), _p(out, fp))
    return out


def pchadj_jac(inv: Inv, nrhs, lrhs, g, fmat):
    """PCHADJ's J = G^T F (COMPLEX*8) and diag(J^H J) per gradient point.
    g: (nrhs, lrhs) complex64 (GRNSFNS((irhs-1)*LRHS + jdof)); returns
    jac (nnpgl, nrhs) complex64 and hdiag (na35,) float32."""
    g = np.ascontiguousarray(g, np.complex64)
    fmat = np.ascontiguousarray(fmat, np.complex64)
    jac = np.zeros((inv.nnpgl, nrhs), np.complex64)
    hd = np.zeros(inv.na35, np.float32)
    lib().orc_pchadj_jac(inv.nnpgl, nrhs, lrhs, _p(inv.mygrad, ip), _p(inv.jcsc, ip),
                         _p(inv.icsc, ip), _p(g, fp), _p(fmat, fp), _p(jac, fp), _p(hd, fp))
    return jac, hd


def gn_hessian(nobs, alpha, nnpgl, jac):
    """GENHLOC's local J^T J: (nnpgl, nnpgl) FP64, H[c2, c1] in row-major =
    sum_j alpha_j Re(J_j(:,c1)^H J_j(:,c2)) (symmetric)."""
    nobs = np.ascontiguousarray(nobs, np.int32)
    alpha = np.ascontiguousarray(alpha, np.float64)
    jac = np.ascontiguousarray(jac, np.complex64)
    h = np.zeros((nnpgl, nnpgl))
    lib().orc_gn_hessian(len(nobs), _p(nobs, ip), _p(alpha, dp), nnpgl, _p(jac, fp), _p(h, dp))
    return h


def ref_write_jac(path, nrhsf, nnpgl, ndim, nrec, lobs, jac, mygrad):
    """The Jacobian file written by PCHADJ's WRITE statements (pchadj.f90:371-395),
    compiled with the reference's compiler (harness REF_WRITE_JAC)."""
    lobs = np.ascontiguousarray(lobs, np.int32)
    jac = np.ascontiguousarray(jac, np.complex64)
    mygrad = np.ascontiguousarray(mygrad, np.int32)
    b = os.fsencode(path)
    ref().ref_write_jac(C.c_char_p(b), len(b), nrhsf, nnpgl, ndim, nrec, _p(lobs, ip), _p(jac, fp), _p(mygrad, ip))


def gnmfree(nobs, alpha, nnpgl, mygrad, na35, jac, p):
    """GNMFREE's z = sum_j alpha_j Re(J_j^H J_j p(MYGRAD)); jac packed (j, c, obs)."""
    nobs = np.ascontiguousarray(nobs, np.int32)
    alpha = np.ascontiguousarray(alpha, np.float64)
    mygrad = np.ascontiguousarray(mygrad, np.int32)
    jac = np.ascontiguousarray(jac, np.complex64)
    p = np.ascontiguousarray(p, np.float64)
    z = np.zeros(na35)
    lib().orc_gnmfree(len(nobs), _p(nobs, ip), _p(alpha, dp), nnpgl, _p(mygrad, ip), na35,
                      _p(jac, fp), _p(p, dp), _p(z, dp))
    return z


def ref_gnmfree(freqs, nsrc, source, lmigr, nnpgl, mygrad, na35, nobs, jac, p, workdir):
    """Compiled reference GNMFREE; the Jacobian files are written under
    workdir/scratch in the reference's own format.  nobs: (nfreq, nsrc)."""
    import os
    freqs = np.ascontiguousarray(freqs, np.float64)
    nfreq = freqs.size
    source = np.asfortranarray(np.asarray(source, np.complex64).reshape(nfreq, nsrc))
    nobs = np.ascontiguousarray(np.asarray(nobs, np.int32).reshape(nfreq, nsrc))
    mygrad = np.ascontiguousarray(mygrad, np.int32)
    jac = np.ascontiguousarray(jac, np.complex64)
    p = np.ascontiguousarray(p, np.float64)
    z = np.zeros(na35)
    ierr = C.c_int(0)
    os.makedirs(os.path.join(workdir, "scratch"), exist_ok=True)
    cwd = os.getcwd()
    os.chdir(workdir)
    try:
        ref().ref_gnmfree(nfreq, nsrc, _p(freqs, dp), source.ctypes.data_as(fp), int(lmigr), nnpgl,
                          na35, _p(mygrad, ip), _p(nobs, ip), _p(jac, fp), _p(p, dp), _p(z, dp),
                          C.byref(ierr))
    finally:
        os.chdir(cwd)
    if ierr.value:
        raise RuntimeError(f"reference GNMFREE failed ({ierr.value})")
    return z


def grad_exact(mesh, model, g, freq, py, u, lam, pml=None):
    """g = Re(lam^H dS/dm u) for anchor (lambda, mu, rho) and (Vp, Vs, rho)."""
    from fem25_amd.configs import PML
    s, keep = _asm_struct(mesh, model, g, pml or PML())
    glmr = np.zeros(3 * mesh.nnpg)
    gvvr = np.zeros(3 * mesh.nnpg)
    u = np.ascontiguousarray(u, np.complex128)
    lam = np.ascontiguousarray(lam, np.complex128)
    if lib().orc_grad_exact(C.byref(s), C.c_double(freq), C.c_double(py), _p(u, dp),
                            _p(lam, dp), _p(glmr, dp), _p(gvvr, dp)):
        raise RuntimeError("orc_grad_exact failed")
    return glmr.reshape(-1, 3), gvvr.reshape(-1, 3)


# ---- element-level entry points ----
def gll(n):
    x = np.zeros(n)
    w = np.zeros(n)
    lib().orc_gll(n, _p(x, dp), _p(w, dp))
    return x, w


def dshl(nord):
    nl = nord + 1
    nint = 2 * nord + 5
    xipts = np.zeros(nl)
    xq = np.zeros(nint)
    wq = np.zeros(nint)
    shl = np.zeros(3 * nl * nl * nint * nint)
    lib().orc_dshl(nl, nint, _p(xipts, dp), _p(xq, dp), _p(wq, dp), _p(shl, dp))
    return xipts, xq, wq, shl.reshape(nint, nint, nl * nl, 3)   # [iz][ix][a][c]


def ref_dshl(nord):
    nl = nord + 1
    nint = 2 * nord + 5
    nen = nl * nl
    xigll = np.zeros((2, nint))          # Fortran XIGLL(NINT,2)
    etagll = np.zeros((2, nint))
    shl = np.zeros(3 * nen * nint * nint)
    xiin = np.zeros(nl)
    i = lambda v: C.byref(C.c_int(v))
    ref().dshl_(i(nen), i(nint), i(nint), i(1), i(nint), i(nint), i(nl), i(nl), _p(xiin, dp),
                _p(xiin, dp), _p(xigll, dp), _p(etagll, dp), _p(shl, dp))
    return xigll[0], xigll[1], shl.reshape(nint, nint, nen, 3)
