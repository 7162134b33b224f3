"""Parallelogram elements (affine.hip) beside elements of general shape: a
sheared mesh whose one displaced anchor leaves four elements non-affine, so
both kinds of kernels write one result.  Batches at the edges of a wave's
vectors (PW of them) and of a workgroup's four waves, against the oracle."""
from __future__ import annotations

import functools

import numpy as np
import pytest
import scipy.sparse as sp

import oracle
from fem25_amd import configs as cf

TWOPI = 2.0 * np.pi


def pw(p: int) -> int:
    """Complex vectors of one wave: half of the even number of (p + 1)-lane groups in 64."""
    return (64 // (p + 1)) // 2


@functools.lru_cache(maxsize=None)
def case(p: int, npml: int = 0):
    nx, nz = (8, 6) if npml else (5, 4)
    m = cf.structured_mesh(nx, nz, p, width=2e3 * nx, depth=2e3 * nz, npml=npml, nbielak=1 if npml else 0)
    if not npml:
        m.xlocs += 0.25 * m.zlocs              # exact in FP64: every element a parallelogram
    a = (nz // 2) * (nx + 1) + nx // 2
    m.xlocs[a] += 310.0
    m.zlocs[a] -= 170.0
    mod = cf.layered_model(m, seed=11, n_anom=4, amp=0.1)
    pml = cf.PML(rcoeff=1e-3, kappa=1.0, fcent=0.05) if npml else cf.PML()
    return m, mod, pml, oracle.graph(m)


@functools.lru_cache(maxsize=None)
def handle(p: int, npml: int = 0):
    from fem25_amd.api import MeshInfo
    m, mod, pml, _ = case(p, npml)
    mi = MeshInfo(m, pml)
    mi.set_model(mod)
    return mi


def batch(n: int):
    om, ky, f, py = cf.freq_ky_batch(3, (n + 2) // 3, 0.02, 0.1, 3500.0)
    return om[:n], ky[:n], f[:n], py[:n]


def err(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def test_mixed_mesh_has_both_kinds():
    for p in (2, 6):
        m, *_ = case(p)
        x, z = m.xlocs[m.ieng - 1], m.zlocs[m.ieng - 1]
        twist = [np.abs(v[:, 0] - v[:, 1] + v[:, 2] - v[:, 3]) for v in (x, z)]
        assert np.count_nonzero(twist[0] + twist[1]) == 4


@pytest.mark.gpu
@pytest.mark.parametrize("p", [2, 3, 4, 5, 6])
def test_gradient(p):
    m, mod, pml, g = case(p)
    mi = handle(p)
    n = 4 * pw(p) + 1
    om, ky, f, py = batch(n)
    u, lam = cf.seeded_complex(g.ndof, batch=n, seed=1), cf.seeded_complex(g.ndof, batch=n, seed=2)
    each = [oracle.grad_exact(m, mod, g, f[b], py[b], u[b], lam[b], pml)[1] for b in range(n)]
    for k in (1, pw(p), pw(p) + 1, n):
        ref, got = sum(each[:k]), mi.gradient(om[:k], ky[:k], u[:k], lam[:k])
        for c in range(3):
            assert err(got[:, c], ref[:, c]) < 1e-12, (k, c)


@pytest.mark.gpu
@pytest.mark.parametrize("npml", [0, 2])
@pytest.mark.parametrize("p", [2, 3, 4, 5, 6])
def test_product(p, npml):
    import torch
    from fem25_amd import _lib
    m, mod, pml, g = case(p, npml)
    mi = handle(p, npml)
    n = 4 * pw(p) + 1
    om, ky, f, py = batch(n)
    x = cf.seeded_complex(g.ndof, batch=n, seed=3)
    probe = sorted({0, pw(p) - 1, pw(p), n - 1})
    ref = {b: sp.csr_matrix((oracle.asmble_z(m, mod, g, f[b], py[b], pml), g.jcptr - 1, g.irptr - 1),
                            shape=(g.ndof, g.ndof)) @ x[b] for b in probe}
    for k in (1, pw(p), pw(p) + 1, n):
        y = mi.apply_batch(om[:k], ky[:k], x[:k])
        for b in probe:
            if b < k:
                assert err(y[b], ref[b]) < 1e-12, (k, b)
    x32 = torch.from_numpy(np.ascontiguousarray(x.T)).to(torch.complex64).cuda()
    y32 = torch.empty_like(x32)
    mi.apply_batch_dev(om, ky, x32, y32, _lib.F25_APPLY_F32)
    y32 = y32.cpu().numpy().T
    assert all(err(y32[b], ref[b]) < 2e-6 for b in probe)


@pytest.mark.gpu
@pytest.mark.parametrize("p", [2, 3, 4])
def test_product_both_sides_of_the_batch_rule(p):
    """2,048 parallelograms: below 2^18 products the element-wise kernel, from
    there on blocks at p2 (and at p3 in FP32).  The same pairs either way,
    within the rounding of each kind."""
    import torch
    from fem25_amd import _lib
    from fem25_amd.api import MeshInfo
    m = cf.structured_mesh(64, 32, p, width=64e3, depth=32e3)
    mi = MeshInfo(m)
    mi.set_model(cf.layered_model(m, seed=11, n_anom=4, amp=0.1))
    om, ky, _, _ = cf.freq_ky_batch(8, 16, 0.02, 0.1, 3500.0)
    x = torch.randn(mi.ndof, 128, dtype=torch.complex128, device="cuda",
                    generator=torch.Generator(device="cuda").manual_seed(5))
    y = {}
    for n in (127, 128):
        xn = x[:, :n].contiguous()
        for mode, xx in ((_lib.F25_APPLY_F64, xn), (_lib.F25_APPLY_F32, xn.to(torch.complex64))):
            out = torch.empty_like(xx)
            mi.apply_batch_dev(om[:n], ky[:n], xx, out, mode)
            y[n, mode] = out.to(torch.complex128)
    for (n, mode), v in y.items():
        ref = y[127, _lib.F25_APPLY_F64]
        e = torch.linalg.norm(v[:, :127] - ref, dim=0) / torch.linalg.norm(ref, dim=0)
        assert float(e.max()) < (1e-12 if mode == _lib.F25_APPLY_F64 else 2e-6), (n, mode)
    mi.close()


@pytest.mark.gpu
@pytest.mark.parametrize("disp", [False, True])
@pytest.mark.parametrize("p", [2, 3, 4, 5, 6])
def test_assembled_with_elements_per_omega(p, disp):
    """PML elements, and in a dispersive medium every element, integrated per
    call, some of general shape (both geometries of the element matrices); and
    the assembled operator's product in both types."""
    import torch
    from fem25_amd.api import MeshInfo
    m, mod, pml, g = case(p, 2)
    if disp:
        mod = cf.with_attenuation(mod, 120.0, 60.0, 1.0)
    mi = MeshInfo(m, pml)
    mi.set_model(mod)
    for f, py in ((0.05, 0.0), (0.08, 9e-5)):
        ref = oracle.asmble_z(m, mod, g, f, py, pml)
        assert err(mi.asmble(b"B", f, py, complex128=True), ref) < 1e-13
        got = mi.asmble(b"B", f, py)
        assert np.max(np.abs(got - ref)) < 1e-6 * np.max(np.abs(ref))
        x = cf.seeded_complex(g.ndof, seed=5)
        want = sp.csr_matrix((ref, g.jcptr - 1, g.irptr - 1), shape=(g.ndof, g.ndof)) @ x
        for dt, tol in ((torch.complex128, 1e-13), (torch.complex64, 1e-6)):
            s, xd = (torch.from_numpy(np.ascontiguousarray(a)).to(dt).cuda() for a in (ref, x))
            y = torch.empty_like(xd)
            mi.csr_apply_dev(s, xd, y)
            assert err(y.cpu().numpy(), want) < tol
    mi.close()
