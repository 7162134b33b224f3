"""The paths that parallelograms and elements of general shape take, each where
its kernels can go wrong: several chunks of pairs a wave and both groups of 64
pairs, sides along the axes and sheared, rings and perturbations of either
kind or both, graphs and residuals."""
from __future__ import annotations

import numpy as np
import pytest
import scipy.sparse as sp

import oracle
from fem25_amd import configs as cf
from tests.helpers import TWOPI, csr, relerr
from tests.test_routes import (F32, F64, batch, err, general, handle, mixed_mesh, product, pw, row_tiles,
                               vectors)

pytestmark = pytest.mark.gpu


def sheared(nx, nz, p, **kw):
    """Parallelograms only, none with sides along the axes (exact in FP64)."""
    m = cf.structured_mesh(nx, nz, p, width=1e3 * nx, depth=1e3 * nz, **kw)
    m.xlocs += 0.25 * m.zlocs
    return m


def new_handle(m, pml=None, seed=11):
    from fem25_amd.api import MeshInfo
    mi = MeshInfo(m, pml or cf.PML())
    mod = cf.layered_model(m, seed=seed, n_anom=4, amp=0.1)
    mi.set_model(mod)
    return mi, mod


@pytest.mark.parametrize("shear", [False, True])
@pytest.mark.parametrize("p", [3, 4, 5, 6])
def test_waves_with_several_chunks_of_pairs(p, shear):
    """1,400 elements a colour: four waves an element, 9 PW + 1 pairs, so that
    every wave walks two or three chunks (the next one's values, omega and ky
    arrive while it works).  FP64 against blocks; FP32 (p4 and up by sum
    factorisation) against the same, four roundings of a stored value."""
    import torch
    m = sheared(80, 70, p) if shear else cf.structured_mesh(80, 70, p, width=80e3, depth=70e3)
    assert not general(m).any()
    mi, _ = new_handle(m)
    n = 9 * pw(p) + 1
    om, ky = batch(n)
    x = vectors(mi, n)
    want = product(mi, om, ky, x, tiles=row_tiles(p))
    e64 = err(product(mi, om, ky, x), want)
    x32 = x.to(torch.complex64)
    got32 = product(mi, om, ky, x32, F32).to(torch.complex128)
    e32 = err(got32, product(mi, om, ky, x32.to(torch.complex128), tiles=row_tiles(p)))
    print(f"p{p} shear {shear} {n} pairs: {e64:.2e} {e32:.2e}", flush=True)
    assert e64 < 1e-13
    assert e32 < (2.4e-7 if p >= 4 else 2e-6)
    mi.close()


@pytest.mark.parametrize("p", [4, 5, 6])
def test_block_product_of_two_pair_groups(p):
    """70 pairs (a second group of 64, partly empty) of a mesh with elements of
    general shape, which runs on blocks, and of parallelograms sent there by
    row tiles, against the oracle's operator."""
    n = 70
    om, ky, f, py = (v[:n] for v in cf.freq_ky_batch(7, 10, 0.02, 0.1, 3500.0))
    for m, tiles in ((mixed_mesh(5, 4, p, every=4), 0), (sheared(5, 4, p), row_tiles(p))):
        assert general(m).any() == (tiles == 0)
        mi, mod = new_handle(m)
        g = oracle.graph(m)
        x = cf.seeded_complex(g.ndof, batch=n, seed=21)
        mi.set_apply_tiles(tiles)
        y = mi.apply_batch(om, ky, x)
        for b in (0, 63, 64, 69):
            S = csr(g, oracle.asmble_z(m, mod, g, f[b], py[b], cf.PML()))
            assert relerr(y[b], S @ x[b]) < 1e-12, (tiles, b)
        mi.close()


def _peff(m, mod, g, pml, freq, py, ue):
    """-S_BE u_E on 'B' rows, +S_EB u_E on 'E' rows from the oracle's operator."""
    S = csr(g, oracle.asmble_z(m, mod, g, freq, py, pml)).tocoo()
    cnp = np.frombuffer(g.cnp, dtype="S1")
    sign = (np.where((cnp[S.row] == b"B") & (cnp[S.col] == b"E"), -1.0, 0.0)
            + np.where((cnp[S.row] == b"E") & (cnp[S.col] == b"B"), 1.0, 0.0))
    return sp.csr_matrix((S.data * sign, (S.row, S.col)), shape=S.shape) @ ue


@pytest.mark.parametrize("p", [2, 4, 6])
@pytest.mark.parametrize("kind", ["rectangles", "sheared", "mixed"])
def test_effective_force_by_kind_of_ring(p, kind):
    """Rings of rectangles and of sheared parallelograms (sum factorisation, its
    own DOF maps in and out), and with elements of general shape (blocks);
    the plane-wave sources in a graph equal the eager ones bit for bit."""
    import torch
    pml = cf.PML(rcoeff=1e-3, kappa=1.0, fcent=0.05)
    kw = dict(npml=1, nbielak=1)
    if kind == "rectangles":
        m = cf.structured_mesh(9, 6, p, width=9e3, depth=6e3, **kw)
    else:
        m = mixed_mesh(9, 6, p, every=3, **kw) if kind == "mixed" else sheared(9, 6, p, **kw)
    assert general(m).any() == (kind == "mixed")
    mi, mod = new_handle(m, pml)
    g = oracle.graph(m)
    n = 66 if p == 2 else 11
    om, ky = batch(n)
    u = vectors(mi, n, seed=7)
    pe = torch.empty_like(u)
    mi.peff_batch_dev(om, ky, u, pe)
    uh, got = u.cpu().numpy(), pe.cpu().numpy()
    for b in (0, n // 2, n - 1):
        want = _peff(m, mod, g, pml, om[b] / TWOPI, ky[b] / om[b], uh[:, b])
        assert np.count_nonzero(want) and relerr(got[:, b], want) < 1e-12, b
    kx, kz = om / 6000.0, 0.5 * om / 6000.0
    bz, ai = np.linspace(-40, 40, n), np.linspace(10, 50, n)
    ue, eager, rep = (torch.empty(mi.ndof * n, dtype=torch.complex128, device="cuda") for _ in range(3))
    mi.bielak_rhs_dev(om, ky, kx, kz, bz, ai, ue, eager)
    for _ in range(3):
        rep.fill_(complex(float("nan"), 0.0))
        mi.bielak_rhs_dev(om, ky, kx, kz, bz, ai, ue, rep, graph=True)
        mi.peff_batch_dev(om, ky, u, pe)            # eager work between the replays
        assert torch.equal(rep, eager)
    mi.close()


@pytest.mark.parametrize("kind", ["sheared", "mixed"])
@pytest.mark.parametrize("p", [2, 4, 6])
def test_model_perturbation_by_kind(p, kind):
    """F v on records alone and on blocks (a small mesh of both kinds) against
    a central difference of the oracle's operator."""
    m = mixed_mesh(5, 4, p, every=4) if kind == "mixed" else sheared(5, 4, p)
    assert general(m).any() == (kind == "mixed")
    mi, mod = new_handle(m)
    g = oracle.graph(m)
    v = np.random.default_rng(51).standard_normal((m.nnpg, 3)) * np.array([50.0, 30.0, 20.0])
    f, py, h = 0.07, 0.6e-4, 1e-3
    u = cf.seeded_complex(g.ndof, seed=52)
    fv = mi.gn_fv(np.array([TWOPI * f]), np.array([TWOPI * f * py]), u, v)[0]
    S = [csr(g, oracle.asmble_z(m, cf.model_from_velocity(mod.vp + s * v[:, 0], mod.vs + s * v[:, 1],
                                                          mod.dens + s * v[:, 2]), g, f, py, cf.PML()))
         for s in (h, -h)]
    assert relerr(fv, (S[0] @ u - S[1] @ u) / (2 * h)) < 1e-9
    mi.close()


def test_both_kinds_in_one_call():
    """A mesh whose colours launch both kernels (4,148 elements, p4): the
    perturbation's records beside its blocks against blocks alone; a captured
    product replayed for new models and frequencies, and the residual, equal
    the eager product bit for bit."""
    import torch
    from fem25_amd import _lib
    p, n = 4, 3
    mi = handle(68, 61, p, 37)
    om, ky = batch(n)
    rng = np.random.default_rng(3)
    v = rng.standard_normal((mi.mesh.nnpg, 3)) * np.array([50.0, 30.0, 20.0])
    u = cf.seeded_complex(mi.ndof, batch=n, seed=4)
    fv = mi.gn_fv(om, ky, u, v)
    mi.set_apply_tiles(row_tiles(p))
    on_blocks = mi.gn_fv(om, ky, u, v)
    mi.set_apply_tiles(0)
    assert relerr(fv, on_blocks) < 1e-13
    x = vectors(mi, n)
    y, r = torch.empty_like(x), torch.empty_like(x)
    for k in range(3):
        mi.set_model(cf.layered_model(mi.mesh, seed=20 + k))
        o = om * (1.0 + 0.1 * k)
        want = product(mi, o, ky, x)
        mi.apply_batch_dev(o, ky, x, y, F64 | _lib.F25_APPLY_GRAPH)
        torch.cuda.synchronize()
        assert torch.equal(y, want), k
        mi.residual_batch_dev(o, ky, x, want, r)
        assert not r.any()
        x.mul_(1.5)
