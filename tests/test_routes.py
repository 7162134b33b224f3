"""Which elements of a batched product run by sum factorisation and which on
their blocks: the rule at the sizes where both were timed, and the products of
meshes that hold both kinds on the two routes."""
from __future__ import annotations

import functools
from fractions import Fraction

import numpy as np
import pytest

from fem25_amd import _lib
from fem25_amd import configs as cf

F64, F32 = _lib.F25_APPLY_F64, _lib.F25_APPLY_F32


def pw(p: int) -> int:
    """Complex vectors of one wave: half of the even number of (p + 1)-lane groups in 64."""
    return (64 // (p + 1)) // 2


def row_tiles(p: int) -> int:
    """The order's own row tiles: asked for, every element runs on its blocks."""
    return 1 if p <= 4 else 2


def general(m) -> np.ndarray:
    """Elements that are no parallelograms (coordinates exact in FP64)."""
    x, z = m.xlocs[m.ieng - 1], m.zlocs[m.ieng - 1]
    return sum(np.abs(v[:, 0] - v[:, 1] + v[:, 2] - v[:, 3]) for v in (x, z)) > 0


def mixed_mesh(nx, nz, p, every=37, shear=0.25, **kw):
    """A sheared mesh with every 37th anchor off the outer sides displaced."""
    m = cf.structured_mesh(nx, nz, p, width=1e3 * nx, depth=1e3 * nz, **kw)
    m.xlocs += shear * m.zlocs
    cn = np.frombuffer(m.cnnpg, "S2")
    ix, iz = np.arange(m.nnpg) % (nx + 1), np.arange(m.nnpg) // (nx + 1)
    a = np.flatnonzero((cn != b"AA") & (ix > 0) & (ix < nx) & (iz > 0) & (iz < nz))[::every]
    m.xlocs[a] += 155.0
    m.zlocs[a] -= 85.0
    return m


@functools.lru_cache(maxsize=1)
def handle(nx, nz, p, every):
    from fem25_amd.api import MeshInfo
    m = mixed_mesh(nx, nz, p, every) if every else cf.structured_mesh(nx, nz, p, width=1e3 * nx, depth=1e3 * nz)
    mi = MeshInfo(m)
    mi.set_model(cf.layered_model(m, seed=11, n_anom=4, amp=0.1))
    return mi


def batch(n: int):
    om, ky, _, _ = cf.freq_ky_batch(3, (n + 2) // 3, 0.02, 0.1, 3500.0)
    return om[:n], ky[:n]


def vectors(mi, n, seed=5):
    import torch
    return torch.randn(mi.ndof, n, dtype=torch.complex128, device="cuda",
                       generator=torch.Generator(device="cuda").manual_seed(seed))


def product(mi, om, ky, x, mode=F64, tiles=0):
    import torch
    y = torch.full_like(x, complex(float("nan"), float("nan")))
    mi.set_apply_tiles(tiles)
    mi.apply_batch_dev(om, ky, x, y, mode)
    mi.set_apply_tiles(0)
    return y


def err(a, b):
    """The largest normwise error of a column."""
    import torch
    return float((torch.linalg.norm(a - b, dim=0) / torch.linalg.norm(b, dim=0)).max())


def parallelogram(x, z) -> bool:
    x, z = np.ascontiguousarray(x, np.float64), np.ascontiguousarray(z, np.float64)
    return _lib.load().f25_selftest_parallelogram(x.ctypes.data_as(_lib.dp), z.ctypes.data_as(_lib.dp)) == 1


def share(m) -> float:
    return float(np.mean([parallelogram(m.xlocs[a - 1], m.zlocs[a - 1]) for a in m.ieng]))


def twist(x, z) -> float:
    """max |J^-1 b| of the bilinear map, in rational arithmetic."""
    x, z = [Fraction(float(v)) for v in x], [Fraction(float(v)) for v in z]
    xx, xe, b1 = x[1] - x[0] + x[2] - x[3], x[3] - x[0] + x[2] - x[1], x[0] - x[1] + x[2] - x[3]
    zx, ze, b2 = z[1] - z[0] + z[2] - z[3], z[3] - z[0] + z[2] - z[1], z[0] - z[1] + z[2] - z[3]
    det = xx * ze - xe * zx
    return float(max(abs((ze * b1 - xe * b2) / det), abs((xx * b2 - zx * b1) / det)))


def test_parallelograms_of_meshes():
    """Structured meshes are all parallelograms, exact shears too; rounded
    shears in part, and what is accepted there has no twist to speak of."""
    for nx, nz in ((200, 100), (97, 61)):
        m = cf.structured_mesh(nx, nz, 2)
        assert share(m) == 1.0
        m.xlocs += 0.25 * m.zlocs
        assert 0.5 < share(m) <= 1.0
        for a in m.ieng[:: 7]:
            if parallelogram(m.xlocs[a - 1], m.zlocs[a - 1]):
                assert twist(m.xlocs[a - 1], m.zlocs[a - 1]) < 1e-15
    m = mixed_mesh(20, 14, 2)
    assert share(m) == 1.0 - np.mean(general(m))


@pytest.mark.parametrize("lx,lz", [(1e4, 10.0), (10.0, 1e4), (400.0, 400.0), (1e5, 1.0)])
def test_twist_is_measured_in_the_elements_own_shape(lx, lz):
    """A twist of the short side, far below the rounding of the long one, is
    refused at any aspect ratio; one within the rounding of the side it moves
    is accepted."""
    x, z = np.array([0.0, lx, lx, 0.0]), np.array([0.0, 0.0, lz, lz])
    assert parallelogram(x, z)
    for v, h in ((x, lx), (z, lz)):
        w = v.copy()
        w[2] += 1e-14 * h
        e = (w, z) if v is x else (x, w)
        assert twist(*e) > 1e-15 and not parallelogram(*e)
    w = z.copy()
    w[2] = np.nextafter(lz, 2 * lz)
    assert parallelogram(x, w) and twist(x, w) < 2.3e-16
    assert not parallelogram(x[[0, 3, 2, 1]], z[[0, 3, 2, 1]])      # clockwise
    assert not parallelogram(x, 0 * z)                              # no area


# (order, elements, parallelograms, PML elements, pairs, mode, sum factorisation faster) as timed
@pytest.mark.parametrize("p,nin,npar,npml,n,mode,sf", [
    (2, 800, 700, 0, 8, F64, False), (2, 5917, 5680, 0, 8, F64, False), (2, 20000, 10600, 0, 8, F64, True),
    (2, 20000, 19000, 0, 40, F64, False), (3, 2048, 1960, 0, 8, F64, False), (3, 5917, 3136, 0, 8, F64, True),
    (3, 5917, 5200, 0, 45, F64, False), (4, 800, 770, 0, 1, F64, False), (4, 5917, 3136, 0, 24, F64, True),
    (4, 5917, 5200, 0, 45, F64, False), (4, 5917, 590, 0, 8, F64, False), (4, 20000, 10600, 0, 40, F64, True),
    (5, 800, 770, 0, 8, F64, False), (5, 2048, 1065, 0, 24, F64, False), (5, 2048, 1536, 0, 75, F64, True),
    (5, 5917, 2958, 0, 128, F64, True), (6, 800, 80, 0, 8, F64, False), (6, 800, 600, 0, 8, F64, True),
    (6, 5917, 590, 0, 8, F64, True), (5, 648, 0, 152, 75, F64, True), (6, 648, 0, 152, 1, F64, True),
    (4, 648, 0, 152, 1, F64, False), (2, 5487, 0, 430, 8, F64, False), (6, 648, 0, 152, 1, F32, False),
    (2, 20000, 19000, 0, 1, F32, False), (3, 20000, 19000, 0, 40, F32, False), (4, 5917, 5680, 0, 8, F32, False),
    (4, 20000, 10600, 0, 40, F32, True), (5, 2048, 1960, 0, 24, F32, False), (5, 5917, 2958, 0, 45, F32, True),
    (6, 800, 770, 0, 8, F32, False), (6, 2048, 1065, 0, 24, F32, True), (6, 2048, 1960, 0, 75, F32, False),
    (6, 5917, 3136, 0, 128, F32, True)])
def test_rule_of_mixed_meshes(p, nin, npar, npml, n, mode, sf):
    assert _lib.load().f25_selftest_route(p, nin, npar, npml, n, mode) == sf


# parallelograms alone: (order, elements, pairs, mode, sum factorisation faster) as timed
@pytest.mark.parametrize("p,nin,n,mode,sf", [
    (2, 800, 160, F64, False), (2, 2048, 48, F64, True), (2, 2048, 64, F64, False), (2, 5917, 40, F64, True),
    (2, 5917, 44, F64, False), (2, 11200, 24, F64, True), (2, 20000, 24, F64, True), (2, 20000, 48, F64, False),
    (3, 20000, 128, F64, True), (2, 800, 640, F32, True), (2, 2048, 128, F32, True), (2, 5917, 20, F32, True),
    (2, 5917, 24, F32, False), (2, 11200, 23, F32, False), (2, 20000, 24, F32, False), (3, 800, 640, F32, True),
    (3, 2048, 48, F32, True), (3, 2048, 64, F32, False), (3, 5917, 8, F32, True), (3, 5917, 20, F32, False),
    (3, 5917, 44, F32, False), (3, 11200, 23, F32, False), (3, 20000, 16, F32, True), (3, 20000, 24, F32, False),
    (4, 20000, 128, F32, True)])
def test_rule_of_parallelograms(p, nin, n, mode, sf):
    assert _lib.load().f25_selftest_route(p, nin, nin, 0, n, mode) == sf


@pytest.mark.parametrize("nin,npar,n,sf", [
    (800, 800, 1, True), (800, 400, 1, False), (800, 400, 4, True), (5917, 3000, 1, True), (5917, 600, 1, False),
    (5917, 600, 4, True), (5917, 100, 8, False), (800, 80, 4, False),
    (800, 80, 45, True), (480, 0, 45, False)])
def test_rule_of_the_gradient(nin, npar, n, sf):
    for p in (2, 4, 6):
        assert _lib.load().f25_selftest_route(p, nin, npar, 0, n, _lib.F25_ROUTE_GRADIENT) == sf


def test_rule_refuses_what_there_is_not():
    route = _lib.load().f25_selftest_route
    for a in ((1, 10, 10, 0, 1, F64), (7, 10, 10, 0, 1, F64), (4, 10, 11, 0, 1, F64), (4, 10, 10, -1, 1, F64),
              (4, 10, 10, 0, 0, F64), (4, 10, 10, 0, 1, 99)):
        assert route(*a) == -1


@pytest.mark.gpu
@pytest.mark.parametrize("p,nx,nz,n,mode", [
    (2, 130, 128, 3, F64), (3, 68, 61, 9, F64), (4, 68, 61, 24, F64), (5, 68, 61, 41, F64), (6, 64, 32, 65, F64),
    (4, 130, 128, 7, F32), (5, 68, 61, 6, F32), (6, 68, 61, 5, F32)])
def test_product_of_both_kinds(p, nx, nz, n, mode):
    """Meshes large enough that each colour launches both kernels, some waves
    with a second chunk of pairs: the product on blocks alone (FP64, other
    points and sums: within a few hundred roundings), and in FP32 the FP64
    product (whose blocks' FP32 sums are known to 2e-6)."""
    import torch
    mi = handle(nx, nz, p, 37)
    g = general(mi.mesh)
    assert 0 < np.count_nonzero(g) < g.size // 2
    assert _lib.load().f25_selftest_route(p, g.size, int(g.size - np.count_nonzero(g)), 0, n, mode) == 1
    om, ky = batch(n)
    x = vectors(mi, n)
    if mode == F32:
        x32 = x.to(torch.complex64)
        got, x = product(mi, om, ky, x32, F32).to(torch.complex128), x32.to(torch.complex128)
    else:
        got = product(mi, om, ky, x)
    e = err(got, product(mi, om, ky, x, tiles=row_tiles(p)))
    print(f"p{p} {nx}x{nz} {n} pairs mode {mode}: {e:.2e}", flush=True)
    assert e < (2e-6 if mode == F32 else 1e-13)


@pytest.mark.gpu
@pytest.mark.parametrize("p,nx,nz,n,mode", [
    (2, 97, 61, 40, F64), (2, 97, 61, 41, F64), (2, 97, 61, 20, F32), (2, 97, 61, 21, F32),
    (3, 97, 61, 16, F32), (3, 97, 61, 17, F32), (2, 64, 32, 170, F32), (3, 40, 20, 300, F32)])
def test_product_both_sides_of_the_pair_rule(p, nx, nz, n, mode):
    """Parallelograms alone, on either side of the number of pairs, and batches
    whose waves take a second chunk of pairs, against blocks in FP64.  In FP32
    a value is rounded when stored, up to four times (a corner node's
    elements), each within 2^-24 of the partial sum; the blocks' sums in FP32
    are known to 2e-6."""
    import torch
    mi = handle(nx, nz, p, 0)
    sf = _lib.load().f25_selftest_route(p, nx * nz, nx * nz, 0, n, mode)
    om, ky = batch(n)
    x = vectors(mi, n)
    if mode == F32:
        x32 = x.to(torch.complex64)
        got, x = product(mi, om, ky, x32, F32).to(torch.complex128), x32.to(torch.complex128)
    else:
        got = product(mi, om, ky, x)
    e = err(got, product(mi, om, ky, x, tiles=row_tiles(p)))
    print(f"p{p} {nx}x{nz} {n} pairs mode {mode} route {sf}: {e:.2e}", flush=True)
    assert e < (1e-13 if mode == F64 else 2.4e-7 if sf else 2e-6)


@pytest.mark.gpu
@pytest.mark.parametrize("p", [2, 4, 6])
def test_gradient_of_both_kinds_with_pml(p):
    """PML elements, parallelograms and elements of general shape in one mesh:
    one triple on the general points alone, more on both, against the oracle."""
    import oracle
    from tests import test_affine as ta
    m, mod, pml, g = ta.case(p, 2)
    mi = ta.handle(p, 2)
    n = pw(p) + 1
    om, ky, f, py = ta.batch(n)
    u, lam = cf.seeded_complex(g.ndof, batch=n, seed=1), cf.seeded_complex(g.ndof, batch=n, seed=2)
    each = [oracle.grad_exact(m, mod, g, f[b], py[b], u[b], lam[b], pml)[1] for b in range(n)]
    for k in (1, n):
        assert _lib.load().f25_selftest_route(p, 16, 12, 32, k, _lib.F25_ROUTE_GRADIENT) == (k > 1)
        ref, got = sum(each[:k]), mi.gradient(om[:k], ky[:k], u[:k], lam[:k])
        for c in range(3):
            assert ta.err(got[:, c], ref[:, c]) < 1e-12, (k, c)


@pytest.mark.gpu
def test_blocks_of_both_types_in_one_pass():
    """Elements of general shape under one new model after another, each applied
    in FP64 and FP32: results of a handle that knows this model only, and the
    blocks built once a model, not once a type (their pass is most of the time:
    both products cost well under one product of each kind with a model of its
    own)."""
    import time

    import torch
    from fem25_amd.api import MeshInfo
    p = 6
    m = mixed_mesh(40, 20, p, every=2)
    assert np.count_nonzero(general(m)) == m.nelem
    models = [cf.layered_model(m, seed=s, n_anom=4, amp=0.1) for s in range(8)]
    mi = MeshInfo(m)
    om, ky = batch(2)

    def run(model, x, x32):
        mi.set_model(model)
        return [product(mi, om, ky, v, k) for v, k in ((x, F64), (x32, F32)) if v is not None]

    def best(x, x32):
        t = []
        for model in models:
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            run(model, x, x32)
            t.append(time.perf_counter() - t0)
        return min(t)

    x = vectors(mi, 2)
    x32 = x.to(torch.complex64)
    for k in (3, 5, 3):
        fresh = MeshInfo(m)
        fresh.set_model(models[k])
        want = [product(fresh, om, ky, x), product(fresh, om, ky, x32, F32)]
        assert all(torch.equal(a, b) for a, b in zip(run(models[k], x, x32), want))
        fresh.close()
    both, f64, f32 = best(x, x32), best(x, None), best(None, x32)
    print(f"per model: FP64 {f64 * 1e3:.3f} ms, FP32 {f32 * 1e3:.3f}, both {both * 1e3:.3f}", flush=True)
    assert both < 0.8 * (f64 + f32)
    mi.close()


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["folded", "clockwise", "flat"])
def test_bad_elements_are_refused_by_every_model(kind):
    """The Jacobians are checked once a mesh: a mesh that fails is refused by
    every new model, not only the first (F25_ERR_JACOBIAN)."""
    from fem25_amd.api import MeshInfo
    m = cf.structured_mesh(6, 4, 3, width=6e3, depth=4e3)
    if kind == "folded":
        m.xlocs[9] += 2.5e3
    elif kind == "clockwise":
        m.ieng[5] = m.ieng[5][[0, 3, 2, 1]]
    else:                                # no height: a parallelogram without area
        m.zlocs[m.ieng[0, 2:] - 1] = m.zlocs[m.ieng[0, 0] - 1]
    mi = MeshInfo(m)
    for seed in (1, 2, 2):
        with pytest.raises(_lib.Fem25Error) as e:
            mi.set_model(cf.layered_model(m, seed=seed))
        assert e.value.code == 2
    mi.close()


@pytest.mark.gpu
@pytest.mark.parametrize("npml", [0, 2])
def test_vectors_eight_bytes_off(npml):
    """complex128 vectors that start 8 bytes past a multiple of 16 (a caller's
    own allocation, through the C entry points): the product and the effective
    force on blocks, bit for bit, the gradient on the general points."""
    import ctypes as C

    import torch
    from fem25_amd.api import MeshInfo
    p, n = 4, 7
    m = cf.structured_mesh(10, 6, p, width=20e3, depth=12e3, npml=npml, nbielak=1 if npml else 0)
    mi = MeshInfo(m, cf.PML(rcoeff=1e-3, kappa=1.0, fcent=0.05) if npml else cf.PML())
    mi.set_model(cf.layered_model(m, seed=3, n_anom=3))
    om, ky = batch(n)
    dev = lambda t: C.c_void_p(t.data_ptr())

    def off(t):
        v = torch.empty(2 * t.numel() + 1, dtype=torch.float64, device="cuda")[1:]
        v.copy_(torch.view_as_real(t).reshape(-1))
        assert v.data_ptr() % 16 == 8
        return v

    def call(name, *a):
        _lib.check(getattr(_lib.load(), name)(mi.h, n, om.ctypes.data_as(_lib.dp), ky.ctypes.data_as(_lib.dp), *a), name)

    x = vectors(mi, n)
    xo, yo = off(x), off(x)
    torch.cuda.synchronize()
    names = ("f25_apply_batch_dev",) + (("f25_peff_batch_dev",) if npml else ())
    for name in names:
        mode = (F64,) if "apply" in name else ()
        a = (dev(xo), dev(yo))
        call(name, *mode, *a)
        got = yo.clone()
        y = torch.empty_like(x)
        for tiles in (0, row_tiles(p)):
            mi.set_apply_tiles(tiles)
            call(name, *mode, dev(x), dev(y))
            want = torch.view_as_real(y).reshape(-1)
            e = float(torch.linalg.norm(got - want) / torch.linalg.norm(want))
            assert e < 1e-13 and (tiles == 0 or e == 0.0), (name, tiles, e)
        mi.set_apply_tiles(0)
    u, lam = x.T.contiguous(), vectors(mi, n, seed=9).T.contiguous()
    g = [torch.zeros(m.nnpg, 3, dtype=torch.float64, device="cuda") for _ in range(3)]
    uo, lo = off(u), off(lam)
    torch.cuda.synchronize()
    for k, (a, b) in enumerate(((u, lam), (uo, lam), (u, lo))):
        call("f25_gradient_dev", dev(a), dev(b), dev(g[k]))
    assert torch.equal(g[1], g[2])
    assert float(torch.linalg.norm(g[1] - g[0]) / torch.linalg.norm(g[0])) < 1e-12
    mi.close()


@pytest.mark.gpu
def test_dispersive_table_is_given_back():
    """Elastic, dispersive and elastic again: the assembled values of either
    medium repeat bit for bit, and the table of every element's positions (4 (3
    NEN)^2 bytes each, 47.5 MB here) is released with the attenuation."""
    import torch
    from fem25_amd.api import MeshInfo
    m = cf.structured_mesh(64, 33, 4, npml=2, nbielak=1)
    mi = MeshInfo(m, cf.PML(rcoeff=1e-3, kappa=1.0, fcent=0.05))
    elastic = cf.layered_model(m, seed=2)
    media = [elastic, cf.with_attenuation(elastic, 300.0, 150.0, 1.0)]
    out = [None, None]
    for k in (0, 1, 0, 1, 0):
        before = torch.cuda.mem_get_info()[0]
        mi.set_model(media[k])
        if k == 0 and out[1] is not None:
            assert torch.cuda.mem_get_info()[0] - before > 40e6
        v = torch.empty(mi.nz, dtype=torch.complex128, device="cuda")
        mi.asmble_dev(b"B", 0.05, 5e-5, v)
        assert out[k] is None or torch.equal(v, out[k])
        out[k] = v
    mi.close()


@pytest.mark.gpu
def test_row_tiles_leave_the_fp32_product_alone():
    """Row tiles are the FP64 block product's: the FP32 product of
    parallelograms keeps its route, bit for bit, whatever they are."""
    import torch
    mi = handle(40, 20, 4, 0)
    om, ky = batch(9)
    x = vectors(mi, 9).to(torch.complex64)
    want = product(mi, om, ky, x, F32)
    for tiles in (1, 2, 3):
        assert torch.equal(product(mi, om, ky, x, F32, tiles), want), tiles


@pytest.mark.gpu
def test_tuner_times_the_librarys_own_choice(capsys):
    """The tuner's candidates hold 0 (no row tiles asked for), so what it calls
    best is no slower than leaving the hook alone."""
    import json

    from fem25_amd import tune_apply
    assert tune_apply.main(["--orders", "4", "6", "--nx", "40", "--nz", "20", "--nfreq", "1", "--nky", "4",
                            "--reps", "5"]) == 0
    lines = [json.loads(ln) for ln in capsys.readouterr().out.splitlines() if ln.startswith("{")]
    for order in (4, 6):
        ms = {d["row_tiles"]: d["kernel_ms_per_step"] for d in lines if d["order"] == order and "row_tiles" in d}
        best = [d for d in lines if d["order"] == order and "best_row_tiles" in d]
        assert 0 in ms and len(best) == 1
        assert best[0]["kernel_ms_per_step"] == min(ms.values()) == ms[best[0]["best_row_tiles"]]
        assert all(d["rel_diff_vs_first"] < 1e-13 for d in lines if "rel_diff_vs_first" in d)
