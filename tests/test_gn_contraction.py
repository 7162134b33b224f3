"""GNMFREE's contraction at the edges of its kernels' tiles: observation counts
around the 512 of a staged tile and the 16 of a column's lanes, a Jacobian
without observations, 861 columns (not a multiple of 64), and batches of so
few observations that the columns run over all Jacobians (k_gn_z)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from tests.helpers import mesh_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nobs", [[1, 2], [15, 16, 17, 33], [512], [0, 513, 63], [1030, 64, 5]])
def test_contraction(nobs):
    from fem25_amd.api import MeshInfo
    m, mod, pml = mesh_case("c1")
    mi = MeshInfo(m, pml)
    mi.set_model(mod)
    inv = mi.inv_setup(b"PP")
    assert inv.nnpgl == 861
    rng = np.random.default_rng(len(nobs))
    nobs = np.array(nobs, np.int32)
    tot = int(nobs.sum()) * inv.nnpgl
    jac = (rng.standard_normal(tot) + 1j * rng.standard_normal(tot)).astype(np.complex64)
    alpha, p = rng.uniform(0.5, 2.0, size=nobs.size), rng.standard_normal(inv.na35)
    z0 = rng.standard_normal(inv.na35)
    ref = z0 + oracle.gnmfree(nobs, alpha, inv.nnpgl, inv.mygrad, inv.na35, jac, p)
    for _ in range(2):   # the second call on the scratch the first one left
        z = mi.gnmfree(nobs, alpha, jac, p, z0.copy())
        assert np.linalg.norm(z - ref) < 1e-12 * np.linalg.norm(ref)
    mi.close()
