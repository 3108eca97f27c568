"""The maps to the nodes in two passes (elements' terms through scratch, then
sums per node) against the oracle, around the sizes where fem_grad's
transpose changes over, at block edges and at the smallest meshes, with every
quadrature rule; with scratch from the caller and without."""
import numpy as np
import pytest
import torch

import admfem
from admfem import _lib, meshgen
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# sums of at most 61 terms of 64-bit products, relative to the largest entry:
# 61 terms x 6 points x a few roundings of 1.1e-16 each
TOL = 1e-12


def rel(a, b):
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)


@pytest.mark.parametrize("degree,m,order", [
    (1, 1, 2), (1, 8, 2), (1, 8, 4), (1, 8, 1), (1, 11, 2), (1, 315, 2), (1, 316, 2), (1, 316, 4),
    (2, 1, 4), (2, 8, 4), (2, 8, 2), (2, 11, 1), (2, 40, 4)])
def test_two_pass_maps_match_oracle(degree, m, order):
    print("two-pass maps", degree, m, order, flush=True)
    c, e = meshgen.jittered_square(m, seed=m)
    gm = admfem.Mesh(c, e, order=order, degree=degree, zero_based=True)
    om = O.OracleMesh(c, e, order, degree)
    rng = np.random.default_rng(m)
    u, go = rng.standard_normal(gm.ndof), rng.standard_normal(gm.ndof)
    nu = rng.random(gm.ngauss) + 0.5
    g2 = rng.standard_normal((gm.ngauss, 2))
    d = lambda a: torch.tensor(a, device="cuda")
    L = _lib.lib()
    want_k, want_g = om.laplace_term(u, nu), om.fem_grad_backward(g2)
    gn0, gu0 = om.laplace_term_backward(u, nu, go)
    for scratch in (True, False):
        work = d(np.full(gm.elem_ndof * gm.nelem, np.nan)) if scratch else None
        du, dnu, dgo, dg2 = d(u), d(nu), d(go), d(g2)
        k, g, gu, gn = (torch.full((n,), np.nan, dtype=torch.float64, device="cuda")
                        for n in (gm.ndof, gm.ndof, gm.ndof, gm.ngauss))
        _lib.check(L.admfem_fem_laplace_term_on(gm.handle, _lib.ptr(du), _lib.ptr(dnu),
                                                _lib.ptr(k), _lib.ptr(work), _lib.stream_ptr()))
        _lib.check(L.admfem_fem_grad_grad_on(gm.handle, _lib.ptr(dg2), _lib.ptr(g),
                                             _lib.ptr(work), _lib.stream_ptr()))
        _lib.check(L.admfem_fem_laplace_term_grad_on(
            gm.handle, _lib.ptr(dgo), _lib.ptr(du), _lib.ptr(dnu), _lib.ptr(gu), _lib.ptr(gn),
            _lib.ptr(work), _lib.stream_ptr()))
        assert rel(k.cpu().numpy(), want_k) < TOL
        assert rel(g.cpu().numpy(), want_g) < TOL
        assert rel(gu.cpu().numpy(), gu0) < TOL
        assert rel(gn.cpu().numpy(), gn0) < TOL
