"""Field maps into buffers of other forms: gradients at an address that is not a
multiple of 16, the Laplace term's gradient in nu over nu itself, either of its
gradients alone."""
import numpy as np
import pytest
import torch

import admfem
from admfem import _lib, meshgen

pytestmark = pytest.mark.gpu


def empty(n, off=0):
    return torch.full((n + off,), float("nan"), dtype=torch.float64, device="cuda")[off:]


@pytest.mark.parametrize("m,order", [(1, 2), (11, 2), (12, 4), (16, 1), (40, 2)])
def test_forms_agree(m, order):
    print("field forms", m, order, flush=True)
    c, e = meshgen.jittered_square(m, seed=m)
    gm = admfem.Mesh(c, e, order=order, zero_based=True)
    g = torch.Generator(device="cuda").manual_seed(m)
    r = lambda n: torch.rand(n, generator=g, dtype=torch.float64, device="cuda")
    u, go, nu = r(gm.ndof), r(gm.ndof), r(gm.ngauss)
    L, p, st = _lib.lib(), _lib.ptr, _lib.stream_ptr()
    a, b = empty(2 * gm.ngauss), empty(2 * gm.ngauss, 1)
    assert a.data_ptr() % 16 == 0 and b.data_ptr() % 16 == 8
    for o in (a, b):
        _lib.check(L.admfem_fem_grad(gm.handle, p(u), p(o), st))
    assert torch.equal(a, b)
    gu, gn = empty(gm.ndof), empty(gm.ngauss)
    gu1, gn1, inplace = empty(gm.ndof), empty(gm.ngauss), nu.clone()
    work = empty(3 * gm.nelem)

    def grad(n, x, y):
        _lib.check(L.admfem_fem_laplace_term_grad_on(gm.handle, p(go), p(u), p(n), p(x), p(y),
                                                     p(work), st))
    grad(nu, gu, gn)
    grad(inplace, gu1, inplace)
    assert torch.equal(gu, gu1) and torch.equal(gn, inplace)
    grad(nu, None, gn1)
    gu1.fill_(float("nan"))
    grad(nu, gu1, None)
    # (other kernels, which may contract differently: a few roundings)
    for x, y in ((gu, gu1), (gn, gn1)):
        assert torch.allclose(x, y, rtol=1e-13, atol=1e-13 * float(x.abs().max()))
