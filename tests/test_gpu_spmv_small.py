"""SparseTensor @ x on both sides of the number of rows where its accumulation
changes, against scipy, with its first and second derivatives; and with few rows
it takes no longer than twice what its index_add_ does (a sort takes four times
as long)."""
import time

import numpy as np
import pytest
import torch

import admfem
from admfem import meshgen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 1024, 1025])
def test_product_and_derivatives(n):
    rng = np.random.default_rng(n)
    nnz = 12 * n
    ind = rng.integers(0, n, (nnz, 2))
    v = torch.tensor(rng.standard_normal(nnz), device="cuda", requires_grad=True)
    x = torch.tensor(rng.standard_normal(n), device="cuda", requires_grad=True)
    g = torch.tensor(rng.standard_normal(n), device="cuda", requires_grad=True)
    A = admfem.SparseTensor(ind, v, n)
    print("product", n, flush=True)
    y = A @ x
    gv, gx = torch.autograd.grad(y, [v, x], g, create_graph=True)
    h = torch.tensor(rng.standard_normal(n), device="cuda")
    (gxv,) = torch.autograd.grad(gx, [v], h, retain_graph=True)  # second derivative
    B = A.to_scipy()
    xn, gn, hn = (t.detach().cpu().numpy() for t in (x, g, h))
    i, j = ind.T
    # sums of some 12 (n = 1: 12) products of order 1: a few ulps of 12
    for a, b in ((y, B @ xn), (gx, B.T @ gn), (gv, gn[i] * xn[j]), (gxv, gn[i] * hn[j])):
        assert np.abs(a.detach().cpu().numpy() - b).max() < 1e-13 * 12


def shortest(f):
    out = []
    for _ in range(30):
        torch.cuda.synchronize()
        t = time.perf_counter()
        f()
        torch.cuda.synchronize()
        out.append(time.perf_counter() - t)
    return min(out)


@pytest.mark.parametrize("degree,m", [(1, 8), (1, 28), (2, 8)])
def test_few_rows_take_no_sort(degree, m):
    c, e = meshgen.jittered_square(m, seed=m)
    mesh = admfem.Mesh(c, e, degree=degree, zero_based=True)
    M = admfem.compute_fem_mass_matrix1(
        torch.ones(mesh.ngauss, dtype=torch.float64, device="cuda"), mesh)
    x = torch.randn(mesh.ndof, dtype=torch.float64, device="cuda")
    i, j = M.indices[:, 0], M.indices[:, 1]
    t = shortest(lambda: M @ x)
    t0 = shortest(lambda: torch.zeros_like(x).index_add_(0, i, M.values * x[j]))
    print("product, few rows", degree, m, t0, t, flush=True)
    assert t < 2 * t0
