"""A solve whose solution overwrites its right-hand side, restarted and checked
several times on the way (check_every 1: the host looks after every iteration,
and the true residual needs the right-hand side each time).

Tolerance: both solves reach a relative residual of 1e-12 at a condition number
below 5000 (P1 24^2): 1e-8 between them."""
import ctypes

import numpy as np
import pytest
import torch

import admfem
from admfem import _lib
from admfem.system import solve_opts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("every", [0, 1])
def test_solution_over_rhs(every):
    m = 24
    mesh = admfem.Mesh(m, m, 1.0 / m)
    bd = admfem.bcnode(mesh)
    K = admfem.compute_fem_laplace_matrix1(
        torch.ones(mesh.ngauss, dtype=torch.float64, device="cuda"), mesh)
    g = torch.Generator(device="cuda").manual_seed(1)
    rhs = torch.rand(mesh.ndof, generator=g, dtype=torch.float64, device="cuda")
    B, r = admfem.impose_Dirichlet_boundary_conditions(K, rhs, bd, np.zeros(len(bd)))
    ind, vv, r = B.indices.contiguous(), B.values.detach().contiguous(), r.detach().contiguous()
    o = solve_opts("fp64", 1e-12, 100000)
    o.check_every = every

    def solve(b, x):
        _lib.check(_lib.lib().admfem_sparse_solve_on(
            mesh.handle, _lib.ptr(ind), _lib.ptr(vv), ind.shape[0], mesh.ndof, _lib.ptr(b),
            _lib.ptr(x), ctypes.byref(o), None, _lib.stream_ptr()))
        return x
    want = solve(r, torch.empty_like(r))
    both = r.clone()
    got = solve(both, both)
    assert torch.linalg.norm(got - want) <= 1e-8 * torch.linalg.norm(want)
