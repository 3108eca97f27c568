"""Solves that multigrid CG cannot do and Jacobi-PCG can end in Jacobi-PCG's
result: a coefficient of 1 and 1e60 in the fields of a checkerboard, more than the
FP32 grids hold.  The diagonally scaled matrix is harmless, and Jacobi-PCG takes as
many iterations as for any such pattern."""
import numpy as np
import pytest
import torch

import admfem
from admfem import meshgen

pytestmark = pytest.mark.gpu


def board(m):
    c, e = meshgen.jittered_square(m, seed=m)
    mesh = admfem.Mesh(c, e, zero_based=True)
    g = admfem.gauss_nodes(mesh)
    black = (np.floor(8 * g[:, 0]) + np.floor(8 * g[:, 1])) % 2 > 0
    kap = torch.tensor(np.where(black, 1e60, 1.0), device="cuda")
    f = torch.tensor(np.random.default_rng(m).uniform(-1, 1, mesh.ngauss), device="cuda")
    return mesh, kap, f, admfem.bcnode(mesh)


def test_system_solve():
    mesh, kap, f, bd = board(64)
    S = admfem.DirichletSystem(mesh, bd)
    S.assemble(kappa=kap, f=f)
    print("fallback, system", flush=True)
    x, st = S.solve(rtol=1e-10, max_iter=5000)
    assert st["status"] == 0 and st["rel_residual"] <= 1e-10
    A, b = S.csr()
    r = b - A @ x.cpu().numpy()
    assert np.linalg.norm(r) <= 2e-10 * np.linalg.norm(b)
    S.assemble(kappa=torch.ones_like(kap), f=f)  # the next matrix is multigrid CG's again
    _, st = S.solve(rtol=1e-10)
    assert st["status"] == 0 and st["iterations"] < 60


def test_operators():
    mesh, kap, f, bd = board(40)
    K = admfem.compute_fem_laplace_matrix1(kap, mesh)
    F = admfem.compute_fem_source_term1(f, mesh)
    B, r = admfem.impose_Dirichlet_boundary_conditions(K, F, bd, np.zeros(bd.size))
    print("fallback, operators", flush=True)
    x = admfem.solve(B, r, rtol=1e-10, max_iter=5000)
    plain = admfem.solve(admfem.SparseTensor(B.indices, B.values, B.n), r, rtol=1e-10,
                         max_iter=5000)
    assert ((x - plain).norm() / plain.norm()).item() < 1e-8
