"""Which solver short heat steps get in the fused path, on both sides of the lines
for matrices with grids above the tail and for P2: Jacobi-PCG takes as many
iterations as it does for the same matrix where its mesh is not known, give or take
the rounding of another row order; multigrid CG 8 to 12 of three products."""
import ctypes

import numpy as np
import pytest
import torch

import admfem
from admfem import _lib, meshgen
from admfem.system import solve_opts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("degree,m,dt,grids", [
    (1, 40, 1e-5, False), (1, 40, 3e-3, True), (1, 400, 5e-6, False), (1, 400, 5e-5, True),
    (2, 20, 1e-6, True), (2, 100, 5e-7, False), (2, 100, 1e-5, True)])
def test_solver_of_a_short_heat_step(degree, m, dt, grids):
    c, e = meshgen.jittered_square(m, seed=m)
    mesh = admfem.Mesh(c, e, degree=degree, zero_based=True)
    S = admfem.DirichletSystem(mesh, admfem.bcnode(mesh))
    rng = np.random.default_rng(m)
    one = torch.ones(mesh.ngauss, dtype=torch.float64, device="cuda")
    up = torch.tensor(rng.standard_normal(mesh.ndof), device="cuda")
    S.assemble(kappa=one, f=one, u_prev=up, lap_coef=dt, mass_coef=1.0, src_coef=dt)
    x, st = S.solve(rtol=1e-10)
    A, b = S.csr()
    A = A.tocoo()
    ind = torch.tensor(np.stack([A.row, A.col], 1).astype(np.int64), device="cuda")
    vv, b, y = (torch.tensor(v, device="cuda") for v in (A.data, b, b))
    o, sp = solve_opts("fp64", 1e-10, 100000), _lib.SolveStats()
    _lib.check(_lib.lib().admfem_sparse_solve(
        _lib.ptr(ind), _lib.ptr(vv), ind.shape[0], mesh.ndof, _lib.ptr(b), _lib.ptr(y),
        ctypes.byref(o), ctypes.byref(sp), _lib.stream_ptr()))
    print("mass lines", degree, m, dt, st["iterations"], sp.iterations, flush=True)
    if grids:
        assert st["iterations"] % 3 == 0 and 21 <= st["iterations"] <= 36
    else:
        assert abs(st["iterations"] - sp.iterations) <= 1
    # (condition numbers below 100)
    assert ((x - y).norm() / y.norm()).item() < 1e-8
