"""Which solver a heat step's matrix gets on a mesh: Jacobi-PCG where the mass
outweighs the stiffness at the scale of the domain (then with as many iterations
as without the mesh, give or take the rounding of another row order), multigrid
CG (at most 30 iterations of three products) where it does not."""
import ctypes

import numpy as np
import pytest
import torch

import admfem
from admfem import _lib, meshgen
from admfem.system import solve_opts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("degree,m,dt,grids", [
    (1, 60, 1e-3, False), (1, 60, 1e-1, True), (1, 60, None, True),
    (2, 30, 1e-3, False), (2, 30, 1e-1, True), (2, 30, None, True)])
def test_solver_of_a_heat_step(degree, m, dt, grids):
    print("mass rule", degree, m, dt, flush=True)
    c, e = meshgen.jittered_square(m, seed=m)
    mesh = admfem.Mesh(c, e, degree=degree, zero_based=True)
    bd = admfem.bcnode(mesh)
    one = torch.ones(mesh.ngauss, dtype=torch.float64, device="cuda")
    A = admfem.compute_fem_laplace_matrix1(one, mesh)
    if dt is not None:
        A = admfem.compute_fem_mass_matrix1(one, mesh) + A * dt
    B, r = admfem.impose_Dirichlet_boundary_conditions(
        A, torch.ones(mesh.ndof, dtype=torch.float64, device="cuda"), bd, np.zeros(len(bd)))
    ind, vv, r = B.indices.contiguous(), B.values.detach().contiguous(), r.detach().contiguous()
    o, it = solve_opts("fp64", 1e-12, 100000), []
    for h in (mesh.handle, None):
        st, x = _lib.SolveStats(), torch.empty_like(r)
        _lib.check(_lib.lib().admfem_sparse_solve_on(
            h, _lib.ptr(ind), _lib.ptr(vv), ind.shape[0], mesh.ndof, _lib.ptr(r), _lib.ptr(x),
            ctypes.byref(o), ctypes.byref(st), _lib.stream_ptr()))
        it.append(st.iterations)
    print(it, flush=True)
    if grids:
        assert it[0] <= 3 * 30 and it[0] % 3 == 0 and it[0] < it[1]
    else:
        assert abs(it[0] - it[1]) <= 2
