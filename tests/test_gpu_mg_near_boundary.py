"""Systems whose rows nearly all neighbour Dirichlet rows are Jacobi-PCG's, by the
fused path, by the operators' and in the engine (some 11 + 7 / F iterations: about 22
where two thirds or three quarters of a row's neighbours are Dirichlet rows, against
33 products of multigrid CG); wider ones are multigrid CG's (multiples of three
products, 11 or 12 iterations).  Solutions are the direct solver's."""
import numpy as np
import pytest
import scipy.sparse.linalg as spla
import torch

import admfem
from admfem import meshgen
from admfem.server import Server

pytestmark = pytest.mark.gpu


def strip(length, width, degree=1):
    c, e = meshgen.rectangle(length, width, 0.01)
    p = np.random.default_rng(1).permutation(c.shape[0])
    out = np.empty_like(c)
    out[p] = c
    return admfem.Mesh(out, p[e], degree=degree, zero_based=True)


@pytest.mark.parametrize("length,width,degree,grids", [
    (2000, 2, 1, False), (2000, 6, 1, True), (200, 3, 1, True), (3000, 1, 2, False),
    (1000, 3, 2, True)])
def test_solver_of_a_strip(length, width, degree, grids):
    mesh = strip(length, width, degree)
    bd = admfem.bcnode(mesh)
    S = admfem.DirichletSystem(mesh, bd)
    rng = np.random.default_rng(2)
    kap = torch.tensor(np.exp(0.3 * rng.standard_normal(mesh.ngauss)), device="cuda")
    f = torch.tensor(rng.uniform(0.5, 1, mesh.ngauss), device="cuda")
    S.assemble(kappa=kap, f=f)
    x, st = S.solve(rtol=1e-10)
    A, b = S.csr()
    ref = spla.spsolve(A.tocsc(), b)
    print("strip", length, width, degree, st, flush=True)
    # (the condition number of these systems is below 100)
    assert np.linalg.norm(x.cpu().numpy() - ref) < 1e-8 * np.linalg.norm(ref)
    it = st["iterations"]
    assert (it % 3 == 0 and it <= 3 * 16) if grids else it <= 26
    K = admfem.compute_fem_laplace_matrix1(kap, mesh)
    F = admfem.compute_fem_source_term1(f, mesh)
    B, r = admfem.impose_Dirichlet_boundary_conditions(K, F, bd, np.zeros(bd.size))
    u = admfem.solve(B, r, rtol=1e-10).cpu().numpy()
    assert np.linalg.norm(u - ref) < 1e-8 * np.linalg.norm(ref)
    sv = Server(1 << 30, rtol=1e-10)
    obs = np.setdiff1d(np.arange(mesh.ndof), bd - 1)[::50].astype(np.int32)
    i = sv.submit(sv.add_topology(S), kappa=kap, f=f, obs_idx=torch.tensor(obs),
                  obs_val=torch.zeros(obs.size))
    sv.run(timeout=60)
    r = sv.result(i)
    assert r["status"] == 0
    assert np.linalg.norm(r["u"] - ref) < 1e-8 * np.linalg.norm(ref)
    both = S.forward_adjoint(obs, np.zeros(obs.size), rtol=1e-10, kappa=kap, f=f)["stats"]
    assert r["iters_fwd"] % 3 == 0 if grids else r["iters_fwd"] <= 28
    print(r["iters_fwd"], [s["iterations"] for s in both], flush=True)


def test_jacobi_time():
    """A solve on a strip of 20000 x 3 quads takes what Jacobi-PCG does, which solves
    the same matrix where its mesh is not known (multigrid CG 1.7 times as long)."""
    mesh = strip(20000, 3)
    bd = admfem.bcnode(mesh)
    one = torch.ones(mesh.ngauss, dtype=torch.float64, device="cuda")
    S = admfem.DirichletSystem(mesh, bd)
    S.assemble(kappa=one, f=one)
    A, b = S.csr()
    A = A.tocoo()
    B = admfem.SparseTensor(np.stack([A.row, A.col], 1), A.data, S.n)
    b = torch.tensor(b, device="cuda")

    def shortest(f):
        t = []
        for _ in range(8):
            e0, e1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            e0.record()
            f()
            e1.record()
            e1.synchronize()
            t.append(e0.elapsed_time(e1))
        return min(t)
    t0 = shortest(lambda: admfem.solve(B, b, rtol=1e-10))
    t = shortest(lambda: S.solve(b, rtol=1e-10))
    print("strip, with its mesh and without", t, t0, flush=True)
    assert t < 1.25 * t0
