"""Solves whose matrix or right-hand side is far outside FP32's range: with A
scaled by 2^a and b by 2^c every FP64 quantity of the solve scales by a power
of two, so the solution is the unscaled one times 2^(c - a), bit for bit, after
as many iterations; the same for the gradient chain and for serving requests."""
import numpy as np
import pytest
import torch

import admfem
from admfem import meshgen
from admfem.server import Server

pytestmark = pytest.mark.gpu

POWERS = [(-130, 0), (130, 0), (0, -130), (0, 130), (90, -90), (-90, 130), (0, -300), (-100, 100)]


def problem(m, degree):
    c, e = meshgen.jittered_square(m, seed=m)
    mesh = admfem.Mesh(c, e, degree=degree, zero_based=True)
    rng = np.random.default_rng(m)
    kap = torch.tensor(np.exp(0.5 * rng.standard_normal(mesh.ngauss)), device="cuda")
    f = torch.tensor(rng.uniform(-1, 1, mesh.ngauss), device="cuda")
    bd = admfem.bcnode(mesh)
    obs = rng.choice(np.setdiff1d(np.arange(mesh.ndof), bd - 1), 20, replace=False)
    return mesh, kap, f, bd, obs.astype(np.int32)


@pytest.mark.parametrize("m,degree", [(20, 1), (90, 1), (24, 2)])
def test_fused_solves_scale(m, degree):
    mesh, kap, f, bd, obs = problem(m, degree)
    S = admfem.DirichletSystem(mesh, bd)
    zero = np.zeros(obs.size)
    for prec in ("fp64", "mixed"):
        def go(a, c):
            return S.forward_adjoint(obs, zero, precision=prec, rtol=1e-12, kappa=kap * 2.0 ** a,
                                     f=f * 2.0 ** c)
        ref = go(0, 0)
        for a, c in POWERS:
            print("range", m, degree, prec, a, c, flush=True)
            out = go(a, c)
            assert [s["iterations"] for s in out["stats"]] == \
                [s["iterations"] for s in ref["stats"]]
            # u and dL/du scale by 2^(c - a), lambda by 2^(c - 2a), the gradient by both
            assert torch.equal(out["u"], ref["u"] * 2.0 ** (c - a))
            assert torch.equal(out["lam"], ref["lam"] * 2.0 ** (c - 2 * a))
            assert torch.equal(out["grad_kappa"], ref["grad_kappa"] * 2.0 ** (2 * c - 3 * a))


@pytest.mark.parametrize("m,degree", [(40, 1), (24, 2)])
def test_sparse_solve_on_a_mesh_scales(m, degree):
    mesh, kap, f, bd, _ = problem(m, degree)
    K = admfem.compute_fem_laplace_matrix1(kap, mesh)
    F = admfem.compute_fem_source_term1(f, mesh)
    B, r = admfem.impose_Dirichlet_boundary_conditions(K, F, bd, np.zeros(bd.size))
    ref = admfem.solve(B, r)
    for a, c in POWERS:
        print("range, operators", m, degree, a, c, flush=True)
        assert torch.equal(admfem.solve(B * 2.0 ** a, r * 2.0 ** c), ref * 2.0 ** (c - a))


def test_serving_requests_scale():
    out = {}
    for k, (a, c) in enumerate([(0, 0)] + POWERS):
        print("range, serving", a, c, flush=True)
        sv = Server(1 << 30, rtol=1e-10)
        ids = []
        for m, degree in ((20, 1), (90, 1), (24, 2)):
            mesh, kap, f, bd, obs = problem(m, degree)
            t = sv.add_topology(admfem.DirichletSystem(mesh, bd))
            ids.append(sv.submit(t, kappa=kap * 2.0 ** a, f=f * 2.0 ** c,
                                 obs_idx=torch.tensor(obs), obs_val=torch.zeros(obs.size)))
        sv.run()
        res = [sv.result(i) for i in ids]
        out = out or {i: r for i, r in enumerate(res)}
        for i, r in enumerate(res):
            assert r["status"] == 0
            assert (r["iters_fwd"], r["iters_adj"]) == (out[i]["iters_fwd"], out[i]["iters_adj"])
            np.testing.assert_array_equal(r["u"], out[i]["u"] * 2.0 ** (c - a))
            np.testing.assert_array_equal(r["grad"], out[i]["grad"] * 2.0 ** (2 * c - 3 * a))
        sv.close()
