"""The multigrid-preconditioned solves against the CPU oracle's direct solve
and gradient chain, at the sizes and forms where the path can go wrong: just
above the size it starts at, odd and even grids, several grid levels, long
thin domains, partial (one-sided) Dirichlet boundaries, a hole, clustered
nodes (which stay with Jacobi-PCG), heat steps on both sides of the
mass-dominance rule, rough coefficients, P2.

Tolerance: a solve at relative residual rtol has a relative error of at most
cond(A) rtol; the worst condition number here is about 4e5 (the 240 x 12 strip
with one Dirichlet side, P2 at 101), so 1e-13 keeps u and the gradient well
below 1e-7; the bound asserted is the suite's FP64 bar, 1e-9, which the
smooth right-hand sides leave a factor of 100 to."""
import numpy as np
import pytest
import torch

import admfem
from admfem import meshgen
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def grid(mx, my, hx, hy, seed, keep=None, warp=None):
    """mx x my quads of size hx x hy, jittered and permuted; ``keep`` drops
    quads, ``warp`` maps the points."""
    c, e = meshgen.rectangle(mx, my, 1.0)
    rng = np.random.default_rng(seed)
    e = e.copy()
    if keep is not None:
        q = np.arange(e.shape[0]) // 2
        e = e[keep(q % mx, q // mx)]
        used = np.unique(e)
        new = -np.ones(c.shape[0], dtype=np.int64)
        new[used] = np.arange(used.size)
        c, e = c[used], new[e]
    c = c * [hx, hy]
    if warp is not None:
        c = warp(c)
    else:
        c = c + rng.uniform(-0.15, 0.15, c.shape) * [hx, hy]
    p = rng.permutation(c.shape[0])
    out = np.empty_like(c)
    out[p] = c
    return out, p[e]


CASES = {
    "square64": dict(g=(64, 64, 1 / 64, 1 / 64)),
    "square65x67": dict(g=(65, 67, 1 / 66, 1 / 66)),
    "square150": dict(g=(150, 150, 1 / 150, 1 / 150)),
    "strip": dict(g=(600, 12, 1 / 100, 1 / 100)),
    "tall": dict(g=(9, 500, 0.02, 0.01)),
    "one side": dict(g=(80, 60, 1 / 80, 1 / 80), bd=lambda c: c[:, 0] < c[:, 0].min() + 0.004),
    "hole": dict(g=(90, 90, 1 / 90, 1 / 90),
                 keep=lambda i, j: (abs(i - 40) > 15) | (abs(j - 50) > 11)),
    "clustered": dict(g=(80, 80, 1 / 80, 1 / 80), warp=lambda c: c ** 3),
    "rough": dict(g=(100, 100, 1 / 100, 1 / 100), rough=True),
    "heat 1e-2": dict(g=(100, 100, 1 / 100, 1 / 100), dt=1e-2),
    "heat 1e-5": dict(g=(100, 100, 1 / 100, 1 / 100), dt=1e-5),
    "P2": dict(g=(40, 41, 1 / 40, 1 / 40), degree=2),
    "P2 heat": dict(g=(40, 40, 1 / 40, 1 / 40), degree=2, dt=1e-3),
}


@pytest.mark.parametrize("name", list(CASES))
def test_multigrid_solve_matches_oracle(name):
    k = CASES[name]
    print(name, flush=True)
    degree, dt = k.get("degree", 1), k.get("dt")
    c, e = grid(*k["g"], seed=3, keep=k.get("keep"), warp=k.get("warp"))
    gm = admfem.Mesh(c, e, degree=degree, zero_based=True)
    om = O.OracleMesh(c, e) if degree == 1 else O.OracleMesh(c, e, degree=2)
    rng = np.random.default_rng(4)
    kap = np.exp(rng.standard_normal(om.ngauss) if k.get("rough")
                 else meshgen.grf(np.stack([om.gx, om.gy], 1), 5, ell=0.3))
    f = rng.uniform(-1, 1, om.ngauss)
    bd = np.flatnonzero(k["bd"](c)) + 1 if "bd" in k else om.bcnode()
    inner = np.setdiff1d(np.arange(gm.ndof), bd - 1)
    obs = rng.choice(inner, 50, replace=False)
    S = admfem.DirichletSystem(gm, bd)
    more, okw = {}, {}
    if dt:
        up = rng.standard_normal(gm.ndof)
        more = dict(u_prev=up, lap_coef=dt, mass_coef=1.0, src_coef=dt)
        okw = dict(dt=dt, u_prev=up)

    def dl(u):
        g = np.zeros_like(u)
        g[obs] = 2 * u[obs]
        return g
    ref = O.forward_adjoint(om, kap, f, bd, np.zeros(bd.size), dl, **okw)
    for prec in ("fp64", "mixed"):
        out = S.forward_adjoint(obs, np.zeros(obs.size), precision=prec, rtol=1e-13, kappa=kap,
                                f=f, **more)
        print(prec, out["stats"], flush=True)
        for a, b in (("u", "u"), ("grad_kappa", "grad_kappa")):
            r = np.linalg.norm(out[a].cpu().numpy() - ref[b]) / np.linalg.norm(ref[b])
            assert r < 1e-9, (a, r)


def test_multigrid_reports_matrices_it_cannot_solve():
    """A negative coefficient (not SPD), a NaN and too few iterations are
    errors, and the system solves again afterwards."""
    c, e = meshgen.jittered_square(70, seed=1)
    gm = admfem.Mesh(c, e, zero_based=True)
    S = admfem.DirichletSystem(gm, admfem.bcnode(gm))
    one = torch.ones(gm.ngauss, dtype=torch.float64, device="cuda")
    bad = one.clone()
    bad[100] = float("nan")
    for kap, opt, code in ((-one, {}, admfem._lib.ERR_BREAKDOWN), (bad, {}, admfem._lib.ERR_NAN),
                           (one, dict(max_iter=3), admfem._lib.ERR_NOT_CONVERGED)):
        S.assemble(kappa=kap, f=one)
        with pytest.raises(admfem.AdmfemError) as ei:
            S.solve(rtol=1e-10, **opt)
        assert ei.value.code == code
    S.assemble(kappa=one, f=one)
    x0, st = S.solve(rtol=1e-12)
    assert st["rel_residual"] <= 1e-12
    x1, _ = S.solve(rtol=1e-12, check_every=1)
    assert torch.equal(x0, x1)  # however often the host looks


@pytest.mark.parametrize("degree,m", [(1, 70), (2, 36)])
def test_operator_chain_with_grids_matches_oracle(degree, m):
    """A \\ rhs for matrices the mesh's operators made (solved on grids laid
    over the mesh), for the same matrix without its mesh, and for another
    mesh's matrix of the same pattern afterwards (its own grids): u and the
    gradients against the oracle's chain, tolerance as above."""
    for seed in (1, 2):
        c, e = meshgen.jittered_square(m, seed=7)
        if seed == 2:  # same connectivity, other node positions
            c = c * [1.0, 0.5]
        om = O.OracleMesh(c, e) if degree == 1 else O.OracleMesh(c, e, degree=2)
        gm = admfem.Mesh(c, e, degree=degree, zero_based=True)
        rng = np.random.default_rng(seed)
        kap, f = np.exp(0.5 * rng.standard_normal(om.ngauss)), rng.uniform(-1, 1, om.ngauss)
        bd = om.bcnode()
        bv = rng.standard_normal(bd.size)
        w = rng.standard_normal(gm.ndof)
        ref = O.forward_adjoint(om, kap, f, bd, bv, lambda u: w)
        for with_mesh in (True, False):
            k = torch.tensor(kap, device="cuda", requires_grad=True)
            K = admfem.compute_fem_laplace_matrix1(k, gm)
            F = admfem.compute_fem_source_term1(torch.tensor(f, device="cuda"), gm)
            A, r = admfem.impose_Dirichlet_boundary_conditions(K, F, bd, bv)
            assert A.mesh is gm and (2.0 * A).mesh is gm and (A + A).mesh is gm
            if not with_mesh:
                A = admfem.SparseTensor(A.indices, A.values, A.n)
                assert A.mesh is None
            u = admfem.solve(A, r, rtol=1e-13)
            (u * torch.tensor(w, device="cuda")).sum().backward()
            for a, b in ((u.detach(), ref["u"]), (k.grad, ref["grad_kappa"])):
                d = np.linalg.norm(a.cpu().numpy() - b) / np.linalg.norm(b)
                print(degree, m, seed, with_mesh, d, flush=True)
                assert d < 1e-9


def test_serving_batches_multigrid_and_jacobi_requests():
    """Requests on meshes on both sides of the multigrid path's smallest size
    and with one, two and three grids above the tail, Poisson and heat, host
    inputs with other coordinates than the topology's, and P2, all in one
    batch: each against the oracle, and bit-identical when served alone or in
    rounds cut short by a timeout."""
    from admfem.server import Server
    rng = np.random.default_rng(0)
    topos = []
    for m, degree in ((30, 1), (63, 1), (64, 1), (130, 1), (260, 1), (40, 2)):
        c, e = meshgen.jittered_square(m, seed=m)
        om = O.OracleMesh(c, e) if degree == 1 else O.OracleMesh(c, e, degree=2)
        gm = admfem.Mesh(c, e, degree=degree, zero_based=True)
        topos.append((m, c, e, om, admfem.DirichletSystem(gm, admfem.bcnode(gm))))
    reqs = []
    for k, (m, c, e, om, S) in enumerate(topos):
        for heat in (False, True):
            c2 = c + rng.uniform(-0.02 / m, 0.02 / m, c.shape) if not heat else None
            o2 = O.OracleMesh(c2, e) if c2 is not None and om.ndof == om.nnode else om
            if o2 is om:
                c2 = None
            bd = om.bcnode()
            obs = rng.choice(np.setdiff1d(np.arange(S.n), bd - 1), 30, replace=False)
            P = dict(kappa=np.exp(0.3 * rng.standard_normal(om.ngauss)),
                     f=rng.uniform(-1, 1, om.ngauss), obs_idx=obs.astype(np.int32),
                     obs_val=np.zeros(30))
            kw = dict(kind="poisson")
            if heat:
                P["u_prev"] = rng.standard_normal(S.n)
                kw = dict(kind="heat", dt=1e-3)

            def dl(u, obs=obs):
                g = np.zeros_like(u)
                g[obs] = 2 * u[obs]
                return g
            ref = O.forward_adjoint(o2, P["kappa"], P["f"], bd, np.zeros(bd.size), dl,
                                    **(dict(dt=1e-3, u_prev=P["u_prev"]) if heat else {}))
            reqs.append((k, dict(P, coords=c2, **kw), ref))

    def serve(which, slices=None):
        sv = Server(2 << 30, rtol=1e-11)
        t = [sv.add_topology(S) for *_, S in topos]
        ids = [sv.submit(t[reqs[i][0]], **reqs[i][1]) for i in which]
        if slices:
            for k in range(200):
                sv.run(timeout=slices * (k + 1))
        sv.run()
        return [sv.result(i) for i in ids]
    mix = serve(range(len(reqs)))
    for r, (k, P, ref) in zip(mix, reqs):
        assert r["status"] == 0
        eu = np.linalg.norm(r["u"] - ref["u"]) / np.linalg.norm(ref["u"])
        eg = np.linalg.norm(r["grad"] - ref["grad_kappa"]) / np.linalg.norm(ref["grad_kappa"])
        print(topos[k][0], P["kind"], r["iters_fwd"], r["iters_adj"], eu, eg, flush=True)
        assert eu < 1e-8 and eg < 1e-8
    cut = serve(range(len(reqs)), slices=2e-4)
    alone = [serve([i])[0] for i in (2, 7, 8)]
    for a, b in list(zip(cut, mix)) + list(zip(alone, [mix[2], mix[7], mix[8]])):
        assert a["status"] == 0
        np.testing.assert_array_equal(a["u"], b["u"])
        np.testing.assert_array_equal(a["grad"], b["grad"])
