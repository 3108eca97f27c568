"""What the serving engine's limits count."""
import numpy as np
import pytest
import torch

import admfem
from admfem import meshgen
from admfem.server import Server

pytestmark = pytest.mark.gpu


def topology(m):
    c, e = meshgen.jittered_square(m, seed=m)
    mesh = admfem.Mesh(c, e, zero_based=True)
    return admfem.DirichletSystem(mesh, admfem.bcnode(mesh))


def serve(S, mode="batched", n=1, budget=1 << 30, **kw):
    sv = Server(budget, mode=mode, rtol=1e-8, **kw)
    t = sv.add_topology(S)
    ids = [sv.submit(t, seed=k + 1) for k in range(n)]
    sv.run(timeout=60)
    out = [sv.result(i) for i in ids]
    sv.close()
    return out


def test_iterations_are_products_with_the_matrix():
    """The same unit in both modes, and the one that max_iter is given in: three a
    multigrid iteration.  Grids of either mode differ by rounding only, so their
    counts differ by an iteration at most.  Twelve products, four iterations, do not
    solve to 1e-8 (an iteration takes about a factor of ten)."""
    S = topology(64)
    a, b = (serve(S, mode)[0] for mode in ("batched", "seq_fp64"))
    print("serving, iterations", a["iters_fwd"], a["iters_adj"], b["iters_fwd"], flush=True)
    for k in ("iters_fwd", "iters_adj"):
        assert a[k] % 3 == 0 and abs(a[k] - b[k]) <= 3
    for mode in ("batched", "seq_fp64"):
        assert serve(S, mode, max_iter=12)[0]["status"] == admfem._lib.ERR_NOT_CONVERGED
        r = serve(S, mode, max_iter=a["iters_fwd"] + 6)[0]
        assert r["status"] == 0 and r["iters_fwd"] <= a["iters_fwd"] + 6


@pytest.mark.parametrize("m", [32, 128])
def test_budget_that_holds_a_request_with_the_smaller_solver(m):
    """A request needs more memory with multigrid CG than with Jacobi-PCG: where the
    budget holds it with the latter only, it is served, one at a time; below that it
    is refused."""
    S = topology(m)
    wide = serve(S)[0]
    small = next(r for r in (serve(S, budget=wide["device_bytes"] * q / 100)[0]
                             for q in range(60, 100)) if r["status"] == 0)
    print("serving, budget", m, wide["device_bytes"], small["device_bytes"], flush=True)
    assert small["iters_fwd"] > 2 * wide["iters_fwd"]
    for r in serve(S, n=3, budget=small["device_bytes"]):
        assert r["status"] == 0
    assert np.linalg.norm(small["grad"] - wide["grad"]) < 1e-6 * np.linalg.norm(wide["grad"])
    r = serve(S, budget=small["device_bytes"] - 4096)[0]
    assert r["status"] == admfem._lib.ERR_BUDGET


def test_a_budget_counts_cached_blocks_as_free():
    """An engine's budget is compared with the free memory of the card, and blocks
    that closed meshes left in the library's cache are free."""
    S = topology(900)
    S.close()
    S.mesh.close()
    before = torch.cuda.mem_get_info()[0]
    print("serving, budget and cache", before, flush=True)
    Server(before + (64 << 20)).close()
    assert torch.cuda.mem_get_info()[0] >= before + (64 << 20)  # (there were as many)
