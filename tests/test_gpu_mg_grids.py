"""The multigrid kernels at the edges of their forms: the smallest system, every
grid in the tail with its rows staged in LDS and, past 7,000 rows, read from
memory, both splits of the first grid's product (20,000 nodes), long strips
whose tail is narrow.

The preconditioner only shapes the iteration, so a wrong entry shows in the
count: 3 products an iteration, at most 30 iterations, twice what the method
takes at every size.  The solution is compared with the oracle's direct solve where
that is quick, to the suite's 1e-9 (relative residual 1e-13 times a condition
number below 4e5 is 4e-8 at the very worst; smooth right-hand sides leave a
factor of 100)."""
import numpy as np
import pytest
import torch

import admfem
from admfem import meshgen
from oracle import oracle as O
from test_gpu_mg import grid

pytestmark = pytest.mark.gpu


def wide_column(c):
    """One column and one row of the mesh 2.6 times as wide as the others: cells
    of about seven rows, 10,201 rows on a grid that fits the tail."""
    h = 1.0 / (100 + 1.6)
    i = np.round(c * 100)
    return h * (i + 1.6 * (i > 50))


CASES = {
    "smallest": dict(g=(15, 14), solve=True),
    "two grids": dict(g=(24, 25), solve=True),
    "staged rows": dict(g=(80, 79), solve=True),
    "rows from memory": dict(g=(100, 100), warp=wide_column, solve=True),
    "strip": dict(g=(700, 8), solve=True),
    "wide product": dict(g=(310, 300)),
    "P2 tail": dict(g=(30, 31), degree=2, solve=True),
}


@pytest.mark.parametrize("name", list(CASES))
def test_iterations_and_solution(name):
    k = CASES[name]
    print(name, flush=True)
    mx, my = k["g"]
    h = 1.0 / max(mx, my)
    c, e = grid(mx, my, h, h, seed=7, warp=k.get("warp"))
    degree = k.get("degree", 1)
    gm = admfem.Mesh(c, e, degree=degree, zero_based=True)
    bd = admfem.bcnode(gm)
    S = admfem.DirichletSystem(gm, bd)
    rng = np.random.default_rng(8)
    kap = np.exp(0.5 * np.sin(7 * np.arange(gm.ngauss) / gm.ngauss))
    f = 1.0 + 0.5 * rng.uniform(-1, 1, gm.ngauss)
    inner = np.setdiff1d(np.arange(gm.ndof), bd - 1)
    obs = rng.choice(inner, 20, replace=False)
    out = S.forward_adjoint(obs, np.zeros(20), rtol=1e-12, kappa=kap, f=f)
    print([s["iterations"] for s in out["stats"]], flush=True)
    for s in out["stats"]:
        assert 0 < s["iterations"] <= 3 * 30
    if not k.get("solve"):
        return
    om = O.OracleMesh(c, e) if degree == 1 else O.OracleMesh(c, e, degree=2)
    b1 = om.bcnode()
    ref = O.forward_adjoint(om, kap, f, b1, np.zeros(b1.size), lambda v: 0 * v)
    u = out["u"].cpu().numpy()
    assert np.linalg.norm(u - ref["u"]) <= 1e-9 * np.linalg.norm(ref["u"])
