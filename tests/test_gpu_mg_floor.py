"""Tolerances just above what FP64 can reach: a solve that reports success has
its true residual within them.  The floor is the smallest residual of solves asked
for 1e-13 to 1e-16, which end there; a tenth above it leaves room for the
roundings of another number of iterations."""
import numpy as np
import pytest
import torch

import admfem
from admfem import meshgen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("degree,m,seed", [(1, 20, 2), (1, 128, 0), (2, 20, 0), (2, 70, 0),
                                           (2, 101, 0)])
def test_residual_within_tolerance(degree, m, seed):
    c, e = meshgen.jittered_square(m, seed=seed + 1)
    mesh = admfem.Mesh(c, e, degree=degree, zero_based=True)
    S = admfem.DirichletSystem(mesh, admfem.bcnode(mesh))
    rng = np.random.default_rng(seed)
    kap = torch.tensor(np.exp(rng.standard_normal(mesh.ngauss)), device="cuda")
    S.assemble(kappa=kap, f=torch.tensor(1 + 0.1 * rng.uniform(-1, 1, mesh.ngauss)))
    floor = min(S.solve(rtol=t)[1]["rel_residual"] for t in (1e-13, 1e-14, 1e-15, 1e-16))
    for q in (1.1, 1.3, 2.0, 5.0):
        st = S.solve(rtol=q * floor)[1]
        print("floor", degree, m, floor, q, st, flush=True)
        assert st["status"] == 0 and st["rel_residual"] <= q * floor
