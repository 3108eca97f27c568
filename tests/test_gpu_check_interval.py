"""The interval between the host's checks, given in iterations, does not have a
solve run on for that long after its end: at 20,000 both forms take what they take
on their own, give or take a factor that leaves out one of hundreds."""
import time

import numpy as np
import pytest
import torch

import admfem
from admfem import meshgen
from admfem.server import Server

pytestmark = pytest.mark.gpu


def shortest(f):
    out = []
    for _ in range(4):
        torch.cuda.synchronize()
        t = time.perf_counter()
        r = f()
        torch.cuda.synchronize()
        out.append(time.perf_counter() - t)
    return r, min(out)


def test_long_intervals_end_with_the_solve():
    c, e = meshgen.jittered_square(64, seed=1)
    mesh = admfem.Mesh(c, e, zero_based=True)
    S = admfem.DirichletSystem(mesh, admfem.bcnode(mesh))
    one = torch.ones(mesh.ngauss, dtype=torch.float64, device="cuda")
    S.assemble(kappa=one, f=one)
    ref, t0 = shortest(lambda: S.solve(rtol=1e-10)[0])
    for every in (1, 5, 20000):
        x, t = shortest(lambda: S.solve(rtol=1e-10, check_every=every)[0])
        print("interval", every, t0, t, flush=True)
        assert torch.equal(x, ref) and t < 20 * t0

    def serve(chunk):
        sv = Server(1 << 30, rtol=1e-9, chunk=chunk)
        t = sv.add_topology(S)
        ids = [sv.submit(t, seed=k + 1) for k in range(4)]
        sv.run(timeout=60)
        return [sv.result(i)["grad"] for i in ids]
    ref, t0 = shortest(lambda: serve(0))
    for chunk in (1, 8, 20000):
        g, t = shortest(lambda: serve(chunk))
        print("chunk", chunk, t0, t, flush=True)
        assert all(np.array_equal(a, b) for a, b in zip(g, ref)) and t < 20 * t0
