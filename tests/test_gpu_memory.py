"""The cache of released device blocks: objects made and closed in turn and by
several threads at once give the same results as the first ones, and
admfem_release_memory returns what is cached."""
import threading

import numpy as np
import pytest
import torch

import admfem
from admfem import _lib, meshgen

pytestmark = pytest.mark.gpu


def solve(m, seed):
    c, e = meshgen.jittered_square(m, seed=seed)
    mesh = admfem.Mesh(c, e, zero_based=True)
    S = admfem.DirichletSystem(mesh, admfem.bcnode(mesh))
    kap = torch.full((mesh.ngauss,), 1.0 + seed, dtype=torch.float64, device="cuda")
    out = S.forward_adjoint(np.arange(m + 3, m + 6), np.zeros(3), kappa=kap, f=kap, rtol=1e-12)
    r = [out[k].cpu().numpy() for k in ("u", "lam", "grad_kappa")]
    S.close()
    mesh.close()
    return r


def test_released_blocks_are_reused_and_given_back():
    cases = [(60, 1), (33, 2), (90, 3)]
    first = [solve(*c) for c in cases]
    bad = []

    def work(k):
        torch.cuda.set_device(0)
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(5):
                for c, ref in zip(cases[k:] + cases[:k], first[k:] + first[:k]):
                    if not all(np.array_equal(a, b) for a, b in zip(solve(*c), ref)):
                        bad.append(c)
    th = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad, bad
    torch.cuda.synchronize()
    _lib.check(_lib.lib().admfem_release_memory())
    free0 = torch.cuda.mem_get_info()[0]
    solve(300, 4)
    assert torch.cuda.mem_get_info()[0] < free0 - (1 << 20)  # blocks are kept
    _lib.check(_lib.lib().admfem_release_memory())
    assert abs(torch.cuda.mem_get_info()[0] - free0) < 64 << 20
