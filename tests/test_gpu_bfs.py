"""The level-by-level search behind the row order of a general sparse solve, on
graphs whose levels are narrow (one workgroup), wide (a launch a level) and
both in turn, longer than a batch of levels, and a single node.

Matrices are graph Laplacians plus the identity, numbered at random: condition
number at most 2 x degree + 1 <= 6001, so a relative residual of 1e-12 keeps
the error below 6001e-12; asserted 1e-8."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spl
import torch

import admfem

pytestmark = pytest.mark.gpu


def path(n, first=0):
    return np.stack([np.arange(n - 1), np.arange(1, n)], 1) + first


def star(n, first=0):
    return np.stack([np.full(n, first), np.arange(first + 1, first + n + 1)], 1)


GRAPHS = {
    "one node": (1, np.zeros((0, 2), dtype=int)),
    "path": (2000, path(2000)),
    "star": (3001, star(3000)),
    "narrow, wide, narrow": (3600, np.concatenate(
        [path(300), star(3000, 299), path(301, 3299)])),
    "level of 1024": (1025, star(1024)),
    "level of 1025": (1026, star(1025)),
}


@pytest.mark.parametrize("name", list(GRAPHS))
def test_solve_on_shuffled_graph(name):
    print(name, flush=True)
    n, e = GRAPHS[name]
    rng = np.random.default_rng(2)
    p = rng.permutation(n)
    i, j = (p[e[:, 0]], p[e[:, 1]]) if len(e) else (np.zeros(0, int), np.zeros(0, int))
    W = sp.coo_matrix((np.ones(len(i)), (i, j)), shape=(n, n)).tocsr()
    W = W + W.T
    A = (sp.diags(np.asarray(W.sum(1)).ravel() + 1.0) - W).tocoo()
    b = rng.standard_normal(n)
    T = admfem.SparseTensor(np.stack([A.row, A.col], 1), A.data, n)
    u = admfem.solve(T, torch.as_tensor(b, device="cuda")).cpu().numpy()
    want = spl.spsolve(A.tocsc(), b)
    assert np.linalg.norm(u - want) <= 1e-8 * np.linalg.norm(want)
