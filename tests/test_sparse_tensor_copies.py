"""SparseTensor objects that hold their mesh are copied and pickled like those that
do not: a copy has the same mesh object (whose library handle cannot be copied),
an unpickled one has none."""
import copy
import ctypes
import pickle

import torch

from admfem.ops import SparseTensor


class Handle:
    def __init__(self):
        self._h = ctypes.c_void_p(1)


def tensor(mesh):
    A = SparseTensor.__new__(SparseTensor)  # (the constructor moves to the GPU)
    A.indices = torch.tensor([[0, 0], [1, 1]])
    A.values, A.n, A.mesh = torch.tensor([1.0, 2.0], dtype=torch.float64), 2, mesh
    return A


def test_copies_keep_the_mesh():
    A = tensor(Handle())
    for B in (copy.copy(A), copy.deepcopy(A), copy.deepcopy({"a": [A]})["a"][0]):
        assert B is not A and B.mesh is A.mesh and B.n == 2
        assert torch.equal(B.values, A.values) and torch.equal(B.indices, A.indices)
    B = copy.deepcopy(A)
    B.values[0] = 5.0
    assert A.values[0] == 1.0


def test_pickles_leave_the_mesh():
    A = tensor(Handle())
    B = pickle.loads(pickle.dumps(A))
    assert B.mesh is None and B.n == 2 and torch.equal(B.values, A.values)
    assert A.mesh is not None
    assert pickle.loads(pickle.dumps(tensor(None))).mesh is None
