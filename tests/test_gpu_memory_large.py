"""Device blocks that are never cached (above 64 MiB) are as large as they are asked
for: from 2508^2 to 2509^2 quads, where an array of a double per Gauss point grows past
an eighth of a power of two, a mesh and its system grow by 0.08%, 3 MB, and by what
their smaller arrays, some eight of at most 64 MiB, may step by an eighth."""
import pytest
import torch

import admfem
from admfem import _lib, meshgen

pytestmark = pytest.mark.gpu


def used(m):
    c, e = meshgen.rectangle(m, m, 1 / m)
    torch.cuda.synchronize()
    _lib.check(_lib.lib().admfem_release_memory())
    before = torch.cuda.mem_get_info()[0]
    mesh = admfem.Mesh(c, e, zero_based=True)
    S = admfem.DirichletSystem(mesh, admfem.bcnode(mesh))
    _lib.check(_lib.lib().admfem_release_memory())
    after = torch.cuda.mem_get_info()[0]
    S.close()
    mesh.close()
    return before - after


def test_large_blocks_are_not_rounded():
    used(100)  # (the runtime's own first allocations)
    a, b = used(2508), used(2509)
    print("large blocks", a, b, flush=True)
    assert b - a < (64 << 20) + (3 << 20)
