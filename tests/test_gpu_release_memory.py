"""release_memory() leaves no block of closed objects with the library."""
import pytest
import torch

import admfem
from admfem import meshgen

pytestmark = pytest.mark.gpu


def test_release_memory():
    def make():
        c, e = meshgen.jittered_square(500, seed=1)
        mesh = admfem.Mesh(c, e, zero_based=True)
        S = admfem.DirichletSystem(mesh, admfem.bcnode(mesh))
        held = torch.cuda.mem_get_info()[0]
        S.close()
        mesh.close()
        return held
    make()
    admfem.release_memory()
    free = torch.cuda.mem_get_info()[0]
    held = make()
    print("release", free, held, flush=True)
    assert held < free - (50 << 20)
    admfem.release_memory()
    assert torch.cuda.mem_get_info()[0] >= free
