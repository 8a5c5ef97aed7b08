"""The planned ILU(0) kernel where its batches and rows end: fewer rows than a
workgroup has wavefronts, a batch that ends inside the rows, workgroups of
one, some and all wavefronts, and (the reference's mesh) rows with more pairs
to a step than the two rounds held in registers.  Bit for bit against the
oracle, the exact sweep twice (the second reads the first's L blocks)."""
import numpy as np
import pytest

import kfun3d_amd as K
import oracle as O

from conftest import lattice, perturbed_state

pytestmark = pytest.mark.gpu


def _same(a, b):
    return np.array_equal(np.asarray(a).view(np.uint64), np.asarray(b).view(np.uint64))


@pytest.mark.parametrize("group", [1, 3, 8])
@pytest.mark.parametrize("dims", [(2, 2, 2), (3, 3, 2), (5, 5, 7), (17, 9, 8), None])
@pytest.mark.parametrize("exact", [1, 0])
def test_ilu_at_batch_edges(mesh_dir, mesh_a, monkeypatch, dims, group, exact):
    monkeypatch.setenv("KF_ILU_GROUP", str(group))
    path = lattice(mesh_dir, *dims, 3) if dims else mesh_a
    m = K.Mesh(path, K.options(ilu_exact=exact))
    orc = O.Oracle(m, ilu_textbook=1 - exact)
    try:
        q = perturbed_state(m.N, 3.0, 17)
        m.set_state(q)
        orc.set_state(q)
        for cfl in (50.0, 400.0):
            for s in (m, orc):
                s.timestep(cfl)
                s.fill()
                s.ilu()
            assert _same(m.blocks().ravel(), orc.blocks().ravel())
        assert m.last_error() == 0
    finally:
        orc.close()
        m.close()
