"""The Jacobian fill where its stores can go wrong: rows of one 64-row slice
and of several, a last slice of one row, isolated remainders of FP32 lines
(rows of odd and even length, a line shared by two rows, a diagonal between
two halves) and the kept copy written beside the matrix.  FP64 bit for bit
against the oracle, the kept copy by the product with it; FP32 within
3e-6 of the largest entry and 1e-6 of the product's norm (the bounds of the
single-precision preconditioner elsewhere).  Every check runs at two states
in turn, so that a block left from the first one shows."""
import numpy as np
import pytest

import kfun3d_amd as K
import oracle as O

from conftest import lattice, perturbed_state

pytestmark = pytest.mark.gpu


def _same(a, b):
    return np.array_equal(np.asarray(a).view(np.uint64), np.asarray(b).view(np.uint64))


@pytest.mark.parametrize("keep", [0, 1])
@pytest.mark.parametrize("dims", [(2, 2, 2), (3, 3, 2), (13, 5, 2), (4, 4, 4), (5, 13, 2), (17, 9, 8), (43, 3, 3), None])
def test_fill_at_slice_and_line_edges(mesh_dir, mesh_a, dims, keep):
    path = lattice(mesh_dir, *dims, 5) if dims else mesh_a
    m = K.Mesh(path, K.options(bsr_operator=keep))
    orc = O.Oracle(m)
    try:
        x = np.random.default_rng(6).standard_normal(m.sz)
        xd, yd = K.DeviceVec(m.sz, x), K.DeviceVec(m.sz)
        for seed, cfl in ((7, 50.0), (8, 400.0)):
            q = perturbed_state(m.N, 3.0, seed)
            m.set_options(K.options(bsr_operator=keep))
            for s in (m, orc):
                s.set_state(q)
                s.timestep(cfl)
                s.fill()
            a = orc.blocks()
            assert _same(m.blocks().ravel(), a.ravel())
            want = orc.spmv(x)
            if keep:
                m.spmv(xd, yd)
                assert _same(yd.numpy(), want)
            m.set_options(K.options(bsr_operator=keep, prec="fp32"))
            m.fill()
            assert np.abs(m.blocks() - a).max() <= 3e-6 * np.abs(a).max()
            if keep:
                m.spmv(xd, yd)
                assert np.linalg.norm(yd.numpy() - want) <= 1e-6 * np.linalg.norm(want)
        assert m.last_error() == 0
    finally:
        orc.close()
        m.close()
