"""The coarse level's A P where its places can go wrong: a last slice of fewer
than 16 rows, one slice only, rows of unequal length and (the reference's
mesh) of more blocks than one batch holds.  The preconditioner's definition
assembled on the CPU, from the oracle's Jacobian and fine solve: FP64 within
1e-9 (2-norm, relative), the bound of the whole-mesh test; FP32 within 1e-4
and BF16 within 5e-2, far above their rounding (1e-6, 1e-2) and far below one
block taken for another, which changes the correction by its own size."""
import numpy as np
import pytest
import scipy.sparse as sp

import kfun3d_amd as K
import oracle as O
from conftest import lattice, perturbed_state
from coarse_ref import block_ilu0, block_ilu0_solve

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(3, 3, 2), (4, 4, 2), (5, 13, 2), (17, 3, 3), (17, 9, 8), None])
def test_apply_at_slice_edges(mesh_dir, mesh_a, dims):
    m = K.Mesh(lattice(mesh_dir, *dims, 5) if dims else mesh_a, K.options(coarse=1))
    orc = O.Oracle(m)
    try:
        q = perturbed_state(m.N, 3.0, 17)
        for s in (m, orc):
            s.set_state(q)
            s.timestep(30.0)
            s.fill()
        rp, col = (a.astype(np.int64) for a in orc.pattern())
        A = orc.blocks().reshape(-1, 4, 4).copy()
        orc.ilu()
        b = np.random.default_rng(5).standard_normal(m.sz)
        bd, xd = K.DeviceVec(m.sz, b), K.DeviceVec(m.sz)
        want = None
        for prec, tol in (("fp64", 1e-9), ("fp32", 1e-4), ("bf16", 5e-2)):
            m.set_options(K.options(coarse=1, prec=prec))
            m.fill()
            m.ilu()
            m.sptrsv(bd, xd)
            if want is None:
                agg, crp, ccol, Ac = m.coarse_matrix()
                agg, nc = agg.astype(np.int64), len(crp) - 1
                if dims is None:   # the batch's end is reached
                    assert max(len(set(agg[col[rp[r]:rp[r + 1]]])) for r in range(m.N)) > 8
                P = sp.csr_matrix((np.ones(m.sz), 4 * np.repeat(agg, 4) + np.tile(np.arange(4), m.N),
                                   np.arange(m.sz + 1)), shape=(m.sz, 4 * nc))
                z = P @ block_ilu0_solve(block_ilu0(crp.astype(np.int64), ccol.astype(np.int64), Ac), P.T @ b)
                want = z + orc.sptrsv(b - sp.bsr_matrix((A, col, rp), shape=(m.sz, m.sz)).tocsr() @ z)
            err = np.linalg.norm(xd.numpy() - want) / np.linalg.norm(want)
            assert err <= tol, (prec, err)
        assert m.last_error() == 0
    finally:
        orc.close()
        m.close()
