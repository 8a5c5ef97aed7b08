"""The residual where its edges and places can go wrong: fewer edges than a
wavefront, a last wavefront that is not full (its fluxes are stored lane by
lane, a full one's by pairs of lanes), slices whose vertices have unequal
shares of edges, and both ways of sharing them out (lattices: an edge's first
end; the reference's mesh: the end with fewer).  Small meshes take one kernel
in place of the edges' and the vertices' (16 lanes to a vertex, which the
reference's mesh's vertices outnumber; past 12,288 vertices 4), except where
the caller's residual lies over the gradient: both ways here.  Bit for bit
against the oracle, twice with different states, and with the time-step
sums."""
import numpy as np
import pytest

import kfun3d_amd as K
import oracle as O

from conftest import lattice, perturbed_state

pytestmark = pytest.mark.gpu


def _same(a, b):
    return np.array_equal(np.asarray(a).view(np.uint64), np.asarray(b).view(np.uint64))


@pytest.mark.parametrize("dims", [(2, 2, 2), (3, 3, 2), (4, 4, 4), (13, 5, 2), (5, 13, 2), (17, 9, 8), (65, 3, 3),
                                  (48, 16, 16), (59, 19, 11), (63, 20, 26), (64, 32, 16), (33, 31, 33), None])
def test_residual_at_wavefront_edges(mesh_dir, mesh_a, dims):
    m = K.Mesh(lattice(mesh_dir, *dims, 5) if dims else mesh_a)
    orc = O.Oracle(m)
    try:
        g = [K.DeviceVec(m.sz) for _ in range(3)]
        r = K.DeviceVec(m.sz)
        for seed in (7, 8):
            q = perturbed_state(m.N, 3.0, seed)
            for s in (m, orc):
                s.set_state(q)
                s.timestep(37.0)
            qd = K.DeviceVec(m.sz, q)
            want = orc.flux(q)[0]
            m.flux(qd, g, r)
            assert _same(r.numpy(), want)
            m.flux(qd, g, g[0])
            assert _same(g[0].numpy(), want)
            m.flux_spectral(qd, g, r)
            assert _same(r.numpy(), want)
            m.timestep_spectral(37.0)
            assert _same(m.cdt(), orc.cdt())
            m.flux_spectral(qd, g, g[1])
            assert _same(g[1].numpy(), want)
            m.timestep_spectral(37.0)
            assert _same(m.cdt(), orc.cdt())
    finally:
        orc.close()
        m.close()
