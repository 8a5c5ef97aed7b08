"""The places of the edges' fluxes (kf_place_edges, by slices in parallel)
against a plain edge-by-edge construction: lists of each vertex's own edges in
ascending edge id, an edge in its n0's list, or in that of the end with fewer
edges so far where this takes fewer places; vertex v's k-th at (row of its
slice + k) 64 + v % 64.  A lattice (the first rule) and the reference's mesh
(the second), each several times: the places must not depend on the threads."""
import ctypes as C

import numpy as np
import pytest

import kfun3d_amd as K
from conftest import lattice


def _places(m):
    L = K.lib()
    prep = C.create_string_buffer(4096)   # a kf_prep, larger than it is
    L.kf_build_prep.argtypes = [C.c_void_p, C.c_void_p]
    L.kf_free_prep.argtypes = [C.c_void_p]
    L.kf_place_edges.argtypes = [C.c_void_p, C.c_void_p, C.c_void_p]
    L.kf_place_edges.restype = C.c_size_t
    L.kf_build_prep.restype = L.kf_free_prep.restype = None
    pos = np.full(m.E, 0xffffffff, dtype=np.uint32)
    L.kf_build_prep(m.ref, prep)
    n = L.kf_place_edges(m.ref, prep, pos.ctypes.data)
    L.kf_free_prep(prep)
    return n, pos


def _listed(N, owner):
    """places and their number with edge e in owner[e]'s list"""
    deg, rank = np.zeros(N, dtype=np.int64), np.empty(len(owner), dtype=np.int64)
    for e, v in enumerate(owner):
        rank[e] = deg[v]
        deg[v] += 1
    length = np.array([deg[s:s + 64].max() for s in range(0, N, 64)])
    row = np.concatenate([[0], np.cumsum(length)])
    return int(row[-1]) * 64, (row[owner >> 6] + rank) * 64 + (owner & 63)


@pytest.mark.parametrize("dims", [None, (2, 2, 2), (13, 7, 5), (24, 10, 9)])
def test_places_match_edge_by_edge_construction(mesh_dir, mesh_a, dims):
    m = K.Mesh(lattice(mesh_dir, *dims, 5) if dims else mesh_a, device=False)
    try:
        h = m.host_arrays()
        n0, n1 = h["e_n0"].astype(np.int64), h["e_n1"].astype(np.int64)
        n, pos = _listed(m.N, n0)
        if 8 * n > 9 * m.E:
            deg, owner = [0] * m.N, np.empty_like(n0)
            for e, (a, b) in enumerate(zip(n0, n1)):
                owner[e] = b if deg[b] < deg[a] else a
                deg[owner[e]] += 1
            even = _listed(m.N, owner)
            if even[0] < n:
                n, pos = even
        for _ in range(3):
            got_n, got = _places(m)
            assert got_n == n
            assert np.array_equal(got.astype(np.int64), pos)
        assert len(np.unique(pos)) == m.E and pos.max() < n
    finally:
        m.close()
