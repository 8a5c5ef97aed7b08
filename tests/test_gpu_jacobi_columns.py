"""The Jacobi sweeps' two ways to a column with seven slots a row: distances
of 16 signed bits where no column is further than 32,767 rows from its row's,
32-bit columns otherwise.  Thin lattices whose furthest column (the cell
diagonal's, nx ny + nx + 1 rows away) lies exactly at the limit, one past it
and well past it; the sliced copy written by the factorisation and packed
afterwards from its factors.  Bit for bit against the CSR sweeps of
kf_sptrsv_jacobi_noalloc in all three precisions, and in FP64 against the
oracle's."""
import numpy as np
import pytest

import kfun3d_amd as K
import oracle as O
from conftest import lattice, perturbed_state

LATTICES = [((129, 253, 3), 32767), ((151, 216, 3), 32768), ((182, 182, 3), 33307)]


def _same(a, b):
    return np.array_equal(np.asarray(a).view(np.uint64), np.asarray(b).view(np.uint64))


def _factor(m, q, prec, sweeps):
    m.set_options(K.options(prec=prec, jacobi_sweeps=sweeps))
    m.set_state(q)
    m.timestep(50.0)
    m.fill()
    m.ilu()


@pytest.mark.parametrize("dims,far", LATTICES)
def test_furthest_column(mesh_dir, dims, far):
    m = K.Mesh(lattice(mesh_dir, *dims, 6), device=False)
    try:
        h = m.host_arrays()
        d = h["e_n1"].astype(np.int64) - h["e_n0"].astype(np.int64)
        assert d.min() > 0 and d.max() == far == dims[0] * dims[1] + dims[0] + 1
        assert max(np.bincount(h["e_n0"]).max(), np.bincount(h["e_n1"]).max()) == 7   # seven slots a side
    finally:
        m.close()


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [d for d, _ in LATTICES])
def test_sweeps_near_and_past_the_limit(mesh_dir, dims):
    m = K.Mesh(lattice(mesh_dir, *dims, 6), K.options())
    try:
        q = perturbed_state(m.N, 3.0, 57)
        b = np.random.default_rng(58).standard_normal(m.sz)
        orc = O.Oracle(m)
        orc.set_state(q)
        orc.timestep(50.0)
        orc.fill()
        orc.ilu()
        want = orc.sptrsv_jacobi(b, 3)
        orc.close()
        bd, xd, yd = K.DeviceVec(m.sz, b), K.DeviceVec(m.sz), K.DeviceVec(m.sz)
        for prec in ("fp64", "fp32", "bf16"):
            # written by the factorisation into a new copy, then over it, then packed after one
            for i, sweeps in enumerate((3, 3, 0)):
                _factor(m, q, prec, sweeps)
                m.set_options(K.options(prec=prec, jacobi_sweeps=3))
                m.sptrsv(bd, xd)
                assert m.sptrsv_noalloc(bd, yd) == 0
                m.synchronize()
                x = xd.numpy()
                assert _same(x, yd.numpy()), (dims, prec, i)
                if prec == "fp64" and i == 0:
                    assert _same(x, want), dims
        assert m.last_error() == 0
        for v in (bd, xd, yd):
            v.free()
    finally:
        m.close()
