"""The learned correction's kernels at the sizes where their tiles end: fewer
vertices than one tile of 32, exactly one, one and a few more, a partition
that ends inside a tile, and a few partitions.  Against oracle/mpnn.py, whose
bf16 mode rounds the operands as the matrix cores do.

Bars, set from what the arithmetic can do: what differs is FP32 summation
order (about 1e-6) and a value now and then whose FP32 and FP64 versions
round to neighbouring bfloat16 numbers, 2^-8 of it; with as few as 8 x 32
values such a flip can move a layer's 2-norm by 2^-8 / 16 and, through three
rounds and a gradient, some times that.  A wrong lane, row or partition, or a
dropped tile, gives errors of order 1e-1 or more.  So 2e-3 in 2-norm for the
forward pass, 2e-2 for each gradient block, 1e-4 for the loss.
"""
import numpy as np
import pytest

import kfun3d_amd as K
from oracle import mpnn as P

from conftest import lattice

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(2, 2, 2), (4, 4, 2), (3, 3, 4), (2, 3, 11), (7, 11, 13), (33, 32, 32)])
def test_network_at_tile_edges(mesh_dir, dims):
    m = K.Mesh(lattice(mesh_dir, *dims, 5), K.options())
    h = m.host_arrays()
    g = P.Graph(h["e_n0"], h["e_n1"], h["e_x0"], h["e_x1"], h["e_x2"], h["e_x3"], m.N)
    theta = P.init_params(seed=12, head_scale=3.0)
    net = K.Network(m, theta)
    rng = np.random.default_rng(sum(dims))
    v, base, target = (rng.standard_normal(4 * m.N) for _ in range(3))
    D = 2.0 * rng.standard_normal(16 * m.N)
    net.set_diag(D)
    net.set_loss("euclid")
    zd, od = K.DeviceVec(m.sz, base), K.DeviceVec(m.sz)
    net.forward(zd, od)
    th = theta.astype(np.float64)
    delta = P.forward(th, g, base, D, round_bf16=True).ravel()
    assert np.linalg.norm(od.numpy() - delta) <= 2e-3 * np.linalg.norm(delta)
    vd, td = K.DeviceVec(m.sz, v), K.DeviceVec(m.sz, target)
    loss, grad = net.loss_grad(vd, zd, td)
    lref, gref = P.loss_and_grad(th, g, v, D, base, target, round_bf16=True)
    assert abs(loss - lref) <= 1e-4 * abs(lref)
    o = 0
    for name, shape in P.PARAM_SHAPES:
        n = int(np.prod(shape))
        a, b = grad[o:o + n].astype(np.float64), gref[o:o + n]
        assert np.linalg.norm(a - b) <= 2e-2 * max(np.linalg.norm(b), 1e-30), name
        o += n
    loss2, grad2 = net.loss_grad(vd, zd, td)
    assert loss2 == loss
    np.testing.assert_array_equal(grad2.view(np.uint32), grad.view(np.uint32))
    net.close()
    m.close()
