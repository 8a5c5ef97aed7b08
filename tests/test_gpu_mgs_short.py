"""Modified Gram-Schmidt in one launch at the lengths where its grid changes:
one to 256 workgroups (256 element pairs each), with and without the half
pair of an odd length, and just past one set and one pass; short and long
calls in turn on one context, since a call's table is made ready by the one
before it.  Every h_k, |w| and w bit for bit against the per-step kernels."""
import ctypes as C

import numpy as np
import pytest

import kfun3d_amd as K

pytestmark = pytest.mark.gpu

P = 256          # element pairs of a workgroup's first set
SLOT = 100
LENGTHS = [2, 3, 2 * P - 1, 2 * P, 2 * P + 1, 2 * P * 255 + 1, 2 * P * 256, 2 * P * 256 + 1, 2 * P * 257, 5,
           2 * P * 1024 - 1, 2 * P * 1024 + 2, 6, 2 * P * 3 * 1024 + 1, 4 * P]


def test_mgs_lengths_in_turn(mesh_a, monkeypatch):
    L = K.lib()
    L.kfs_mgs.restype = None
    L.kfs_mgs.argtypes = [K.GP, C.c_size_t, C.c_void_p, C.c_size_t, C.c_int, C.c_void_p, C.c_int]
    L.kfs_fetch.restype = None
    L.kfs_fetch.argtypes = [K.GP, C.c_int, C.c_int, C.c_void_p]
    L.kfs_mgs_launches.restype = C.c_ulonglong
    L.kfs_mgs_launches.argtypes = [K.GP]
    m = {}
    for name, val in (("step", "0"), ("resident", "2")):
        monkeypatch.setenv("KF_MGS_RESIDENT", val)
        m[name] = K.Mesh(mesh_a, K.options())
    try:
        rng = np.random.default_rng(3)
        for i, n in enumerate(LENGTHS):
            nv = 1 + i % 4
            stride = n + (n & 1) + 2
            V = rng.standard_normal((nv, stride)) / np.sqrt(n)
            w0 = rng.standard_normal(n)
            got = {}
            for name, mesh in m.items():
                vd, wd = K.DeviceVec(V.size, V.ravel()), K.DeviceVec(n, w0)
                before = L.kfs_mgs_launches(mesh.ref)
                L.kfs_mgs(mesh.ref, n, vd.ptr, stride, nv, wd.ptr, SLOT)
                h = np.empty(nv + 1)
                L.kfs_fetch(mesh.ref, SLOT, nv + 1, h.ctypes.data)
                assert L.kfs_mgs_launches(mesh.ref) - before == (name == "resident")
                got[name] = np.concatenate([h, wd.numpy()])
                vd.free()
                wd.free()
            assert np.array_equal(got["step"].view(np.uint64), got["resident"].view(np.uint64)), n
    finally:
        for mesh in m.values():
            mesh.close()
