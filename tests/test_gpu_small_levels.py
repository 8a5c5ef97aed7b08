"""The multilevel preconditioner's small levels in one launch
(k_jac_small_levels): every precision, chains that end at one row, at the
level's limit of 128 rows, in as many levels as there may be, one and
several sweeps, and (the reference's mesh) rows longer than the held slots.
One application against the same with a launch per sweep and level
(KF_JAC_SMALL=0, read once per process): bit for bit."""
import os
import subprocess
import sys

import pytest

from conftest import lattice

pytestmark = pytest.mark.gpu

_CHILD = """
import sys
sys.path[:0] = [sys.argv[1], sys.argv[1] + "/tests"]
import hashlib
import numpy as np
import kfun3d_amd as K
from conftest import perturbed_state
for path in sys.argv[2:]:
    m = K.Mesh(path, K.options())
    q = perturbed_state(m.N, 3.0, 17)
    b = np.random.default_rng(5).standard_normal(m.sz)
    bd, xd = K.DeviceVec(m.sz, b), K.DeviceVec(m.sz)
    for prec in ("fp64", "fp32", "bf16"):
        for coarse, sweeps, csweeps in ((1, 2, 1), (2, 1, 3), (5, 2, 4), (8, 2, 2)):
            m.set_options(K.options(prec=prec, coarse=coarse, jacobi_sweeps=sweeps, coarse_sweeps=csweeps))
            m.set_state(q)
            m.timestep(30.0)
            m.fill()
            m.ilu()
            for _ in range(2):
                m.sptrsv(bd, xd)
            x = xd.numpy()
            assert np.all(np.isfinite(x)) and m.last_error() == 0
            print(m.N, prec, coarse, hashlib.sha256(x.tobytes()).hexdigest())
    m.close()
"""


def test_one_launch_matches_many(mesh_dir, mesh_a):
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    paths = [lattice(mesh_dir, *d, 5) for d in ((3, 3, 2), (16, 8, 8), (17, 9, 8), (40, 16, 12))] + [mesh_a]
    out = {}
    for flag in ("1", "0"):
        r = subprocess.run([sys.executable, "-c", _CHILD, root] + paths, env=dict(os.environ, KF_JAC_SMALL=flag),
                           stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=100)
        assert r.returncode == 0, r.stderr[-2000:]
        out[flag] = r.stdout.split("\n")
    assert len(out["1"]) == 12 * len(paths) + 1
    assert out["1"] == out["0"]
