"""Stages of the mixed-radix pencil kernels by the size of the pass (three where two leave the chip short of waves, but
for powers of two) and the thread-team columns of 7 times a power of two, on both sides of each rule, against the generic
pass kernel: relative L2 and Linf <= 1e-12 (FP64), 1e-5 (FP32 storage)."""
import numpy as np
import pytest

try:
    import torch  # noqa: F401
except Exception:   # pragma: no cover
    torch = None

import flups_amd as fl
from tests.test_gpu_parity import TOL, rel_err
from tests.test_gpu_routes import launches

pytestmark = pytest.mark.gpu

E, O, P, U = 0, 1, 3, 4
# (nglob, bc, center, lda): h = 80, 112, 160, 224, 225, 448, 896 columns of kinds I, II and IV in small fields, at 84 x 1024
# threads of two stages and above; rows of 2 x 128, 225, 240 and 256 points; few columns times three components
CASES = {
    "IV-160-few": ((64, 320, 16), [[E, E], [E, O], [P, P]], 1, 1),
    "IV-160-limit": ((83, 320, 64), [[E, E], [O, E], [P, P]], 1, 1),   # 84 x 64 columns of 16 threads
    "IV-160-many": ((84, 320, 64), [[E, E], [E, O], [P, P]], 1, 1),
    "IV-80-few": ((40, 160, 33), [[E, E], [E, O], [P, P]], 1, 1),
    "II-112-few": ((35, 224, 33), [[E, E], [O, O], [P, P]], 1, 1),
    "II-112-many": ((70, 224, 90), [[E, E], [E, E], [P, P]], 1, 1),
    "IV-112-many": ((70, 224, 90), [[E, E], [O, E], [P, P]], 1, 1),
    "I-112-many": ((71, 113, 89), [[E, E], [O, O], [P, P]], 0, 1),
    "IV-224-few": ((33, 448, 32), [[E, E], [E, O], [P, P]], 1, 1),
    "IV-224-many": ((72, 448, 75), [[E, E], [E, O], [P, P]], 1, 1),
    "I-224-many": ((75, 225, 75), [[O, O], [E, E], [P, P]], 0, 1),
    "semi-224": ((75, 113, 75), [[O, O], [E, U], [P, P]], 0, 1),
    "I-896": ((33, 897, 33), [[O, O], [O, O], [P, P]], 0, 1),
    "IV-225": ((34, 450, 30), [[E, E], [O, E], [P, P]], 1, 1),
    "IV-448": ((33, 896, 32), [[E, E], [E, O], [P, P]], 1, 1),
    "rows-128": ((256, 32, 32), [[P, P], [E, E], [P, P]], 1, 1),
    "rows-225": ((450, 36, 32), [[P, P], [E, E], [P, P]], 1, 1),
    "rows-240": ((240, 70, 64), [[U, U], [E, E], [P, P]], 1, 1),
    "rows-256-many": ((512, 72, 64), [[P, P], [O, O], [P, P]], 1, 1),
    "rows-node-256": ((513, 41, 33), [[P, P], [E, E], [P, P]], 0, 1),
    "strided-r2c-224": ((33, 448, 32), [[O, O], [P, P], [P, P]], 1, 1),
    "vector-IV-160": ((40, 320, 36), [[E, E], [E, O], [P, P]], 1, 3),
}


def setup(nglob, bc, center, lda, fp32=False):
    h = [1.0 / (max(nglob) - (1 - center))] * 3
    s = fl.Solver(fl.Topology(0, lda, list(nglob), [1, 1, 1], False), bc, h, [h[0] * (m - (1 - center)) for m in nglob],
                  center_type=[center] * 3)
    s.set_green_type(0)
    if fp32:
        s.set_precision(True)
    s.setup()
    return s


@pytest.mark.parametrize("fp32", [False, True], ids=["fp64", "fp32"])
@pytest.mark.parametrize("name", CASES)
def test_stages_by_size(name, fp32, monkeypatch):
    nglob, bc, center, lda = CASES[name]
    rhs = np.random.default_rng(29).normal(size=(lda, nglob[2], nglob[1], nglob[0]))
    rhs -= rhs.mean(axis=(1, 2, 3), keepdims=True)
    din, dout = fl.DeviceArray.from_numpy(rhs), fl.DeviceArray(rhs.shape)
    s = setup(nglob, bc, center, lda, fp32)
    assert s.pass_kernels[1] > 0, s.pass_kernels
    s.solve(dout, din)
    got = dout.numpy()
    monkeypatch.setenv("FLUPS_GENERIC_PASS", "1")
    monkeypatch.setenv("FLUPS_FORCE_GENERIC", "1")
    g = setup(nglob, bc, center, lda)
    assert all(k <= 0 for k in g.pass_kernels)
    g.solve(dout, din)
    e2, ei = rel_err(got, dout.numpy())
    assert max(e2, ei) <= (1e-5 if fp32 else TOL), (e2, ei)


def test_small_passes_get_the_threads():
    """65 x 16 columns of 160 points: 40 threads each (three stages), not the 16 of stages of radix 10 and 16"""
    nglob, bc, center, lda = CASES["IV-160-few"]
    grid, block = launches(setup(nglob, bc, center, lda), nglob)[1]
    assert (grid, block) == (16 * 9, 8 * 40)   # tiles of 8
