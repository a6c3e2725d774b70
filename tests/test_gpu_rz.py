"""An r2c last direction fused with the multiply at lengths with factors 2, 3, 5, 7 (walls or semi-unbounded
directions before it) against the oracle: relative L2 and Linf <= 1e-12 (FP64), 1e-5 (FP32 storage)."""
import numpy as np
import pytest

try:
    import torch  # noqa: F401
except Exception:   # pragma: no cover
    torch = None

import flups_amd as fl
from tests import oracle_lib as orc
from tests.test_gpu_parity import TOL, rel_err

pytestmark = pytest.mark.gpu

E, O, P, U, X = 0, 1, 3, 4, 9
# (nglob, bc, center, lda): two to four stages, radices above 10, odd x (a column without partner), odd
# lengths, padded and full columns, one tile and a ragged one, two dimensions
CASES = {
    "walls-z48": ((20, 18, 24), [[O, O], [E, E], [U, U]], 1, 1),
    "walls-z50": ((33, 16, 25), [[O, O], [E, E], [U, U]], 1, 1),
    "node-z192": ((33, 41, 97), [[O, O], [E, E], [U, U]], 0, 1),
    "periodic-z18": ((31, 20, 18), [[E, E], [O, E], [P, P]], 1, 1),
    "periodic-odd-z45": ((20, 21, 45), [[E, E], [O, O], [P, P]], 1, 1),
    "periodic-z224": ((17, 16, 224), [[E, O], [O, O], [P, P]], 1, 1),
    "periodic-z1500": ((18, 16, 1500), [[E, E], [O, O], [P, P]], 1, 1),
    "vector-z100": ((25, 24, 50), [[O, O], [E, E], [U, U]], 1, 3),
    "plane-y120": ((37, 60, 1), [[E, E], [U, U], [X, X]], 1, 1),
}


@pytest.mark.parametrize("fp32", [False, True], ids=["fp64", "fp32"])
@pytest.mark.parametrize("name", CASES)
def test_r2c_last_direction(name, fp32):
    nglob, bc, center, lda = CASES[name]
    rhs = np.random.default_rng(5).normal(size=(lda, nglob[2], nglob[1], nglob[0]))
    rhs -= rhs.mean(axis=(1, 2, 3), keepdims=True)
    h = [1.0 / (max(nglob) - (1 - center))] * 3
    L = [h[0] * max(m - (1 - center), 1) for m in nglob]
    s = fl.Solver(fl.Topology(0, lda, list(nglob), [1, 1, 1], False), bc, h, L, center_type=[center] * 3)
    s.set_green_type(0)
    if fp32:
        s.set_precision(True)
    s.setup()
    assert s.path == (5 if fp32 else 3)
    din, dout = fl.DeviceArray.from_numpy(rhs), fl.DeviceArray(rhs.shape)
    s.solve(dout, din)
    e2, ei = rel_err(dout.numpy(), orc.solve(list(nglob), bc, lda, h, L, center, 0, rhs))
    assert max(e2, ei) <= (1e-5 if fp32 else TOL), (e2, ei)
