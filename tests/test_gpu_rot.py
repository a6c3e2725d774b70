"""The rotational (Biot-Savart) last directions, fused with the curl: the fused pipeline's persistent z pass
and the general path's mixed-radix one, against the oracle: relative L2 and Linf <= 1e-12 (FP64), 1e-5 (FP32)."""
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

P, U = 3, 4
# (nglob, bc, center, odiff): every z length of the pipeline, zero-padded (cell, node) and full columns, more
# items than blocks (256-256-16, 128-128-64), x tiles with a remainder, one row without a mirror
PIPELINE = {
    "256-256-16": ((256, 256, 16), [[U, U]] * 3, 1, 1),
    "128-128-64": ((128, 128, 64), [[U, U]] * 3, 1, 4),
    "node-65-33-33": ((65, 33, 33), [[U, U]] * 3, 0, 1),
    "node-33-65-129": ((33, 65, 129), [[U, U]] * 3, 0, 2),
    "node-33-33-257": ((33, 33, 257), [[U, U]] * 3, 0, 1),
    "32-32-512": ((32, 32, 512), [[U, U]] * 3, 1, 6),
    "periodic-32-64-32": ((32, 64, 32), [[P, P]] * 3, 1, 1),
    "periodic-64-32-1024": ((64, 32, 1024), [[P, P]] * 3, 1, 1),
    "duct-64-32-64": ((64, 32, 64), [[P, P], [U, U], [U, U]], 1, 1),
}
# the general path: column lengths of 2 to 4 stages and every tile width, mirrored and single rows, powers of two
# (32, 128, 1024), 3, 5 and 7 times one, odd lengths, x unbounded after a periodic y, node-centred
GENERAL = {
    "open-48-40-24": ((48, 40, 24), [[U, U]] * 3, 1, 1),
    "layer-40-40-40": ((40, 40, 40), [[P, P], [P, P], [U, U]], 1, 1),
    "layer-fd4-36-50-45": ((36, 50, 45), [[P, P], [P, P], [U, U]], 1, 4),
    "periodic-36-45-18": ((36, 45, 18), [[P, P]] * 3, 1, 2),
    "periodic-24-36-32": ((24, 36, 32), [[P, P]] * 3, 1, 1),
    "periodic-24-20-1024": ((24, 20, 1024), [[P, P]] * 3, 1, 1),
    "duct-48-28-64": ((48, 28, 64), [[P, P], [U, U], [U, U]], 1, 6),
    "node-open-41-31-26": ((41, 31, 26), [[U, U]] * 3, 0, 1),
    "y-first-42-36-35": ((42, 36, 35), [[U, U], [P, P], [U, U]], 1, 1),
    "z-160": ((24, 20, 160), [[P, P], [P, P], [U, U]], 1, 1),
    "z-315": ((22, 20, 315), [[U, U]] * 3, 1, 1),
    "z-675": ((20, 18, 675), [[U, U]] * 3, 1, 1),
}


def solve(nglob, bc, center, odiff, rhs, fp32=False):
    h = [1.0 / (max(nglob) - (1 - center))] * 3
    L = [h[0] * (m - (1 - center)) for m in nglob]
    topo = fl.Topology(0, 3, list(nglob), [1, 1, 1], False)
    s = fl.Solver(topo, bc, h, L, order_diff=odiff, center_type=[center] * 3)
    s.set_green_type(0)
    if fp32:
        s.set_precision(True)
    s.setup()
    din, dout = fl.DeviceArray.from_numpy(rhs), fl.DeviceArray(rhs.shape)
    s.solve(dout, din, 1)
    return dout.numpy(), s.path, orc.solve(list(nglob), bc, 3, h, L, center, 0, rhs, 1, odiff)


def field(nglob, seed=23):
    rhs = np.random.default_rng(seed).normal(size=(3, nglob[2], nglob[1], nglob[0]))
    return rhs - rhs.mean(axis=(1, 2, 3), keepdims=True)


@pytest.mark.parametrize("fp32", [False, True], ids=["fp64", "fp32"])
@pytest.mark.parametrize("name", PIPELINE)
def test_pipeline_rot(name, fp32):
    got, path, ora = solve(*PIPELINE[name], field(PIPELINE[name][0]), fp32)
    assert path == (2 if fp32 else 1)
    e2, ei = rel_err(got, ora)
    assert max(e2, ei) <= (1e-5 if fp32 else TOL), (e2, ei)


@pytest.mark.parametrize("fp32", [False, True], ids=["fp64", "fp32"])
@pytest.mark.parametrize("name", GENERAL)
def test_general_rot(name, fp32):
    got, path, ora = solve(*GENERAL[name], field(GENERAL[name][0]), fp32)
    assert path == (5 if fp32 else 3)
    e2, ei = rel_err(got, ora)
    assert max(e2, ei) <= (1e-5 if fp32 else TOL), (e2, ei)
