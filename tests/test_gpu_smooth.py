"""The run-time mixed-radix kernels (lengths with factors 2, 3, 5, 7 beyond those of the register
kernels) against the generic pass kernel and the oracle: relative L2 and Linf <= 1e-12 (FP64), 1e-5
(FP32 storage)."""
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
# (nglob, bc, center): FFT lengths of 2 to 4 stages and every radix, the smallest (18) and the largest
# of the ranges, odd ones, ragged tiles, shifts, padding, periodic copies, both layouts
CASES = {
    "open-100-72-50": ((100, 72, 50), [[U, U]] * 3, 1),
    "open-18-21-25": ((18, 21, 25), [[U, U]] * 3, 1),
    "periodic-36-45-27": ((36, 45, 27), [[P, P]] * 3, 1),
    "periodic-node-181-51-37": ((181, 51, 37), [[P, P]] * 3, 0),
    "wide-radix-252-14-15": ((252, 30, 18), [[P, P], [P, P], [P, P]], 1),
    "long-x-1500": ((1500, 18, 20), [[P, P]] * 3, 1),
    "long-y-1470": ((40, 1470, 18), [[P, P]] * 3, 1),
    "long-z-2000": ((36, 20, 2000), [[P, P]] * 3, 1),
    "walls-ee-oo-eo": ((60, 100, 36), [[E, E], [O, O], [E, O]], 1),
    "walls-oe-eo-ee": ((72, 36, 90), [[O, E], [E, O], [E, E]], 1),
    "walls-node": ((101, 61, 46), [[E, E], [O, O], [E, E]], 0),
    "walls-node-oo-eo": ((49, 73, 37), [[O, O], [E, O], [O, E]], 0),
    "semi-x": ((50, 36, 18), [[E, U], [P, P], [U, U]], 1),
    "semi-unb-odd": ((36, 50, 18), [[U, O], [P, P], [U, E]], 1),
    "semi-node": ((46, 37, 37), [[U, E], [O, U], [P, P]], 0),
    "y-after-walls": ((36, 100, 50), [[E, E], [P, P], [U, U]], 1),
    "y-unb-after-walls": ((36, 45, 50), [[O, O], [U, U], [P, P]], 1),
    "node-per-y-after-walls": ((37, 101, 51), [[E, E], [P, P], [P, P]], 0),
    "x-last": ((50, 36, 60), [[U, U], [E, E], [O, O]], 1),
    "x-c2c": ((45, 36, 50), [[U, U], [P, P], [U, U]], 1),
    "x-c2c-node": ((46, 37, 51), [[U, U], [P, P], [P, P]], 0),
    "channel-120-50-90": ((120, 50, 90), [[P, P], [E, E], [P, P]], 1),
    "plane-200-150": ((200, 150, 1), [[U, U], [U, U], [X, X]], 1),
    "ragged-tile-21": ((42, 36, 50), [[P, P], [E, O], [U, U]], 1),
}


def solve(nglob, bc, center, rhs, lda=1, typ=0, fp32=False, off=0):
    h = [1.0 / (max(nglob) - (1 - center))] * 3
    L = [h[0] * max(m - (1 - center), 1) for m in nglob]
    topo = fl.Topology(0, lda, list(nglob), [1, 1, 1], False)
    s = fl.Solver(topo, bc, h, L, order_diff=1 if typ else 0, center_type=[center] * 3)
    s.set_green_type(0)
    if fp32:
        s.set_precision(True)
    s.setup()
    n = rhs.size
    flat = np.zeros(n + 1)
    flat[off:off + n] = rhs.ravel()
    din, dout = fl.DeviceArray.from_numpy(flat), fl.DeviceArray((n + 1,))
    fl.lib().flups_clear_last_error()
    fl.lib().flups_solve(s._solver, dout.ptr + 8 * off, din.ptr + 8 * off, typ)
    assert fl.last_error() == "", fl.last_error()
    return dout.numpy()[off:off + n].reshape(rhs.shape), s.pass_kernels, h, L


def field(nglob, lda, seed=17):
    rhs = np.random.default_rng(seed).normal(size=(lda, nglob[2], nglob[1], nglob[0]))
    return rhs - rhs.mean(axis=(1, 2, 3), keepdims=True)


@pytest.mark.parametrize("name", CASES)
def test_smooth_passes(name, monkeypatch):
    """every pass on its own kernel, and with the last direction fused, against the generic kernel and the oracle"""
    nglob, bc, center = CASES[name]
    rhs = field(nglob, 1)
    fused, kf, h, L = solve(nglob, bc, center, rhs)
    monkeypatch.setenv("FLUPS_FORCE_GENERIC", "1")
    single, ks, _, _ = solve(nglob, bc, center, rhs, off=1)   # rows 8 bytes off a 16-byte boundary
    monkeypatch.setenv("FLUPS_GENERIC_PASS", "1")
    gen, kg, _, _ = solve(nglob, bc, center, rhs)
    assert 0 not in kf and 0 not in ks and all(k <= 0 for k in kg), (kf, ks, kg)
    ora = orc.solve(list(nglob), bc, 1, h, L, center, 0, rhs)
    for what, got in (("fused", fused), ("passes", single), ("generic", gen)):
        e2, ei = rel_err(got, ora)
        assert e2 <= TOL and ei <= TOL, (what, e2, ei)


@pytest.mark.parametrize("name", ["open-100-72-50", "walls-ee-oo-eo", "x-c2c-node", "channel-120-50-90", "y-unb-after-walls"])
def test_smooth_passes_fp32_storage(name):
    nglob, bc, center = CASES[name]
    rhs = field(nglob, 1)
    got, kinds, h, L = solve(nglob, bc, center, rhs, fp32=True)
    assert 0 not in kinds, kinds
    e2, ei = rel_err(got, orc.solve(list(nglob), bc, 1, h, L, center, 0, rhs))
    assert e2 <= 1e-5 and ei <= 1e-5, (e2, ei)


@pytest.mark.parametrize("bc", [[[U, U]] * 3, [[P, P], [P, P], [U, U]], [[P, P]] * 3])
def test_smooth_passes_three_components(bc):
    """STD and ROT solves of three components at smooth lengths"""
    nglob = (36, 50, 45)
    rhs = field(nglob, 3)
    for typ in (0, 1):
        got, _, h, L = solve(nglob, bc, 1, rhs, lda=3, typ=typ)
        ora = orc.solve(list(nglob), bc, 3, h, L, 1, 0, rhs, typ, 1 if typ else 0)
        e2, ei = rel_err(got, ora)
        assert e2 <= TOL and ei <= TOL, (typ, e2, ei)
