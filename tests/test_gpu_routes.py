"""Which kernels a solve launches: the z pass of the fused pipeline under each schedule (row pairs in one block or
not), and the fused rotational last direction of the general path."""
import ctypes

import numpy as np
import pytest

try:
    import torch  # noqa: F401
except Exception:   # pragma: no cover
    torch = None

import flups_amd as fl
from tests.test_gpu_parity import TOL, rel_err
from tests.test_gpu_rot import GENERAL, field as rot_field, solve as rot_solve

pytestmark = pytest.mark.gpu

O, P, U = 1, 3, 4
# columns of 1120 points (three components and one column take 53760 of 54272 bytes), 1024, and 945 of a full column
LONG = {
    "z-560": ((20, 18, 560), [[U, U]] * 3, 1, 1),
    "z-512": ((20, 18, 512), [[P, P], [P, P], [U, U]], 1, 2),
    "periodic-z-945": ((18, 20, 945), [[P, P]] * 3, 1, 1),
}
# 1350 points: no tile fits; walls: their derivative is no multiplication by i K
NOT_FUSED = {
    "z-675": GENERAL["z-675"],
    "walls-z-40": ((24, 20, 40), [[O, O], [P, P], [U, U]], 1, 1),
}
ROT = {**GENERAL, **LONG, **NOT_FUSED}


class KernelNode(ctypes.Structure):   # hipKernelNodeParams
    _fields_ = [("block", ctypes.c_uint * 3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p), ("grid", ctypes.c_uint * 3),
                ("params", ctypes.c_void_p), ("shared", ctypes.c_uint)]


def launches(solver, nglob):
    """(grid, block) x extents of one solve's launches, in order: a captured flups_solve_noalloc"""
    hip = fl.lib()   # the HIP runtime that the library is linked with
    stream = fl.Stream()
    solver.set_stream(stream)
    h = ctypes.c_void_p(stream.handle)
    din, dout = fl.DeviceArray((1,) + nglob[::-1]), fl.DeviceArray((1,) + nglob[::-1])
    graph, n = ctypes.c_void_p(), ctypes.c_size_t(0)
    assert hip.hipStreamBeginCapture(h, 2) == 0
    hip.flups_clear_last_error()
    hip.flups_solve_noalloc(solver._solver, dout.ptr, din.ptr, 0)
    err = fl.last_error()
    assert hip.hipStreamEndCapture(h, ctypes.byref(graph)) == 0
    assert err == "", err
    assert hip.hipGraphGetNodes(graph, None, ctypes.byref(n)) == 0
    nodes = (ctypes.c_void_p * n.value)()
    assert hip.hipGraphGetNodes(graph, nodes, ctypes.byref(n)) == 0
    out = []
    for node in nodes:
        k = KernelNode()
        assert hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(k)) == 0
        out.append((int(k.grid[0]), int(k.block[0])))
    assert hip.hipGraphDestroy(graph) == 0
    solver.set_stream(None)
    return out


@pytest.mark.parametrize("nglob,small", [((32, 32, 32), True), ((64, 64, 64), True), ((128, 64, 32), True), ((128, 128, 256), False)])
def test_schedule_is_what_runs(monkeypatch, nglob, small):
    """the mirror rows of the z pass lie in neighbouring blocks where the field is small and in one block where it is large,
    the other way round with bit 5 of the schedule; the schedule that a solver reports launches what the
    solver launches; x slabs do as the whole field does; the results are the same bits"""
    def run(env):
        for k in ("FLUPS_ZSCHED", "FLUPS_YSCHED", "FLUPS_ORDER", "FLUPS_SLAB_MB"):
            monkeypatch.delenv(k, raising=False)
        for k, v in env.items():
            monkeypatch.setenv(k, str(v))
        s = fl.Solver(fl.Topology(0, 1, list(nglob), [1, 1, 1], False), [[U, U]] * 3, [1.0 / 64] * 3, [n / 64 for n in nglob])
        s.set_green_type(2)
        if not small:
            s.set_precision(True)   # the stage arrays of a captured solve: 128 MiB at most
        s.setup()
        assert s.path == (1 if small else 2)
        s.solve(out, rhs)
        results.append(out.numpy())
        return [g for g, _ in launches(s, nglob)], s.schedule

    results = []
    rhs = fl.DeviceArray.from_numpy(np.random.default_rng(2).normal(size=(1,) + nglob[::-1]))
    out = fl.DeviceArray((1,) + nglob[::-1])
    default, sched = run({})
    assert len(default) == 5
    assert run({"FLUPS_ZSCHED": sched[0]})[0] == default
    for z in (0, 4, 8, 16, 20):
        own, other = run({"FLUPS_ZSCHED": z})[0], run({"FLUPS_ZSCHED": z | 32})[0]
        apart, pairs = (own, other) if small else (other, own)
        assert apart[2] == 2 * pairs[2], (z, own, other)
    # x slabs (whole tiles): as many blocks in all as the whole field takes
    slabs = run({"FLUPS_SLAB_MB": 0.25, "FLUPS_ZSCHED": 20})[0]
    assert len(slabs) > 5
    assert sum(slabs[2:-1:3]) == default[2], (slabs, default)
    assert all(np.array_equal(r, results[0]) for r in results)


@pytest.mark.parametrize("fp32", [False, True], ids=["fp64", "fp32"])
@pytest.mark.parametrize("name", ROT)
def test_rotational_last_direction_is_fused(name, fp32):
    """the curl runs inside the last direction (two passes, the fused one, two passes) wherever its columns fit a block, and
    as three passes, the multiply and three passes where they do not"""
    nglob, bc, center, odiff = ROT[name]
    h = [1.0 / (max(nglob) - (1 - center))] * 3
    r = fl.ServeRequest.make(nglob, bc, h, [h[0] * (m - (1 - center)) for m in nglob], green=0, lda=3, center=center, fp32=fp32,
                             solver_type=1, order_diff=odiff)
    b = fl.Batch([r], [fl.DeviceArray(r.shape())], [fl.DeviceArray(r.shape())])
    n = b.launches(False)
    assert n >= 7 if name in NOT_FUSED else n == 5, n


@pytest.mark.parametrize("fp32", [False, True], ids=["fp64", "fp32"])
@pytest.mark.parametrize("name", LONG)
def test_rotational_columns_of_one_per_block(name, fp32):
    """the longest columns that fit: one per block"""
    nglob, bc, center, odiff = LONG[name]
    got, path, ora = rot_solve(nglob, bc, center, odiff, rot_field(nglob), fp32)
    assert path == (5 if fp32 else 3)
    e2, ei = rel_err(got, ora)
    assert max(e2, ei) <= (1e-5 if fp32 else TOL), (e2, ei)
