"""Device memory of the general path with its last direction fused: what a request is admitted with bounds what its
solver holds, and no array is held that no solve uses."""
import numpy as np
import pytest

try:
    import torch  # noqa: F401
except Exception:   # pragma: no cover
    torch = None

import flups_amd as fl

pytestmark = pytest.mark.gpu

E, O, P, U, X = 0, 1, 3, 4, 9
# (nglob, bc, lda, rotational, fp32): the fused last direction of every kind, and vector problems whose rotational solve
# is not fused (walls; columns whose three components do not fit a block), sizes at which its compressed
# Green's function is well above the bound's slack of 4 MiB
CASES = {
    "open-200-144-100": ((200, 144, 100), [[U, U]] * 3, 1, False, False),
    "open-200-144-100-fp32": ((200, 144, 100), [[U, U]] * 3, 1, False, True),
    "layer-256-256-128": ((256, 256, 128), [[P, P], [P, P], [U, U]], 1, False, False),
    "walls-x-160-120-100": ((160, 120, 100), [[E, E], [P, P], [U, U]], 1, False, False),
    "corner-r2c-160-120-100": ((160, 120, 100), [[O, O], [E, E], [U, U]], 1, False, False),
    "plane-1000": ((1000, 1000, 1), [[U, U], [U, U], [X, X]], 1, False, False),
    "rot-open-100-96-90": ((100, 96, 90), [[U, U]] * 3, 3, True, False),
    "rot-walls-120-100-90": ((120, 100, 90), [[O, O], [P, P], [U, U]], 3, True, False),
    "rot-open-64-64-675": ((64, 64, 675), [[U, U]] * 3, 3, True, False),
}


@pytest.mark.parametrize("name", CASES)
def test_request_bytes_bound_what_is_held(name):
    nglob, bc, lda, rot, fp32 = CASES[name]
    h = [1.0 / max(nglob)] * 3
    r = fl.ServeRequest.make(nglob, bc, h, [h[0] * m for m in nglob], green=0, lda=lda, fp32=fp32,
                             solver_type=1 if rot else 0, order_diff=1 if rot else 0)
    bound = r.device_bytes()
    b = fl.Batch([r], [fl.DeviceArray(r.shape())], [fl.DeviceArray(r.shape())])
    assert b.device_bytes() <= bound, (b.device_bytes(), bound)


@pytest.mark.parametrize("nglob,bc,lda", [((40, 36, 50), [[U, U]] * 3, 1), ((36, 40, 45), [[P, P], [P, P], [U, U]], 3),
                                          ((36, 45, 50), [[O, O], [E, E], [U, U]], 1), ((72, 90, 1), [[U, U], [U, U], [X, X]], 1)])
def test_steps_and_solves_of_a_fused_solver(nglob, bc, lda):
    """the advanced interface's steps and the allocation-free solve on a solver without the last stage array"""
    rot = lda == 3
    h = [1.0 / max(nglob)] * 3
    s = fl.Solver(fl.Topology(0, lda, list(nglob), [1, 1, 1], False), bc, h, [h[0] * m for m in nglob], order_diff=1 if rot else 0)
    s.set_green_type(0)
    s.setup()
    assert s.path == 3
    rhs = np.random.default_rng(3).normal(size=(lda, nglob[2], nglob[1], nglob[0]))
    din, dref, dout = fl.DeviceArray.from_numpy(rhs), fl.DeviceArray(rhs.shape), fl.DeviceArray(rhs.shape)
    for typ in (0, 1) if rot else (0,):
        s.solve(dref, din, typ)
        fl.lib().flups_clear_last_error()
        fl.lib().flups_solve_noalloc(s._solver, dout.ptr, din.ptr, typ)
        assert fl.last_error() == "", fl.last_error()
        ref = dref.numpy()
        assert np.array_equal(dout.numpy(), ref)
        inner, phys, out = s.inner_buffer(), s.inner_topo_physical(), np.zeros_like(rhs)
        s.do_copy(phys, rhs, fl.FORWARD)
        s.do_fft(inner, fl.FORWARD)
        s.do_mult(inner, typ)
        s.do_fft(inner, fl.BACKWARD_DIFF if typ else fl.BACKWARD)
        s.do_copy(phys, out, fl.BACKWARD)
        assert np.max(np.abs(out - ref)) <= 1e-12 * np.max(np.abs(ref))
