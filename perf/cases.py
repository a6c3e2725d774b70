"""Timed workloads of the FLUPS solve path, through the package's public entry points.

A case is one Poisson (STD) or Biot-Savart (ROT) problem as a simulation keeps it: a Solver set up
once, a right-hand side and a field in device memory, one `solve` per time step; or a Batch of
independent problems. `listed()` names the standing cases, `draw()` gives more of the same ranges:
24 to about 320 points per axis (513 at most), cell- and node-centred data, the boundary sets of
BOUNDARY, lda 1 and 3, FP64 and FP32 transforms, solves queued on a caller stream, synchronous
solves on device arrays and on host arrays.
"""
import math

import numpy as np
import torch

import flups_amd as fl

E, O, P, U, X = 0, 1, 3, 4, 9   # EVEN, ODD, PER, UNB, NONE

# boundary sets (x, y, z) and what they stand for
BOUNDARY = {
    "open": [[U, U], [U, U], [U, U]],        # isolated vorticity or charge
    "periodic": [[P, P], [P, P], [P, P]],    # homogeneous turbulence
    "duct": [[P, P], [U, U], [U, U]],        # one periodic direction: wakes, jets
    "layer": [[P, P], [P, P], [U, U]],       # two periodic directions: mixing layers
    "mixed": [[E, O], [P, P], [U, U]],       # symmetric x, periodic y, open z
    "channel": [[P, P], [E, E], [P, P]],     # walls (Neumann) in y
    "corner": [[O, O], [E, E], [U, U]],      # two wall pairs, open z
    "plate": [[E, E], [U, U], [U, U]],       # walls in x, open elsewhere
    "plane": [[U, U], [U, U], [X, X]],       # 2-D open problem
}


def listed():
    return [
        # the smallest standing problem: a coarse open-domain solve inside a time-stepping loop
        dict(name="open64", bc="open", n0=64, n1=64, n2=64),
        # drop-in use from a host code: numpy arrays in and out, each call returns the result
        dict(name="open128_host", bc="open", n0=128, n1=128, n2=128, where="host"),
        # the headline problem of bench.py, FP64 and FP32
        dict(name="open256", bc="open", n0=256, n1=256, n2=256),
        dict(name="open256_fp32", bc="open", n0=256, n1=256, n2=256, fp32=True),
        # decimal grid sizes, unequal axes: the open problem as users size it
        dict(name="open_200x144x100", bc="open", n0=200, n1=144, n2=100),
        # symmetric / periodic / open at the headline size
        dict(name="mixed256", bc="mixed", n0=256, n1=256, n2=256),
        # pressure solve of a channel flow, 3-5-smooth sizes
        dict(name="channel_240x100x180", bc="channel", n0=240, n1=100, n2=180),
        # node-centred walls, ragged odd extents
        dict(name="corner_node_129x161x97", bc="corner", n0=129, n1=161, n2=97, node=True),
        # velocity from vorticity in a doubly periodic layer, three components, FP32 transforms
        dict(name="layer160_rot_fp32", bc="layer", n0=160, n1=160, n2=160, lda=3, fp32=True),
        # 2-D open problem, one synchronous call at a time on device arrays
        dict(name="plane1024_sync", bc="plane", n0=1024, n1=1024, n2=1, where="sync"),
        # velocity from vorticity of a vortex ring, the largest workload of bench.py
        dict(name="open513_node_rot", bc="open", n0=513, n1=513, n2=513, lda=3, node=True),
        # independent small problems of mixed shapes and boundaries, set up once, solved together
        dict(name="batch32", problems=32, mix=11),
    ]


def _smooth(n):
    for p in (2, 3, 5, 7):
        while n % p == 0:
            n //= p
    return n == 1


SMOOTH = [n for n in range(24, 321, 2) if _smooth(n)]


def draw(rng):
    if rng.random() < 0.1:
        return dict(problems=rng.randint(8, 32), mix=rng.randint(0, 10 ** 6))
    bc = rng.choice(list(BOUNDARY))
    if bc == "plane":
        n = [int(math.exp(rng.uniform(math.log(128), math.log(1024)))) // 2 * 2 for _ in range(2)] + [1]
    else:
        c = math.exp(rng.uniform(math.log(32), math.log(240)))
        n = []
        for _ in range(3):
            t = min(max(c * math.exp(rng.uniform(-0.3, 0.3)), 24), 320)
            if rng.random() < 0.85:   # users pick lengths with small factors; some do not
                n.append(min(SMOOTH, key=lambda s: abs(s - t)))
            else:
                n.append(int(t))
    node = bc not in ("plane",) and rng.random() < 0.25
    if node:
        n = [m + 1 for m in n]
    rot = bc in ("open", "duct", "layer", "periodic") and not node and all(m % 2 == 0 for m in n) and rng.random() < 0.3
    case = dict(bc=bc, n0=n[0], n1=n[1], n2=n[2], node=node, lda=3 if rot else 1, fp32=rng.random() < 0.25,
                where=rng.choice(["queued", "queued", "queued", "sync", "host"]))
    return case


# ---------------------------------------------------------------------------
def _problem(case):
    """(shape, bc, h, L, kernel, lda) of a single-problem case; isotropic grids, longest side about 1"""
    n = [case["n0"], case["n1"], case["n2"]]
    node, bc = case.get("node", False), BOUNDARY[case["bc"]]
    h = 1.0 / (max(n) - 1 if node else max(n))
    L = [h * (m - 1 if node and m > 1 else m) for m in n]
    kernel = {"open": fl.GreenType.HEJ_2, "mixed": fl.GreenType.LGF_4}.get(case["bc"], fl.GreenType.CHAT_2)
    return n, bc, h, L, kernel, case.get("lda", 1)


def _mix(case):
    """the single-problem cases of a batch"""
    rng = np.random.default_rng(case["mix"])
    sizes = [32, 48, 64, 80, 96, 112, 128]
    out = []
    for _ in range(case["problems"]):
        n = [int(v) for v in rng.choice(sizes, 3)]
        bc = ["open", "duct", "mixed", "periodic"][int(rng.integers(4))]
        lda = 3 if bc != "mixed" and rng.random() < 0.25 else 1   # three components: Biot-Savart
        out.append(dict(bc=bc, n0=n[0], n1=n[1], n2=n[2], lda=lda))
    return out


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _rhs(case, seed, device):
    """Gaussian blobs (centres in the middle of the box, widths 3-6 % of its longest side, amplitudes
    N(0,1)) with 1e-3 noise, per component; zero mean where no direction is open"""
    n, bc, h, L, _, lda = _problem(case)
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device=device)
    gen.manual_seed(int(seed) & 0x7FFFFFFF)
    off = 0.0 if case.get("node", False) else 0.5
    xs = [(torch.arange(m, device=device, dtype=torch.float64) + off) * h for m in n]
    f = torch.randn((lda, n[2], n[1], n[0]), generator=gen, device=device, dtype=torch.float64)
    f *= 1e-3
    for c in range(lda):
        for _ in range(4):
            sg, amp = rng.uniform(0.03, 0.06), rng.normal()
            g = []
            for d in range(3):
                cen = rng.uniform(0.3, 0.7) * L[d]
                g.append(torch.ones_like(xs[d]) if bc[d][0] == X else torch.exp(-(xs[d] - cen) ** 2 / (2 * sg * sg)))
            f[c].addcmul_(g[2][:, None, None] * g[1][None, :, None], g[0][None, None, :].expand(1, n[1], n[0]), value=amp)
    if not any(b == [U, U] for b in bc):
        f -= f.mean(dim=(1, 2, 3), keepdim=True)
    return f


def _solver(case):
    n, bc, h, L, kernel, lda = _problem(case)
    rot = lda == 3
    topo = fl.Topology(0, lda, n, [1, 1, 1], False)
    center = fl.CenterType.NODE_CENTER if case.get("node", False) else fl.CenterType.CELL_CENTER
    s = fl.Solver(topo, bc, [h] * 3, L, order_diff=fl.DiffType.SPE if rot else fl.DiffType.NOD, center_type=[center] * 3)
    s.set_green_type(kernel)
    if case.get("fp32", False):
        s.set_precision(True)
    s.setup()
    return s


_STREAM = []


def _stream():
    """the stream of the simulation that the solves are queued on"""
    if not _STREAM:
        _STREAM.append(torch.cuda.Stream())
    return _STREAM[0]


def prepare(case, seed):
    torch.cuda.init()   # torch's HIP runtime first, as the package asks
    if "problems" in case:
        reqs, rhs, field = [], [], []
        for i, one in enumerate(_mix(case)):
            n, bc, h, L, kernel, lda = _problem(one)
            reqs.append(fl.ServeRequest.make(n, bc, [h] * 3, L, green=kernel, lda=lda,
                                             solver_type=fl.SolverType.ROT if lda == 3 else fl.SolverType.STD,
                                             order_diff=fl.DiffType.SPE if lda == 3 else fl.DiffType.NOD))
            rhs.append(_rhs(one, seed * 1000 + i, "cuda"))
            field.append(torch.zeros_like(rhs[-1]))
        torch.cuda.synchronize()
        return {"batch": fl.Batch(reqs, rhs, field), "rhs": rhs, "field": field}
    where = case.get("where", "queued")
    rhs = _rhs(case, seed, "cuda")
    if where == "host":
        rhs = rhs.cpu().numpy()
        field = np.zeros_like(rhs)
    else:
        field = torch.zeros_like(rhs)
    torch.cuda.synchronize()
    s = _solver(case)
    if where == "queued":
        s.set_stream(_stream().cuda_stream)
    return {"solver": s, "rhs": rhs, "field": field, "type": fl.SolverType.ROT if case.get("lda", 1) == 3 else fl.SolverType.STD,
            "fp32": case.get("fp32", False), "where": where}


def run(state):
    if "batch" in state:
        state["batch"].run()
        return state["field"]
    field = state["field"]
    state["solver"].solve(field, state["rhs"], state["type"])
    if state["fp32"]:   # a single-precision simulation: the double field goes back into its own arrays
        if state["where"] == "host":
            return field.astype(np.float32)
        if state["where"] == "sync":
            return field.to(torch.float32)
        with torch.cuda.stream(_stream()):
            return field.to(torch.float32)
    return field


# ---------------------------------------------------------------------------
def _transform_length(b, n, node):
    if b == [X, X]:
        return 1
    if b == [U, U]:
        return 2 * (n - 1) if node else 2 * n
    return n


def work(case):
    if "problems" in case:
        w = [work(c) for c in _mix(case)]
        return {"bytes": sum(x["bytes"] for x in w), "flops": sum(x["flops"] for x in w)}
    n, bc, _, _, _, lda = _problem(case)
    node = case.get("node", False)
    N = float(n[0] * n[1] * n[2])
    M = [_transform_length(bc[d], n[d], node) for d in range(3)]
    # the field once in and once out, the Green's function once (one octant where it is even)
    g = 1.0
    for d in range(3):
        g *= M[d] // 2 + 1 if bc[d] in ([U, U], [P, P]) else M[d]
    nbytes = 2.0 * N * 8 * lda + g * (4 if case.get("fp32", False) else 8)
    # real transforms along x, then complex half-spectra: x pencils n1 n2, y pencils (M0/2) n2, z pencils (M0/2) M1,
    # each there and back, 5 n log2 n per complex transform of n points
    half = M[0] / 2.0 + 1

    def fft(m):
        return 5.0 * m * math.log2(m) if m > 1 else 0.0
    flops = 2.0 * lda * (0.5 * fft(M[0]) * n[1] * n[2] + fft(M[1]) * half * n[2] + fft(M[2]) * half * M[1])
    return {"bytes": nbytes, "flops": flops}


# ---------------------------------------------------------------------------
# the same convolution in 64 bits with torch alone: extend the field by the symmetries of its
# boundaries (and by zeros where open) to a periodic box, multiply by the Green's function's spectrum
def _extend(f, dim, b, node):
    m = f.shape[dim]
    if b == [X, X]:
        return f
    if b == [P, P]:
        return f.narrow(dim, 0, m - 1) if node else f
    if b == [U, U]:
        ext = 2 * (m - 1) if node else 2 * m
        shape = list(f.shape)
        shape[dim] = ext - m
        return torch.cat([f, torch.zeros(shape, dtype=f.dtype, device=f.device)], dim)
    r = 1.0 if b[1] == E else -1.0   # reflected in the right boundary
    if node:
        f = f.clone()                # the field vanishes on an odd boundary
        if b[0] == O:
            f.select(dim, 0).zero_()
        if b[1] == O:
            f.select(dim, m - 1).zero_()
        g = torch.cat([f, r * f.narrow(dim, 1, m - 2).flip(dim)], dim)
    else:
        g = torch.cat([f, r * f.flip(dim)], dim)
    return g if b[0] == b[1] else torch.cat([g, -g], dim)   # unlike boundaries: antiperiodic


def _restrict(f, dim, b, n, node):
    if b == [P, P] and node:
        return torch.cat([f, f.narrow(dim, 0, 1)], dim)
    return f.narrow(dim, 0, n)


def _axis_shape(v, d):
    s = [1, 1, 1]
    s[2 - d] = -1
    return v.reshape(s)


def _symbol4(t):
    return 5.0 / 2.0 - 8.0 / 3.0 * torch.cos(t) + 1.0 / 6.0 * torch.cos(2 * t)


def _lattice1d(c, n):
    """g(n) = 1/(2 pi) int cos(n t) / (c + s(t)) dt, s the symbol above, c > 0: with mu = cos t - 1 the
    denominator is (mu - mu1)(mu - mu2) / 3, and 1 / (cos t - w) has the lattice function -lambda^n / sqrt(w^2 - 1)"""
    c = c.to(torch.complex128)
    q = torch.sqrt(9.0 - 3.0 * c)
    mu = [3.0 + q, 3.0 * c / (3.0 + q)]
    g = []
    for m in mu:
        s = torch.sqrt(m * (m + 2.0))
        s = torch.where((1.0 + m - s).abs() > 1.0, -s, s)
        g.append(-(1.0 + m - s) ** n / s)
    return (3.0 / (mu[0] - mu[1]) * (g[0] - g[1])).real


def _green(bc, h, ext, kernel, device):
    """spectrum of h^k G on the extended box, (M2, M1, M0 / 2 + 1), real"""
    sigma = 2.0 * h
    idx = [torch.arange(m, device=device, dtype=torch.float64) for m in ext]
    mir = [torch.minimum(i, m - i) for i, m in zip(idx, ext)]
    opn = [d for d in range(3) if bc[d] == [U, U]]
    per = [d for d in range(3) if d not in opn and bc[d] != [X, X]]
    r2 = sum((_axis_shape((mir[d] * h) ** 2, d) for d in opn), torch.zeros(1, 1, 1, device=device, dtype=torch.float64))
    k2 = torch.zeros(1, 1, 1, device=device, dtype=torch.float64)
    for d in per:   # k^2, or the fourth-order stencil's symbol
        t = mir[d] * (2 * math.pi / ext[d])
        t = t[: ext[0] // 2 + 1] if d == 0 else t
        k2 = k2 + _axis_shape(_symbol4(t) if kernel == fl.GreenType.LGF_4 else (t / h) ** 2, d)
    if len(opn) == 3:
        r = r2.sqrt()
        if kernel == fl.GreenType.HEJ_2:
            g = torch.erf(r / (sigma * math.sqrt(2.0))) / r
            g *= -1.0 / (4.0 * math.pi)
            g[0, 0, 0] = -math.sqrt(2.0) / 4.0 / (sigma * math.sqrt(math.pi ** 3))
        else:
            g = -1.0 / (4.0 * math.pi * r)
            g[0, 0, 0] = -0.5 * (1.5 / (2.0 * math.pi) * h ** 3) ** (2.0 / 3.0) / h ** 3
        g *= h ** 3
        return torch.fft.rfftn(g).real
    if not opn:
        g = -1.0 / k2
        g[0, 0, 0] = 0.0
        return g
    r, k = r2.sqrt(), k2.sqrt()
    zero = torch.zeros_like(r * k)
    if kernel == fl.GreenType.LGF_4:
        g = -h * h * _lattice1d(k2, r / h)
    elif len(opn) == 1:
        g = torch.where(k > 0, -0.5 * torch.exp(-k * r) / torch.where(k > 0, k, 1.0), 0.5 * r + zero) * h
    else:
        req = h / math.sqrt(math.pi)
        kr = (torch.where(k > 0, k, 1.0) * torch.where(r > 0, r, 1.0)).cpu()
        far = -torch.special.modified_bessel_k0(kr).to(device) / (2.0 * math.pi)
        q = torch.where(k > 0, k * req, 1.0).cpu()
        near = (-(1.0 - q * torch.special.modified_bessel_k1(q)) / (math.pi * q * q)).to(device)
        mean = torch.log(torch.where(r > 0, r, 1.0)) / (2.0 * math.pi) + zero
        g = torch.where(k > 0, torch.where(r > 0, far, near + zero), mean)
        g[0, 0, 0] = 0.25 / (2.0 * math.pi) * (math.pi - 6.0 + 2.0 * math.log(0.5 * math.pi * req * req))
        g = g * h * h
    if 0 in opn:
        g = torch.fft.rfft(g, dim=2).real
        opn = [d for d in opn if d != 0]
    return torch.fft.fftn(g, dim=[2 - d for d in opn]).real if opn else g


def _spectrum(f, bc, node):
    g = f
    for d in (2, 1, 0):
        g = _extend(g, 2 - d, bc[d], node)
    shape = [g.shape[2], g.shape[1], g.shape[0]]
    return torch.fft.rfftn(g), shape


def _back(w, ext, bc, n, node):
    w = torch.fft.ifftn(w, dim=[0, 1])
    w = _restrict(_restrict(w, 0, bc[2], n[2], node), 1, bc[1], n[1], node).contiguous()
    w[:, :, 0].imag.zero_()
    if ext[0] % 2 == 0:
        w[:, :, -1].imag.zero_()
    return _restrict(torch.fft.irfft(w, n=ext[0], dim=2), 2, bc[0], n[0], node)


def _wave(d, ext, h, device):
    """wave numbers of one axis, the middle one positive"""
    m = ext[d]
    i = torch.arange(m // 2 + 1 if d == 0 else m, device=device, dtype=torch.float64)
    i = torch.where(i > m / 2.0, i - m, i)
    return _axis_shape(i * (2 * math.pi / (m * h)), d)


def _exact(case, seed):
    n, bc, h, _, kernel, lda = _problem(case)
    node, device = case.get("node", False), _device()
    rhs = _rhs(case, seed, device)
    out = torch.empty_like(rhs)
    w = []
    g = None
    for c in range(lda):
        s, ext = _spectrum(rhs[c], bc, node)
        if g is None:
            g = _green(bc, h, ext, kernel, device)
        s *= g
        w.append(s)
    del g
    if lda == 1:
        out[0] = _back(w[0], ext, bc, n, node)
        return out
    for c in range(3):   # u = i k x psi
        a, b = (c + 1) % 3, (c + 2) % 3
        u = _wave(a, ext, h, device) * w[b]
        u -= _wave(b, ext, h, device) * w[a]
        u *= 1j
        out[c] = _back(u, ext, bc, n, node)
        del u
    return out


def exact(case, seed):
    if "problems" in case:
        return [_exact(c, seed * 1000 + i).cpu() for i, c in enumerate(_mix(case))]
    out = _exact(case, seed).cpu()
    return out.numpy() if case.get("where") == "host" else out
