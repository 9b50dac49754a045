"""The work this framework is used for, as cases that can be timed and checked.

Most cases are one segment of a restarted run, which is how a program with
time limits, sweeps or checkpoints uses the library: the held state (the
fields a cycle carries over, in pinned host memory) is uploaded into a context
that was created once, the problem advances by a number of cycles, and the
same fields come back.  The held state is the Sedov blast of the reference
after `warm` cycles; its energy multiplier is drawn from the seed, so every
seed is another trajectory.  The other entry points are the dt constraints on
arrays the caller holds on the device (lgpu_time_constraints_noalloc).

The FP64 forms return what the library returns.  The mixed form's fields carry
FP32 accuracy and are kept in FP32, as a program that writes snapshots of such
a run does.

exact() is the same physics in 64 bits in plain torch, without this package
(lulesh.cc:166-222, 494-2596; a repeat count of the equation of state repeats
identical work, so the region layout does not enter).
"""
import ctypes
import math

import numpy as np
import torch

import lulesh_amd as la

#: The fields a cycle carries over (lulesh.h:266-367).
STATE = ["x", "y", "z", "xd", "yd", "zd", "e", "p", "q", "v", "ss"]
NODAL = STATE[:6]
TIMES = ["time", "deltatime", "dtcourant", "dthydro"]
PRECISION = {"fp64": la.FP64, "mixed": la.MIXED, "fma": la.FP64_FMA}


def listed():
    run = dict(kind="device", regions=11, balance=1, cost=1, precision="fp64")
    return [
        # the dt constraints alone, on the caller's own arrays: one small call
        dict(name="constraints_s45", kind="constraints", n=45 ** 3, list=False),
        # the smallest run in the tests: only launches and latency
        dict(run, name="s8_fp64", s=8, warm=10, cycles=20),
        # the reference's default problem
        dict(run, name="s30_fp64", s=30, warm=60, cycles=100),
        # the reference's usual larger problem, its loop on the host: TimeIncrement
        # and a read-back of dt every cycle
        dict(run, name="s45_fp64_hostloop", kind="host", s=45, warm=40, cycles=60),
        # an odd size with an uneven region layout and dear materials, mixed form
        dict(run, name="s63_mixed", s=63, regions=16, balance=3, cost=4, precision="mixed", warm=60, cycles=100),
        # a mesh that is not taken as a brick: the gather kernels
        dict(run, name="s64_generic", kind="generic", s=64, warm=20, cycles=40),
        # the middle of the range, with fused multiply-adds
        dict(run, name="s96_fma", s=96, precision="fma", warm=100, cycles=100),
        # a middle size that fits no tile, few regions
        dict(run, name="s101_fp64", s=101, regions=5, cost=0, warm=60, cycles=100),
        # the headline workload: load-imbalanced regions at s=192
        dict(run, name="s192_r21_fp64", s=192, regions=21, balance=2, cost=2, warm=200, cycles=200),
        # the mixed form's workload
        dict(run, name="s192_r11_mixed", s=192, precision="mixed", warm=200, cycles=200),
        # 64 problems of 16..64 elements per edge advanced together
        dict(name="ensemble64_fp64", kind="ensemble", members=64, lo=16, hi=64, draw=1234, precision="fp64",
             warm=20, cycles=40),
        # a sweep of small problems, mixed form
        dict(name="ensemble24_mixed", kind="ensemble", members=24, lo=5, hi=24, draw=77, precision="mixed",
             warm=10, cycles=30),
    ]


def draw(rng):
    def log_int(lo, hi):
        return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))

    kind = rng.choice(["device"] * 5 + ["host", "generic", "ensemble", "ensemble", "constraints"])
    if kind == "constraints":
        return dict(kind=kind, n=log_int(64, 100 ** 3), list=rng.random() < 0.5)
    precision = rng.choice(["fp64", "fp64", "mixed", "fma"])
    if kind == "ensemble":
        lo = rng.randint(4, 24)
        return dict(kind=kind, members=rng.randint(2, 40), lo=lo, hi=lo + rng.randint(4, 30),
                    draw=rng.randrange(1 << 20), precision=precision, warm=rng.randint(4, 10),
                    cycles=rng.randint(10, 30))
    s = log_int(5, 72 if kind == "generic" else 140)
    return dict(kind=kind, s=s, regions=rng.choice([1, 5, 11, 16, 21]), balance=rng.randint(1, 3),
                cost=rng.randint(0, 4), precision=precision, warm=rng.randint(4, max(5, min(80, 2 * s))),
                cycles=rng.randint(10, max(12, min(100, 4 * s))))


def _multiplier(rng):
    return float(np.exp(rng.uniform(math.log(0.5), math.log(2.0))))


def _members(case):
    """Sizes, balances and costs of an ensemble: part of the case, not of the seed."""
    r = np.random.RandomState(case["draw"])
    n = case["members"]
    return (r.randint(case["lo"], case["hi"] + 1, n).astype(np.int32), r.randint(1, 3, n).astype(np.int32),
            r.randint(1, 3, n).astype(np.int32))


def _constraint_arrays(case, seed, device):
    """ss, vdov, arealg as a blast has them: a part of the mesh at rest."""
    g = np.random.RandomState(seed)
    n = case["n"]
    ss = g.uniform(0.1, 3.0, n) * 1e3
    vdov = g.standard_normal(n) * 10.0 ** g.uniform(-2, 3, n)
    vdov[g.random_sample(n) < 0.3] = 0.0
    area = g.uniform(0.5, 1.5, n) * 1.125 / 45
    lists = torch.from_numpy(g.permutation(n)[: max(1, (3 * n) // 4)].astype(np.int32)) if case["list"] else None
    return ([torch.from_numpy(a).to(device) for a in (ss, vdov, area)],
            None if lists is None else lists.to(device))


class _State:
    pass


def _pinned(n):
    return torch.empty(n, dtype=torch.float64, pin_memory=True)


def _context(st):
    """The lgpu_ctx of the program's problem."""
    return st.problem.device() if st.kind == "host" else st.problem.ptr


def _copy(st, call, buffers):
    ctx = _context(st)
    for f, ptr in buffers:
        la.check(call(ctx, f, ctypes.cast(ptr, ctypes.POINTER(ctypes.c_double))), ctx)


def _copy_members(st, call, buffers):
    for f, ptr, starts in buffers:
        for m, at in enumerate(starts):
            la.check(call(st.problem.dev, m, f, ctypes.cast(ptr + 8 * at, ctypes.POINTER(ctypes.c_double))))


def prepare(case, seed):
    st = _State()
    st.kind = case["kind"]
    if st.kind == "constraints":
        st.arrays, st.elems = _constraint_arrays(case, seed, "cuda")
        st.out = torch.empty(2, dtype=torch.float64, device="cuda")
        return st
    rng = np.random.RandomState(seed)
    st.precision = case["precision"]
    prec = PRECISION[st.precision]
    lib = la.gpu_lib()
    if st.kind == "ensemble":
        sizes, balances, costs = _members(case)
        st.problem = la.Ensemble(sizes, np.array([_multiplier(rng) for _ in sizes]), balances, costs, precision=prec)
        st.times = st.problem.time_states()
        la.check(lib.lgpu_ensemble_run(st.problem.dev, st.times, case["warm"], None))
        nodes, elems = (sizes.astype(np.int64) + 1) ** 3, sizes.astype(np.int64) ** 3
    else:
        s = case["s"]
        args = (s, case["regions"], case["balance"], case["cost"], _multiplier(rng))
        if st.kind == "host":
            st.problem = la.HostDomain(*args)
            st.problem.attach_device(prec)
            la.check(st.problem.run(case["warm"]))
            st.times = {n: st.problem.get(n) for n in TIMES + ["cycle"]}
        else:
            flags = la.native.FLAG_GENERIC if st.kind == "generic" else 0
            st.problem = la.SedovDevice(*args, precision=prec, flags=flags)
            la.check(st.problem.run(case["warm"]))
            st.times = la.TimeState.from_buffer_copy(st.problem.ts)
        nodes, elems = np.array([(s + 1) ** 3]), np.array([s ** 3])
    st.cycles = case["cycles"]
    st.end = case["warm"] + case["cycles"]

    # the held state, and the buffers the results come back in
    count = {f: int((nodes if f in NODAL else elems).sum()) for f in STATE}
    starts = {f: np.concatenate([[0], np.cumsum(nodes if f in NODAL else elems)[:-1]]).tolist() for f in STATE}
    st.held = {f: _pinned(count[f]) for f in STATE}
    st.result = {f: _pinned(count[f]) for f in STATE}
    st.narrow = {f: torch.empty(count[f], dtype=torch.float32) for f in STATE} if st.precision == "mixed" else None
    many = st.kind == "ensemble"

    def places(held):
        return [(la.FIELDS.index(f), t.data_ptr()) + ((starts[f],) if many else ()) for f, t in held.items()]

    st.upload, st.download = places(st.held), places(st.result)
    if many:
        _copy_members(st, lib.lgpu_ensemble_download, st.upload)
    else:
        _copy(st, lib.lgpu_download, st.upload)
    return st


def run(st):
    lib = la.gpu_lib()
    if st.kind == "constraints":
        ss, vdov, area = st.arrays
        la.check(lib.lgpu_time_constraints_noalloc(
            ss.data_ptr(), vdov.data_ptr(), area.data_ptr(), st.elems.data_ptr() if st.elems is not None else None,
            st.elems.numel() if st.elems is not None else ss.numel(), 2.0, 0.1, st.out.data_ptr(),
            torch.cuda.current_stream().cuda_stream))
        return st.out
    if st.kind == "ensemble":
        _copy_members(st, lib.lgpu_ensemble_upload, st.upload)
        ts = (la.TimeState * st.problem.n).from_buffer_copy(st.times)
        la.check(lib.lgpu_ensemble_run(st.problem.dev, ts, st.end, None))
        _copy_members(st, lib.lgpu_ensemble_download, st.download)
        times = {n: torch.tensor([getattr(t, n) for t in ts], dtype=torch.float64) for n in TIMES}
        cycle = torch.tensor([t.cycle for t in ts])
    else:
        _copy(st, lib.lgpu_upload, st.upload)
        if st.kind == "host":
            d = st.problem
            for n, v in st.times.items():
                d.set(n, v)
            la.check(d.run(st.end))
            times, cycle = {n: d.get(n) for n in TIMES}, int(d.get("cycle"))
        else:
            d = st.problem
            d.ts = la.TimeState.from_buffer_copy(st.times)
            la.check(d.run(st.cycles))
            times, cycle = {n: d.get(n) for n in TIMES}, d.ts.cycle
        _copy(st, lib.lgpu_download, st.download)
    if st.narrow is not None:
        for f in STATE:
            st.narrow[f].copy_(st.result[f])
    return {**(st.narrow if st.narrow is not None else st.result), **times, "cycle": cycle}


def _mean_repeats(s, regions, balance, cost):
    """Mean repeat count of the equation of state over the elements, from the
    expected region sizes (weights (i+1)^balance, lulesh-init.cc:401-510)."""
    w = [(i + 1.0) ** balance for i in range(regions)]
    rep = [1 if i < regions // 2 else 1 + cost if i < regions - (regions + 15) // 20 else 10 * (1 + cost)
           for i in range(regions)]
    return sum(a * b for a, b in zip(w, rep)) / sum(w)


def work(case):
    if case["kind"] == "constraints":
        n = case["n"]
        m = max(1, (3 * n) // 4) if case["list"] else n
        return {"bytes": (28 if case["list"] else 24) * m + 16, "flops": 12 * m}
    if case["kind"] == "ensemble":
        sizes, balances, costs = _members(case)
        problems = [(int(s), 11, int(b), int(c)) for s, b, c in zip(sizes, balances, costs)]
    else:
        problems = [(case["s"], case["regions"], case["balance"], case["cost"])]
    pqs = 4 if case["precision"] == "mixed" else 8
    byts = flops = 0.0
    for s, regions, balance, cost in problems:
        n, e = (s + 1) ** 3, s ** 3
        # a cycle reads and writes positions and velocities, p, q, ss, e and v
        # once, and reads the masses, volo and the symmetry mask
        byts += case["cycles"] * (n * (2 * 48 + 8 + 1) + e * (2 * (16 + 3 * pqs) + 16))
        # the held state in, the result out, on host and device
        byts += 4 * (48 * n + (16 + 3 * pqs) * e)
        # reference formulas: nodal forces and update 1,821, kinematics and Q
        # 900, dt and material 60, one pass of the equation of state 90
        flops += case["cycles"] * e * (1821 + 900 + 60 + 90 * _mean_repeats(s, regions, balance, cost))
    return {"bytes": byts, "flops": flops}


# ---------------------------------------------------------------------------
# The physics in 64 bits, in plain torch.  Node fields are (s+1)^3 arrays in
# z, y, x order, element fields flat; a corner array is (8, E) in the hex
# numbering of lulesh-init.cc:252-259.

_OFFSETS = [(0, 0, 0), (0, 0, 1), (0, 1, 1), (0, 1, 0), (1, 0, 0), (1, 0, 1), (1, 1, 1), (1, 1, 0)]
_FACES = [(0, 1, 2, 3), (0, 4, 5, 1), (1, 5, 6, 2), (2, 6, 7, 3), (3, 7, 4, 0), (4, 7, 6, 5)]
_AREA_FACES = [(0, 1, 2, 3), (4, 5, 6, 7), (0, 1, 5, 4), (1, 2, 6, 5), (2, 3, 7, 6), (3, 0, 4, 7)]
_VOLUDER = {0: (1, 2, 3, 4, 5, 7), 3: (0, 1, 2, 7, 4, 6), 2: (3, 0, 1, 6, 7, 5), 1: (2, 3, 0, 5, 6, 4),
            4: (7, 6, 5, 0, 3, 1), 5: (4, 7, 6, 1, 0, 2), 6: (5, 4, 7, 2, 1, 3), 7: (6, 5, 4, 3, 2, 0)}
_GAMMA = [[1, 1, -1, -1, -1, -1, 1, 1], [1, -1, -1, 1, -1, 1, 1, -1], [1, -1, 1, -1, 1, -1, 1, -1],
          [-1, 1, -1, 1, 1, -1, 1, -1]]


def _corners(a):
    """(3, s+1, s+1, s+1) -> (3, 8, E)."""
    s = a.shape[1] - 1
    return torch.stack([a[:, k:k + s, j:j + s, i:i + s].reshape(3, -1) for k, j, i in _OFFSETS], 1)


def _sum_to_nodes(f, s):
    out = torch.zeros((3, s + 1, s + 1, s + 1), dtype=f.dtype, device=f.device)
    for c, (k, j, i) in enumerate(_OFFSETS):
        out[:, k:k + s, j:j + s, i:i + s] += f[:, c].reshape(3, s, s, s)
    return out


def _cross(a, b):
    return torch.stack([a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]])


def _dot(a, b):
    return (a * b).sum(0)


def _volume(X):
    def triple(u, v, w):
        return _dot(u, _cross(v, w))

    d = lambda a, b: X[:, a] - X[:, b]  # noqa: E731
    return (triple(d(3, 1) + d(7, 2), d(6, 3), d(2, 0)) + triple(d(4, 3) + d(5, 7), d(6, 4), d(7, 0)) +
            triple(d(1, 4) + d(2, 5), d(6, 1), d(5, 0))) / 12.0


def _nodal(st, dt):
    """LagrangeNodal, lulesh.cc:1223-1269."""
    X, U = _corners(st["x"]), _corners(st["u"])
    normal = torch.zeros_like(X)
    for f in _FACES:
        a, b, c, d = (X[:, n] for n in f)
        area = 0.25 * _cross(0.5 * (d + c - b - a), 0.5 * (c + b - d - a))
        for n in f:
            normal[:, n] += area
    force = _sum_to_nodes((st["p"] + st["q"]) * normal, st["s"])
    deriv = torch.empty_like(X)
    for n, (a, b, c, d, e, g) in _VOLUDER.items():
        def form(p, q):
            return ((p[b] + p[c]) * (q[a] + q[b]) - (p[a] + p[b]) * (q[b] + q[c]) + (p[a] + p[e]) * (q[d] + q[e]) -
                    (p[d] + p[e]) * (q[a] + q[e]) - (p[c] + p[g]) * (q[d] + q[g]) + (p[d] + p[g]) * (q[c] + q[g]))
        x, y, z = X
        deriv[0, n], deriv[1, n], deriv[2, n] = form(y, z) / 12.0, -form(x, z) / 12.0, -form(y, x) / 12.0
    determ = st["volo"] * st["v"]
    coef = -3.0 * 0.01 * st["ss"] * st["mass"] / determ.pow(1.0 / 3.0)
    total = torch.zeros_like(X)
    for g in _GAMMA:
        sign = torch.tensor(g, dtype=X.dtype, device=X.device)[:, None]
        mode = sign - (deriv * (X * sign).sum(1)[:, None]).sum(0) / determ
        total += mode * (mode * U).sum(1)[:, None]
    force += _sum_to_nodes(coef * total, st["s"])
    a = force / st["nodalmass"]
    a[0, :, :, 0] = 0.0
    a[1, :, 0, :] = 0.0
    a[2, 0, :, :] = 0.0
    u = st["u"] + a * dt
    u[u.abs() < 1e-7] = 0.0
    st["u"] = u
    st["x"] = st["x"] + u * dt


def _kinematics(st, dt):
    """CalcLagrangeElements and CalcMonotonicQGradientsForElems,
    lulesh.cc:1504-1757."""
    X, U = _corners(st["x"]), _corners(st["u"])
    volume = _volume(X)
    vnew = volume / st["volo"]
    area2 = torch.zeros_like(volume)
    for a, b, c, d in _AREA_FACES:
        f, g = (X[:, c] - X[:, a]) - (X[:, d] - X[:, b]), (X[:, c] - X[:, a]) + (X[:, d] - X[:, b])
        area2 = torch.maximum(area2, _dot(f, f) * _dot(g, g) - _dot(f, g) ** 2)
    arealg = 4.0 * volume / area2.sqrt()

    def face(A, i, j):
        return 0.25 * (A[:, i].sum(1) - A[:, j].sum(1))

    j, i, k = ([0, 1, 5, 4], [3, 2, 6, 7]), ([1, 2, 6, 5], [0, 3, 7, 4]), ([4, 5, 6, 7], [0, 1, 2, 3])
    dj, di, dk = -face(X, *j), face(X, *i), face(X, *k)
    vol, norm = st["volo"] * vnew, 1.0 / (st["volo"] * vnew + 1e-36)
    grad = []
    for a, du in ((_cross(dj, dk), face(U, *i)), (_cross(dk, di), -face(U, *j)), (_cross(di, dj), face(U, *k))):
        grad.append((vol / (_dot(a, a) + 1e-36).sqrt(), _dot(a * norm, du)))
    # strain rate on the half-step positions
    H = X - 0.5 * dt * U

    def centre(A):
        a, b, g, h = A[:, 6] - A[:, 0], A[:, 5] - A[:, 3], A[:, 7] - A[:, 1], A[:, 4] - A[:, 2]
        return 0.125 * (a + b - g - h), 0.125 * (a - b + g - h), 0.125 * (a + b + g + h)

    hx, he, hz = centre(H)
    ux, ue, uz = centre(U)
    cx, ce, cz = _cross(he, hz), _cross(hz, hx), _cross(hx, he)
    vdov = (_dot(cx, ux) + _dot(ce, ue) + _dot(cz, uz)) / _dot(he, ce)
    return vnew, arealg, vdov, grad


def _pressure(e, comp, vnewc):
    bvc = 2.0 / 3.0 * (comp + 1.0)
    p = bvc * e
    p = torch.where(p.abs() < 1e-7, 0.0, p)
    p = torch.where(vnewc >= 1e9, 0.0, p)
    return p.clamp(min=0.0), bvc


def _sound(e, vol, bvc, p):
    c = 2.0 / 3.0 * e + vol * vol * bvc * p
    return torch.where(c <= 0.1111111e-36, 0.3333333e-18, c.clamp(min=0.1111111e-36).sqrt())


def _elements(st, vnew, arealg, vdov, grad):
    """Monotonic Q, equation of state, volume update and the dt constraints,
    lulesh.cc:1761-2596; returns the latter."""
    s = st["s"]
    phis = []
    for d, (_, delv) in enumerate(grad):
        own = delv.reshape(s, s, s)
        axis = 2 - d
        first, last = own.narrow(axis, 0, 1), own.narrow(axis, 0, 1) * 0.0
        minus = torch.cat([first, own.narrow(axis, 0, s - 1)], axis)
        plus = torch.cat([own.narrow(axis, 1, s - 1), last], axis)
        norm = 1.0 / (own + 1e-36)
        m, p = minus * norm, plus * norm
        phi = torch.minimum(torch.minimum(0.5 * (m + p), 2.0 * m), 2.0 * p).clamp(0.0, 1.0)
        phis.append(phi.reshape(-1))
    rho = st["mass"] / (st["volo"] * vnew)
    lin = quad = 0.0
    for (delx, delv), phi in zip(grad, phis):
        t = (delv * delx).clamp(max=0.0)
        lin, quad = lin + t * (1.0 - phi), quad + t * t * (1.0 - phi * phi)
    ql = torch.where(vdov > 0.0, 0.0, -0.5 * rho * lin)
    qq = torch.where(vdov > 0.0, 0.0, 2.0 / 3.0 * rho * quad)

    vnewc, delv = vnew.clamp(1e-9, 1e9), vnew - st["v"]
    e0, p0, q0 = st["e"], st["p"], st["q"]
    comp, half = 1.0 / vnewc - 1.0, 1.0 / (vnewc - 0.5 * delv) - 1.0
    half = torch.where(vnewc <= 1e-9, comp, half)

    def cut(e):
        return torch.where(e.abs() < 1e-7, 0.0, e).clamp(min=-1e15)

    e = (e0 - 0.5 * delv * (p0 + q0)).clamp(min=-1e15)
    ph, bvc = _pressure(e, half, vnewc)
    q = torch.where(delv > 0.0, 0.0, _sound(e, 1.0 / (1.0 + half), bvc, ph) * ql + qq)
    e = cut(e + 0.5 * delv * (3.0 * (p0 + q0) - 4.0 * (ph + q)))
    p, bvc = _pressure(e, comp, vnewc)
    qt = torch.where(delv > 0.0, 0.0, _sound(e, vnewc, bvc, p) * ql + qq)
    e = cut(e - (7.0 * (p0 + q0) - 8.0 * (ph + q) + (p + qt)) * delv / 6.0)
    p, bvc = _pressure(e, comp, vnewc)
    qn = _sound(e, vnewc, bvc, p) * ql + qq
    q = torch.where(delv <= 0.0, torch.where(qn.abs() < 1e-7, 0.0, qn), q)
    ss = _sound(e, vnewc, bvc, p)
    st.update(e=e, p=p, q=q, ss=ss, v=torch.where((vnew - 1.0).abs() < 1e-10, 1.0, vnew))
    return _constraints(ss, vdov, arealg)


def _constraints(ss, vdov, arealg):
    """CalcTimeConstraintsForElems, lulesh.cc:2447-2596."""
    f = ss * ss + torch.where(vdov < 0.0, 64.0 * 4.0 * (arealg * vdov) ** 2, 0.0)
    moving = vdov != 0.0
    big = torch.tensor(1e20, dtype=ss.dtype, device=ss.device)
    courant = torch.where(moving, arealg / f.sqrt(), big).min()
    hydro = torch.where(moving, 0.1 / (vdov.abs() + 1e-20), big).min()
    return torch.minimum(courant, big), torch.minimum(hydro, big)


def _sedov(s, multiplier, cycles, device):
    """The Sedov problem from its start (lulesh-init.cc:16-194) over `cycles`
    cycles of the main loop."""
    edge = 1.125 * torch.arange(s + 1, dtype=torch.float64, device=device) / s
    z, y, x = torch.meshgrid(edge, edge, edge, indexing="ij")
    st = {"s": s, "x": torch.stack([x, y, z])}
    st["u"] = torch.zeros_like(st["x"])
    st["volo"] = _volume(_corners(st["x"]))
    st["mass"] = st["volo"]
    st["nodalmass"] = _sum_to_nodes((st["volo"] / 8.0).expand(3, 8, -1), s)[0]
    for f in ("e", "p", "q", "ss"):
        st[f] = torch.zeros_like(st["volo"])
    st["v"] = torch.ones_like(st["volo"])
    start = 3.948746e7 * (s / 45.0) ** 3 * multiplier
    st["e"][0] = start
    t = {"time": 0.0, "deltatime": 0.5 * float(st["volo"][0]) ** (1.0 / 3.0) / math.sqrt(2.0 * start),
         "dtcourant": 1e20, "dthydro": 1e20}
    cycle = 0
    while t["time"] < 1e-2 and cycle < cycles:
        # TimeIncrement, lulesh.cc:166-222
        target = 1e-2 - t["time"]
        if cycle:
            old, new = t["deltatime"], 1e20
            if t["dtcourant"] < new:
                new = t["dtcourant"] / 2.0
            if t["dthydro"] < new:
                new = t["dthydro"] * 2.0 / 3.0
            if new / old >= 1.0:
                new = old if new / old < 1.1 else min(new, 1.2 * old)
            t["deltatime"] = min(new, 1e-2)
        dt = t["deltatime"]
        if dt < target < 4.0 * dt / 3.0:
            target = 2.0 * dt / 3.0
        dt = t["deltatime"] = min(dt, target)
        t["time"] += dt
        cycle += 1
        _nodal(st, dt)
        c, h = _elements(st, *_kinematics(st, dt))
        t["dtcourant"], t["dthydro"] = float(c), float(h)
    out = {n: a.reshape(-1) for n, a in zip(NODAL, [*st["x"], *st["u"]])}
    out.update({f: st[f] for f in STATE[6:]})
    return out, t, cycle


def exact(case, seed):
    device = "cuda" if torch.cuda.is_available() else "cpu"
    if case["kind"] == "constraints":
        (ss, vdov, area), elems = _constraint_arrays(case, seed, device)
        if elems is not None:
            ss, vdov, area = (a[elems.long()] for a in (ss, vdov, area))
        return torch.stack(_constraints(ss, vdov, area))
    rng = np.random.RandomState(seed)
    cycles = case["warm"] + case["cycles"]
    sizes = _members(case)[0].tolist() if case["kind"] == "ensemble" else [case["s"]]
    # about 10 ms a cycle, or 60 ns an element of it
    if sum(cycles * max(1e-2, 6e-8 * s ** 3) for s in sizes) > 12.0:
        return None
    got = [_sedov(s, _multiplier(rng), cycles, device) for s in sizes]
    if case["kind"] == "ensemble":
        fields = {f: torch.cat([g[0][f] for g in got]) for f in STATE}
        return {**fields, **{n: torch.tensor([g[1][n] for g in got], dtype=torch.float64) for n in TIMES},
                "cycle": None}
    return {**got[0][0], **got[0][1], "cycle": None}
