"""The work this framework is timed on: knn_rms and knn_data through the
public entry points of mdsctk_amd.knn, and the XTC reader in front of them.

Seven kinds of call, each a thing a user's program does:

  trajectory  one trajectory in host memory, made resident and queried
              against itself (what the knn_rms executable does with a file)
  self        a resident set queried against itself, outputs on the device
  cross       query frames on the device against a resident set
  serve       requests of several sizes from host buffers, submitted together
              and waited for
  data        knn_data: FP64 vectors on the host, self or cross
  rows        --sort false: whole distance rows
  xtc         an XTC file decoded into device memory

Frames come from the two generators the tests and the benchmark use: a
random-walk structure with Gaussian noise of a per-frame width ("walk"), and
metastable states with near-duplicate frames ("states").
"""
import ctypes
import math
import os
import tempfile
import weakref

import numpy as np
import torch

from mdsctk_amd import knn

DEV = "cuda"


# ---------------------------------------------------------------------------
# cases


def listed():
    return [
        # the shipped example's shape: one short backbone trajectory, loaded
        # and analysed in one go; launches, allocations and copies count
        dict(name="trajectory_1000x60", kind="trajectory", frames="walk", n_ref=1000, natoms=60,
             k=30, precision="bf16", mass="backbone"),
        # the CPU tool's ordinary workload
        dict(name="self_2000x304", kind="self", frames="walk", n_ref=2000, natoms=304, k=30,
             precision="bf16", mass="uniform"),
        # the graph pipeline's set (kNN graph for the spectral stage)
        dict(name="self_30000x150", kind="self", frames="states", n_ref=30000, natoms=150, k=32,
             precision="bf16", mass="uniform"),
        # the headline workload at full size
        dict(name="self_200000x1000", kind="self", frames="states", n_ref=200000, natoms=1000,
             k=64, precision="bf16", mass="uniform"),
        # plain FP32 form, one trajectory against another
        dict(name="cross_fp32_50000x304", kind="cross", frames="walk", n_ref=50000, n_fit=50000,
             natoms=304, k=100, precision="fp32", mass="uniform", nofit=False),
        # an out-of-sample batch against a large resident set
        dict(name="cross_4096_100000x500", kind="cross", frames="walk", n_ref=100000, n_fit=4096,
             natoms=500, k=50, precision="bf16", mass="uniform", nofit=False),
        # frames that are aligned already (--nofit), ragged sizes, FP16 form
        dict(name="cross_nofit_8191_30011x151", kind="cross", frames="states", n_ref=30011,
             n_fit=8191, natoms=151, k=32, precision="fp16", mass="random", nofit=True),
        # the shortest served request
        dict(name="serve_1_100000x500", kind="serve", frames="walk", n_ref=100000, natoms=500,
             k=50, precision="bf16", mass="uniform", requests="1"),
        # a burst of uneven requests against long frames
        dict(name="serve_burst_20000x2000", kind="serve", frames="walk", n_ref=20000, natoms=2000,
             k=32, precision="bf16", mass="uniform", requests="3,1877,40,1,611,129,17,256"),
        # dihedral sin/cos vectors, every vector against the others
        dict(name="data_self_40007x90", kind="data", n_ref=40007, n_fit=0, vdim=90, k=100,
             precision="bf16", metric="euclidean"),
        # whole rows (--sort false), as the dense matrix builders read them
        dict(name="rows_501_20011x304", kind="rows", frames="walk", n_ref=20011, n_fit=501,
             natoms=304, precision="bf16", mass="backbone", nofit=False),
        # a trajectory file at the usual 1e-3 nm
        dict(name="xtc_10000x304", kind="xtc", frames="walk", n_ref=10000, natoms=304,
             quantum=1000.0),
    ]


# Pair-atoms a drawn query may take (the largest listed case takes 2e13).
_MAX_PAIR_ATOMS = {"bf16": 1.5e13, "fp16": 1.2e13, "fp32": 5e12}


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _frames_case(rng, kind):
    prec = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    return dict(kind=kind, frames=rng.choice(["walk", "states"]), natoms=_log(rng, 10, 2000),
                k=_log(rng, 1, 200), precision=prec,
                mass=rng.choice(["uniform", "backbone", "random"]))


def draw(rng):
    kind = rng.choice(["trajectory", "self", "self", "cross", "cross", "serve", "data", "rows",
                       "xtc"])
    if kind == "trajectory":
        c = _frames_case(rng, kind)
        c.update(n_ref=_log(rng, 100, 5000), natoms=_log(rng, 10, 500))
    elif kind == "self":
        c = _frames_case(rng, kind)
        top = math.sqrt(2 * _MAX_PAIR_ATOMS[c["precision"]] / c["natoms"])
        c["n_ref"] = min(_log(rng, 300, 200000), int(top), int(2e8 / c["natoms"]))
    elif kind == "cross":
        c = _frames_case(rng, kind)
        c["n_ref"] = min(_log(rng, 500, 200000), int(1.5e8 / c["natoms"]))
        top = _MAX_PAIR_ATOMS[c["precision"]] / 4 / c["natoms"] / c["n_ref"]
        c["n_fit"] = max(1, min(_log(rng, 1, 50000), int(top), int(1e8 / c["natoms"])))
        c["nofit"] = rng.random() < 0.25
    elif kind == "serve":
        c = _frames_case(rng, kind)
        c["n_ref"] = min(_log(rng, 5000, 100000), int(6e7 / c["natoms"]))
        c["k"] = _log(rng, 1, 100)
        sizes = [_log(rng, 1, 2048) for _ in range(rng.randint(1, 10))]
        while sum(sizes) > 5000:
            sizes.remove(max(sizes))
        c["requests"] = ",".join(str(s) for s in sizes or [1])
    elif kind == "data":
        c = dict(kind=kind, n_ref=_log(rng, 1000, 60000), n_fit=0, vdim=_log(rng, 8, 1500),
                 k=_log(rng, 1, 200), precision=rng.choice(["bf16", "bf16", "fp32"]),
                 metric=rng.choice(["euclidean", "correlation"]))
        c["n_ref"] = min(c["n_ref"], int(3e7 / c["vdim"]))
        if rng.random() < 0.5:
            c["n_fit"] = min(_log(rng, 1, 20000), int(1e7 / c["vdim"]))
    elif kind == "rows":
        c = dict(kind=kind, frames=rng.choice(["walk", "states"]), n_ref=_log(rng, 500, 20000),
                 natoms=_log(rng, 10, 1000), precision=rng.choice(["bf16", "fp32", "exact"]),
                 mass=rng.choice(["uniform", "backbone", "random"]), nofit=rng.random() < 0.25)
        c["n_fit"] = max(1, min(_log(rng, 16, 2000), int(1.2e7 / c["n_ref"])))
    else:
        c = dict(kind=kind, frames=rng.choice(["walk", "states"]), natoms=_log(rng, 10, 1000),
                 quantum=rng.choice([1000.0, 1000.0, 10000.0]))
        c["n_ref"] = min(_log(rng, 200, 40000), int(4e6 / c["natoms"]))
    return c


# ---------------------------------------------------------------------------
# inputs, from the seed alone


def _gen(seed, stream):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 1009 + stream)
    return g


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device=DEV, dtype=torch.float64)


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32)


def _rotations(n, g):
    u = _rand(g, 3, n)
    a, b = (1 - u[0]).sqrt(), u[0].sqrt()
    w, x = a * torch.sin(2 * math.pi * u[1]), a * torch.cos(2 * math.pi * u[1])
    y, z = b * torch.sin(2 * math.pi * u[2]), b * torch.cos(2 * math.pi * u[2])
    r = [1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w),
         2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w),
         2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)]
    return torch.stack(r, 1).reshape(n, 3, 3)


def _frames(kind, n, natoms, seed, aligned=False):
    """n frames [n, natoms, 3], float32 nm: a random walk of 0.38 nm steps
    with per-frame noise U(0.05, 0.3) nm ("walk"), or 50 states 0.3 nm apart
    with 0.1 nm noise and 5 % near-duplicates at 1e-4 nm ("states"); then a
    random rigid motion (aligned: a small translation only)."""
    g = _gen(seed, 1)
    v = torch.randn(natoms, 3, generator=g, device=DEV, dtype=torch.float64)
    v = v / v.norm(dim=1, keepdim=True)
    v[0] = 0
    base = torch.cumsum(0.38 * v, 0)
    out = torch.empty(n, natoms, 3, device=DEV, dtype=torch.float32)
    step = max(1, min(n, int(2.4e7 // (3 * natoms))))
    if kind == "states":
        centres = base + 0.3 * torch.randn(50, natoms, 3, generator=g, device=DEV,
                                           dtype=torch.float64)
        label = torch.randint(0, 50, (n,), generator=g, device=DEV)
        u, pick = _rand(g, n), _rand(g, n)
        for f0 in range(0, n, step):
            m = min(step, n - f0)
            out[f0:f0 + m] = (centres[label[f0:f0 + m]] + 0.1 * _normal(g, m, natoms, 3)).float()
        # near-duplicates of an earlier frame
        dup = torch.nonzero(u < 0.05).flatten()
        dup = dup[dup > 0]
        src = (pick[dup] * dup).long()
        src = torch.where(u[src] < 0.05, torch.zeros_like(src), src)
        for f0 in range(0, len(dup), step):
            d, s = dup[f0:f0 + step], src[f0:f0 + step]
            out[d] = out[s] + 1e-4 * _normal(g, len(d), natoms, 3)
    else:
        sigma = 0.05 + 0.25 * _rand(g, n, 1, 1)
        for f0 in range(0, n, step):
            m = min(step, n - f0)
            out[f0:f0 + m] = (base + sigma[f0:f0 + m] * _normal(g, m, natoms, 3)).float()
    for f0 in range(0, n, step):
        m = min(step, n - f0)
        x = out[f0:f0 + m].double()
        if aligned:
            x = x + 0.2 * (_rand(g, m, 1, 3) - 0.5)
        else:
            x = torch.matmul(x, _rotations(m, g)) + 10 * (_rand(g, m, 1, 3) - 0.5)
        out[f0:f0 + m] = x.float()
    return out


def _masses(kind, natoms, seed):
    if kind == "backbone":
        return np.resize(np.array([14.0067, 12.011, 12.011], np.float32), natoms)
    if kind == "random":
        return np.random.default_rng(seed).uniform(1.0, 32.0, natoms).astype(np.float32)
    return np.ones(natoms, np.float32)


def _vectors(n, vdim, seed):
    """n FP64 vectors of sin/cos pairs of angles around 20 conformations."""
    g = _gen(seed, 2)
    half = (vdim + 1) // 2
    centres = 2 * math.pi * (_rand(g, 20, half) - 0.5)
    label = torch.randint(0, 20, (n,), generator=g, device=DEV)
    ang = centres[label] + 0.3 * _normal(g, n, half).double()
    return torch.stack([ang.sin(), ang.cos()], 2).reshape(n, 2 * half)[:, :vdim].contiguous()


def _requests(case):
    return [int(s) for s in case["requests"].split(",")]


def _n_fit(case):
    if case["kind"] == "serve":
        return sum(_requests(case))
    return case.get("n_fit", 0)


def _inputs(case, seed):
    """(resident set, query set or None, masses or None) on the device."""
    n, m = case["n_ref"], _n_fit(case)
    if case["kind"] == "data":
        x = _vectors(n + m, case["vdim"], seed)
        return x[:n], (x[n:] if m else None), None
    x = _frames(case["frames"], n + m, case["natoms"], seed, aligned=case.get("nofit", False))
    w = None if case["kind"] == "xtc" else _masses(case["mass"], case["natoms"], seed)
    return x[:n], (x[n:] if m else None), w


def _flags(case):
    return ((knn.KNN_NOFIT if case.get("nofit") else 0) |
            (knn.KNN_FULL_ROWS if case["kind"] == "rows" else 0))


def _write_xtc(path, x, quantum):
    L = knn.load()
    rc = L.mdsctk_xtc_write(path.encode(), x.ctypes.data, x.shape[0], x.shape[1],
                            ctypes.c_float(quantum), None, None, None)
    if rc < 0:
        raise RuntimeError("xtc_write: %d" % rc)


class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.case = case
    ref, fit, w = _inputs(case, seed)
    kind = case["kind"]
    if kind == "xtc":
        fd, s.path = tempfile.mkstemp(suffix=".xtc")
        os.close(fd)
        weakref.finalize(s, os.unlink, s.path)
        _write_xtc(s.path, ref.cpu().numpy(), case["quantum"])
        return s
    s.ctx = knn.KnnContext(0, case["precision"])
    if kind == "trajectory":
        s.x, s.w = ref.cpu().numpy(), w
        return s
    if kind == "data":
        s.ctx.set_data_reference(ref.cpu().numpy(), case["metric"])
        s.q = None if fit is None else fit.cpu().numpy()
        return s
    torch.cuda.synchronize()
    s.ctx.set_reference_device(ref.data_ptr(), case["n_ref"], case["natoms"], w)
    if kind == "serve":
        host = fit.cpu().numpy()
        ends = np.cumsum(_requests(case))
        s.q = [np.ascontiguousarray(a) for a in np.split(host, ends[:-1])]
        return s
    s.q = None if fit is None else fit.clone()
    s.n_fit = case["n_ref"] if fit is None else fit.shape[0]
    width = s.ctx.row_width(case.get("k", 0), _flags(case))
    s.dist = torch.zeros(s.n_fit, width, device=DEV, dtype=torch.float64)
    s.idx = torch.zeros(s.n_fit, width, device=DEV, dtype=torch.int32)
    return s


class _Borrowed:
    """A device buffer of the library, as torch.as_tensor takes one."""

    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = dict(shape=shape, typestr="<f4", data=(ptr, False),
                                             version=3, strides=None)


def run(s):
    c = s.case
    kind = c["kind"]
    if kind == "trajectory":
        s.ctx.set_reference(s.x, s.w)
        return s.ctx.query(None, c["k"])
    if kind in ("self", "cross", "rows"):
        s.ctx.query_device(0 if s.q is None else s.q.data_ptr(), s.n_fit, c.get("k", 0), _flags(c),
                           s.dist.data_ptr(), s.idx.data_ptr())
        return s.dist, s.idx
    if kind == "serve":
        reqs = [s.ctx.submit(q, c["k"]) for q in s.q]
        for r in reqs:
            s.ctx.wait(r)
        return [(r.dist, r.idx) for r in reqs]
    if kind == "data":
        return s.ctx.data_query(s.q, c["k"])
    L = knn.load()
    d, n = ctypes.c_void_p(), ctypes.c_int64()
    rc = L.mdsctk_xtc_read_device(s.path.encode(), c["natoms"], 0, ctypes.byref(d), ctypes.byref(n))
    if rc < 0:
        raise RuntimeError("xtc_read_device: %d" % rc)
    x = torch.as_tensor(_Borrowed(d.value, (n.value, c["natoms"], 3)), device=DEV).clone()
    torch.cuda.current_stream().synchronize()  # the copy is done: the buffer may go
    L.mdsctk_xtc_free_device(d)
    return x


def work(case):
    kind, n = case["kind"], case["n_ref"]
    if kind == "xtc":
        # about 5 bytes of packed block an atom (3 x 13 bits), 12 out
        return {"bytes": n * (92 + 17.0 * case["natoms"]), "flops": 0.0}
    m = _n_fit(case)
    if kind == "data":
        frame, per_pair = 8.0 * case["vdim"], 2.0 * case["vdim"]
    else:
        frame, per_pair = 12.0 * case["natoms"], (6.0 if case.get("nofit") else 18.0) * case["natoms"]
    width = n if kind == "rows" else min(case["k"], n - 1)
    pairs = m * n if m else n * (n - 1) / 2
    return {"bytes": (n + m) * frame + (m or n) * width * 12.0, "flops": pairs * per_pair}


# ---------------------------------------------------------------------------
# the same in 64 bits


def _centred(x, w):
    w = torch.as_tensor(w, device=DEV, dtype=torch.float64)
    x = x.double()
    x = x - (w[:, None] * x).sum(1, keepdim=True) / w.sum()
    x = x * w.sqrt()[:, None]
    return [x[:, :, c].contiguous() for c in range(3)], (x * x).sum((1, 2))


def _newton(S, g, steps):
    """Largest root of the quartic of the key matrix of S (nine tensors),
    from the upper bound g downwards."""
    xx, xy, xz, yx, yy, yz, zx, zy, zz = [t / g for t in S]
    fro = sum(t * t for t in (xx, xy, xz, yx, yy, yz, zx, zy, zz))
    det = xx * (yy * zz - yz * zy) - xy * (yx * zz - yz * zx) + xz * (yx * zy - yy * zx)
    c2, c1 = -2 * fro, -8 * det
    # c0 = det K = fro^2 - 4 |S^T S| second invariant (K's eigenvalues are
    # sums of the singular values of S with signs)
    a, b, d = xx * xx + yx * yx + zx * zx, xx * xy + yx * yy + zx * zy, xx * xz + yx * yz + zx * zz
    e, f = xy * xy + yy * yy + zy * zy, xy * xz + yy * yz + zy * zz
    h = xz * xz + yz * yz + zz * zz
    second = a * e - b * b + a * h - d * d + e * h - f * f
    c0 = fro * fro - 4 * second
    l = torch.ones_like(xx)
    for _ in range(steps):
        l2 = l * l
        p = (l2 + c2) * l2 + c1 * l + c0
        dp = (4 * l2 + 2 * c2) * l + c1
        l = l - torch.where(dp.abs() > 1e-280, p / dp, torch.zeros_like(p))
    return l * g


def _scores(a, b, nofit):
    """Squared deviations of all pairs of two centred sets."""
    (xa, ga), (xb, gb) = a, b
    if nofit:
        tr = sum(xa[c] @ xb[c].t() for c in range(3))
        return ga[:, None] + gb[None, :] - 2 * tr
    S = [xa[c] @ xb[d].t() for c in range(3) for d in range(3)]
    g = 0.5 * (ga[:, None] + gb[None, :])
    return 2 * (g - _newton(S, g, 12))


def _refine(a, b, idx, nofit):
    """The scores of the pairs (row, idx[row, j]) again, to convergence."""
    (xa, ga), (xb, gb) = a, b
    out = torch.empty(idx.shape, device=DEV, dtype=torch.float64)
    rows = max(1, int(1.5e8 // (idx.shape[1] * 3 * xa[0].shape[1])))
    for r in range(0, idx.shape[0], rows):
        j = idx[r:r + rows]
        p = [x[r:r + rows, None, :] for x in xa]
        q = [x[j] for x in xb]
        S = [(p[c] * q[d]).sum(-1) for c in range(3) for d in range(3)]
        g = 0.5 * (ga[r:r + rows, None] + gb[j])
        lam = (S[0] + S[4] + S[8]) if nofit else _newton(S, g, 60)
        out[r:r + rows] = 2 * (g - lam)
    return out


def _exact_frames(ref, fit, w, k, nofit, full):
    W = float(np.asarray(w, np.float64).sum())
    b = _centred(ref, w)
    a = b if fit is None else _centred(fit, w)
    n, m = b[1].shape[0], a[1].shape[0]
    rows = max(1, int(4e7 // n))
    got = []
    for r in range(0, m, rows):
        part = ([x[r:r + rows] for x in a[0]], a[1][r:r + rows])
        s = _scores(part, b, nofit)
        if not full:
            idx = s.topk(min(n, k + 9), dim=1, largest=False).indices
            s = _refine(part, b, idx, nofit).sort(dim=1).values[:, 1:k + 1]
        got.append(10 * (s.clamp(min=0) / W).sqrt())
    return torch.cat(got)


def _exact_data(ref, fit, k, metric):
    a = ref if fit is None else fit
    if metric == "correlation":
        unit = lambda x: torch.nn.functional.normalize(x - x.mean(1, keepdim=True), dim=1)  # noqa: E731
        ref, a = unit(ref), unit(a)
    n, v = ref.shape
    nb = (ref * ref).sum(1)
    got = []
    rows = max(1, int(1e8 // n))
    for r in range(0, a.shape[0], rows):
        p = a[r:r + rows]
        s = (p * p).sum(1)[:, None] + nb[None] - 2 * (p @ ref.t())
        idx = s.topk(min(n, k + 9), dim=1, largest=False).indices
        sub = max(1, int(1e8 // (idx.shape[1] * v)))
        d = torch.cat([((p[q:q + sub, None] - ref[idx[q:q + sub]]) ** 2).sum(-1)
                       for q in range(0, p.shape[0], sub)])
        got.append(d.sort(dim=1).values[:, 1:k + 1].sqrt() * (0.5 if metric == "correlation" else 1))
    return torch.cat(got)


def exact(case, seed):
    kind, n = case["kind"], case["n_ref"]
    m = _n_fit(case) or n
    if kind == "xtc":
        x, q = _inputs(case, seed)[0], case["quantum"]
        if case["natoms"] <= 9:
            return x.double()
        v = x.double() * q
        return torch.trunc(v + 0.5 * v.sign()) / q
    atoms = case["vdim"] / 3 if kind == "data" else case["natoms"]
    if n * m * (18 * atoms / 3e13 + 5e3 / 4e12) > 12:
        return None
    ref, fit, w = _inputs(case, seed)
    if kind == "data":
        return _exact_data(ref, fit, min(case["k"], n - 1), case["metric"]), None
    d = _exact_frames(ref, fit, w, min(case.get("k", 0), n - 1), case.get("nofit", False),
                      kind == "rows")
    if kind == "serve":
        return [(p, None) for p in d.split(_requests(case))]
    return d, None
