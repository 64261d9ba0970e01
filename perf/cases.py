"""The work a program has this library do, as timed cases.

A simulation step of a resident colony (tree, neighbour lists, sums), eager
and as a captured graph; the same step from a host program's arrays; the
transfers between cells and the field grid in both directions; and the
environment solve.  Sizes follow this repository's generators, benchmark and
tests: colonies from a few thousand to some millions of cells, one or many,
of one or two cell types, in two and three dimensions, and grids from the
reference's own 17^3 (a 2048^3 box at resolution 128) to 384^3.

A case is a dict of plain values; `prepare` gives what a program holds before
the call, `run` makes one pass and returns its whole outputs, `exact` gives
the same outputs in 64 bits from plain torch operations.
"""
import ctypes
import math

import numpy as np
import torch

import timothy_amd as tm

# cell types of the generators: radius 1 with h = 2, radius 1.5 with h = 3
SIZES = (1.0, 1.5)
REACH = (2.0, 3.0)
YOUNG = 2100.0
DT = 16000.0
FIELD_MEAN = 0.1575


def _types(k):
    return [dict(size=SIZES[i], h=REACH[i], h2=REACH[i] ** 2, h3=REACH[i] ** 3, h4=REACH[i] ** 4) for i in range(k)]


def _step(name, cells, shape, precision, colonies=1, large=0.0, captured=False):
    return dict(name=name, kind="step", cells=cells, shape=shape, precision=precision, colonies=colonies, large=large,
                captured=captured)


def listed():
    return [
        # the environment solve at the reference's own grid and parameters
        # (D 1.82e-5, resolution 128, dt 16000, a point source): one call per
        # simulation step, latency alone
        dict(name="env_17", kind="solve", nx=17, ny=17, nz=17, z=1.8e-5, substeps=1, source="point"),
        # a growing culture on a plate: a two-dimensional colony, bit-exact form
        _step("sheet_30k_fp64", 30011, "sheet", "fp64"),
        # a program that keeps its cells on the host (as the reference does)
        # and has each step's results copied back
        dict(name="host_20k_fp64", kind="host", cells=20000, shape="ball", precision="fp64"),
        # an ordinary spheroid, bit-exact form
        _step("step_300k_fp64", 300007, "ball", "fp64"),
        # the benchmark's colony, mixed form
        _step("step_2m_mixed", 2000000, "gaussian", "mixed"),
        # many small independent colonies in one set of launches, captured
        _step("batch_128_mixed", 4000000, "gaussian", "mixed", colonies=128, captured=True),
        # a large colony with 5% larger cells
        _step("step_6m_two_types", 6000001, "gaussian", "mixed", large=0.05),
        # cells to the field grid: the deposit by phase, and by volume
        dict(name="deposit_2m_256", kind="deposit", cells=2000000, shape="gaussian", nodes=256, weight="phase"),
        # the field grid to cells: gradient and interpolation, FP64 and FP32
        dict(name="sample_2m_256_f64", kind="sample", cells=2000000, shape="gaussian", nodes=256, field="f64"),
        dict(name="sample_5m_384_f32", kind="sample", cells=5000000, shape="gaussian", nodes=384, field="f32"),
        # the environment solve with a strong coupling and every node a source
        dict(name="env_96x80x112", kind="solve", nx=96, ny=80, nz=112, z=0.5, substeps=2, source="cells"),
        dict(name="env_256", kind="solve", nx=256, ny=256, nz=256, z=2.0, substeps=1, source="cells"),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "batch", "sheet", "host", "deposit", "sample", "solve", "solve"])
    shape = rng.choice(["ball", "gaussian"])
    precision = rng.choice(["mixed", "fp64"])
    if kind == "step":
        large = rng.choice([0.0, 0.0, 0.05])
        return dict(kind="step", cells=int(_log(rng, 2e3, 4e6)), shape=shape, precision=precision, colonies=1,
                    large=large, captured=rng.random() < 0.3)
    if kind == "batch":
        colonies = int(_log(rng, 4, 256))
        return dict(kind="step", cells=int(colonies * _log(rng, 2e3, 3e6 / colonies)), shape=shape,
                    precision=precision, colonies=colonies, large=0.0, captured=rng.random() < 0.5)
    if kind == "sheet":
        return dict(kind="step", cells=int(_log(rng, 2e3, 3e5)), shape="sheet", precision=precision, colonies=1,
                    large=0.0, captured=False)
    if kind == "host":
        return dict(kind="host", cells=int(_log(rng, 2e3, 2e5)), shape=shape, precision=precision)
    if kind == "deposit":
        return dict(kind="deposit", cells=int(_log(rng, 1e4, 4e6)), shape=shape, nodes=int(_log(rng, 24, 320)),
                    weight=rng.choice(["phase", "volume"]))
    if kind == "sample":
        return dict(kind="sample", cells=int(_log(rng, 1e4, 4e6)), shape=shape, nodes=int(_log(rng, 24, 320)),
                    field=rng.choice(["f64", "f32"]))
    side = _log(rng, 16, 200)
    n = [max(8, int(side * rng.uniform(0.7, 1.3))) for _ in range(3)]
    return dict(kind="solve", nx=n[0], ny=n[1], nz=n[2], z=_log(rng, 1e-5, 3.0), substeps=rng.choice([1, 1, 2]),
                source=rng.choice(["point", "cells", "none"]))


# ---- inputs, from the seed alone


def _gen(seed, sub):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + 7919 * sub) % (1 << 62))
    return g


def _uniform(g, *shape):
    return torch.rand(*shape, generator=g, dtype=torch.float64, device="cuda")


def _points(shape, n, g):
    """n positions of one colony: a ball at volume fraction 0.6, a Gaussian
    spheroid (sigma 0.35 of the half width, 0.7 of that in z, cut off at the
    half width) at the benchmark's density, or a disk at area fraction 0.6"""
    got, have = [], 0
    while have < n:
        m = 2 * (n - have) + 64
        if shape == "gaussian":
            w = 146.6 * (n / 2e6) ** (1.0 / 3.0)
            p = torch.randn(m, 3, generator=g, dtype=torch.float64, device="cuda")
            p = p * torch.tensor([0.35 * w, 0.35 * w, 0.245 * w], dtype=torch.float64, device="cuda")
            p = p[(p.abs() <= w).all(1)]
        elif shape == "ball":
            r = (n / 0.6) ** (1.0 / 3.0)
            p = (2 * _uniform(g, m, 3) - 1) * r
            p = p[(p * p).sum(1) <= r * r]
        else:
            r = math.sqrt(n / 0.6)
            p = (2 * _uniform(g, m, 3) - 1) * r
            p[:, 2] = 0.0
            p = p[(p * p).sum(1) <= r * r]
        got.append(p)
        have += len(p)
    return torch.cat(got)[:n]


def _offsets(case, seed):
    """cells per colony, log-uniform over a factor of 50, as offsets"""
    k, n = case.get("colonies", 1), case["cells"]
    if k == 1:
        return [0, n]
    r = np.random.default_rng(int(seed) + 17)
    w = np.exp(r.uniform(0.0, math.log(50.0), k))
    sizes = np.maximum(64, np.floor(n * w / w.sum()).astype(np.int64))
    sizes[np.argmax(sizes)] += n - sizes.sum()
    return [0] + [int(v) for v in np.cumsum(sizes)]


def _colony(case, seed):
    off = _offsets(case, seed)
    n = off[-1]
    p = torch.cat([_points(case["shape"], off[i + 1] - off[i], _gen(seed, 10 + i)) for i in range(len(off) - 1)])
    g = _gen(seed, 1)
    ctype = (_uniform(g, n) < case.get("large", 0.0)).to(torch.int32)
    size = torch.tensor(SIZES, dtype=torch.float64, device="cuda")[ctype.long()]
    young = (YOUNG + 100.0 * (2.0 * _uniform(g, n) - 1.0)).float()
    # phases of a growing culture: a tenth resting (0), a twentieth dead (5)
    u = _uniform(g, n)
    phase = torch.ones(n, dtype=torch.int32, device="cuda")
    phase[u < 0.1] = 0
    phase[u > 0.95] = 5
    return dict(off=off, n=n, x=p[:, 0].contiguous(), y=p[:, 1].contiguous(), z=p[:, 2].contiguous(), size=size,
                young=young, ctype=ctype, phase=phase, dim=2 if case["shape"] == "sheet" else 3)


class _Buffer:
    """a torch tensor in the place of a tm.DeviceArray"""

    def __init__(self, t):
        self.t = t
        self.ptr = t.data_ptr()
        self.dtype = np.dtype(str(t.dtype).replace("torch.", ""))


class _View:
    """device memory of a context, for torch.as_tensor (keeps the context)"""

    def __init__(self, ctx, ptr, n, typestr):
        self.ctx = ctx
        self.__cuda_array_interface__ = dict(shape=(n,), typestr=typestr, data=(ptr, False), strides=None, version=2)


def _bound(case, seed):
    col = _colony(case, seed)
    ctx = tm.Context(0)
    ctx.set_celltypes(_types(2), col["dim"])
    torch.cuda.synchronize()
    ctx.bind_device(col["n"], *[col[k].data_ptr() for k in ("x", "y", "z", "size", "young", "ctype", "phase")],
                    colony_offsets=col["off"] if len(col["off"]) > 2 else None)
    return ctx, col


def _box_grid(col, nodes):
    """a cubic grid spanning the cells, every corner of every cell inside"""
    p = torch.stack([col["x"], col["y"], col["z"]], 1)
    lower = p.min(0).values.cpu().numpy()
    ext = float((p.max(0).values.cpu().numpy() - lower).max())
    res = np.float32(ext / (nodes - 2))
    if float(res) * (nodes - 2) < ext:
        res = np.nextafter(res, np.float32(np.inf))
    return _grid([nodes] * 3, lower, res)


def _grid(ls, lower, res):
    return dict(lower=lower, resolution=np.float32(res), loweridx=[0, 0, 0], upperidx=[v - 1 for v in ls], localsize=ls)


def _field(grid, seed, dtype):
    """a smooth concentration: eight Gaussians on the grid's nodes"""
    ls = grid["localsize"]
    g = _gen(seed, 3)
    r = _uniform(g, 8, 5).cpu().numpy()
    out = torch.zeros(ls, dtype=torch.float64, device="cuda")
    ax = [(torch.arange(v, device="cuda", dtype=torch.float64) + 0.5) / v for v in ls]
    for k in range(8):
        s = 0.05 + 0.15 * r[k, 4]
        e = [torch.exp(-((ax[a] - r[k, a]) ** 2) / (2 * s * s)) for a in range(3)]
        out += (0.5 + r[k, 3]) * e[0][:, None, None] * e[1][None, :, None] * e[2][None, None, :]
    return out.reshape(-1).to(dtype)


def _solve_inputs(case, seed):
    ls = [case["nx"], case["ny"], case["nz"]]
    n = ls[0] * ls[1] * ls[2]
    res = np.float32(128.0)
    diffusion = case["z"] * float(res * res) / DT
    g = _gen(seed, 4)
    u0 = FIELD_MEAN + 0.01 * _uniform(g, n)
    src = None
    if case["source"] == "point":
        src = torch.zeros(n, dtype=torch.float64, device="cuda")
        src[(5 * ls[1] + 5) * ls[2] + 5] = 100.0
    elif case["source"] == "cells":
        src = 1e-2 * _uniform(g, n) * (_uniform(g, n) < 0.2)
    par = tm.Diffusion.make(diffusion, DT, FIELD_MEAN, 0.0, 1e-12, 400, case["substeps"])
    return _grid(ls, [-1024.0] * 3, res), u0, src, par


def prepare(case, seed):
    kind = case["kind"]
    s = dict(kind=kind, precision=tm.MIXED if case.get("precision") == "mixed" else tm.FP64)
    if kind == "solve":
        grid, u0, src, par = _solve_inputs(case, seed)
        s.update(ctx=tm.Context(0), grid=grid, u0=u0, u=_Buffer(torch.empty_like(u0)), par=par,
                 src=None if src is None else _Buffer(src))
        s["stream"] = torch.cuda.ExternalStream(tm.lib().tm_stream(s["ctx"].h))
    elif kind == "host":
        col = _colony(case, seed)
        s["cells"] = {k: col[k].cpu().numpy() for k in ("x", "y", "z", "size", "young", "ctype", "phase")}
        s["ctx"] = tm.Context(0)
        s["ctx"].set_celltypes(_types(2), col["dim"])
    else:
        s["ctx"], s["col"] = _bound(case, seed)
        ctx, n = s["ctx"], s["col"]["n"]
        if kind == "step" and case["captured"]:
            ctx.graph_capture(s["precision"])
        s["captured"] = case.get("captured", False)
        if kind in ("deposit", "sample"):
            ctx.build()
            s["grid"] = _box_grid(s["col"], case["nodes"])
            total = case["nodes"] ** 3
            if kind == "deposit":
                s["weight"] = 1 if case["weight"] == "volume" else 0
                s["production"] = _Buffer(torch.empty(total, dtype=torch.float64, device="cuda"))
            else:
                dt = torch.float32 if case["field"] == "f32" else torch.float64
                s["field"] = _Buffer(_field(s["grid"], seed, dt))
                s["gradient"] = _Buffer(torch.empty(3 * total, dtype=dt, device="cuda"))
                s["values"] = _Buffer(torch.empty(4 * n, dtype=torch.float64, device="cuda"))
    torch.cuda.synchronize()
    return s


def _device_results(ctx, n):
    p = [ctypes.c_void_p() for _ in range(7)]
    ctx._check(tm.lib().tm_device_results(ctx.h, *[ctypes.byref(v) for v in p]))
    names = ("density", "v", "mindist", "fx", "fy", "fz", "order")
    return {k: torch.as_tensor(_View(ctx, v.value, n, "<i4" if k == "order" else "<f8"), device="cuda")
            for k, v in zip(names, p)}


def run(s):
    ctx = s["ctx"]
    if s["kind"] == "solve":
        # the stepped field is the program's next state; the old one is kept
        with torch.cuda.stream(s["stream"]):
            s["u"].t.copy_(s["u0"])
        ctx.diffusion_step(s["grid"], s["par"], s["u"], s["src"])
        return {"field": s["u"].t}
    if s["kind"] == "host":
        c = s["cells"]
        ctx.upload(c["x"], c["y"], c["z"], c["size"], c["young"], c["ctype"], c["phase"])
        ctx.step(s["precision"])
        return ctx.results()
    if s["kind"] == "step":
        if s["captured"]:
            ctx.graph_launch()
        else:
            ctx.step(s["precision"])
        return _device_results(ctx, s["col"]["n"])
    if s["kind"] == "deposit":
        ctx.cic_deposit(s["grid"], s["production"], s["weight"])
        return {"production": s["production"].t}
    ctx.field_gradient(s["grid"], s["field"], s["gradient"])
    ctx.cic_interp(s["grid"], s["field"], s["gradient"], s["values"])
    return {"gradient": s["gradient"].t, "values": s["values"].t}


def work(case):
    """what a pass cannot do without: every input read once, every output
    written once, and the arithmetic of about 16 neighbours per cell, of the
    eight corners of a cell, or of the solver's iterations"""
    kind = case["kind"]
    if kind == "solve":
        n = case["nx"] * case["ny"] * case["nz"]
        kappa = 1.0 + 12.0 * case["z"]
        its = max(1.0, 0.5 * math.sqrt(kappa) * math.log(2e12)) if case["z"] > 1e-3 else 2.0
        return {"bytes": case["substeps"] * n * (16.0 + (8.0 if case["source"] != "none" else 0.0)),
                "flops": case["substeps"] * its * n * 20.0}
    n = case["cells"]
    if kind in ("step", "host"):
        return {"bytes": n * (48.0 + 52.0), "flops": n * 16.0 * 40.0}
    g = case["nodes"] ** 3
    if kind == "deposit":
        return {"bytes": 36.0 * n + 8.0 * g, "flops": n * 40.0}
    size = 4.0 if case["field"] == "f32" else 8.0
    return {"bytes": n * (24.0 + 32.0) + 4.0 * size * g, "flops": n * 100.0 + 6.0 * g}


# ---- the same outputs in 64 bits, from plain torch operations


def _spread(v):
    """21 bits of v to every third bit"""
    out = torch.zeros_like(v)
    for b in range(21):
        out |= ((v >> b) & 1) << (3 * b)
    return out


def _order(col):
    """the cells in Morton order of their 29-bit codes, colony by colony"""
    n, off = col["n"], col["off"]
    cid = torch.repeat_interleave(torch.arange(len(off) - 1, device="cuda"),
                                  torch.tensor(np.diff(off), device="cuda"))
    ext = torch.tensor(REACH, dtype=torch.float64, device="cuda")[col["ctype"].long()] + 0.01
    pos = [col[k] for k in "xyz"]
    shift, span = [], []
    for p in pos:
        lo = torch.full((len(off) - 1,), math.inf, dtype=torch.float64, device="cuda")
        lo.scatter_reduce_(0, cid, p - ext, "amin")
        hi = torch.full_like(lo, -math.inf)
        hi.scatter_reduce_(0, cid, p + ext, "amax")
        shift.append(lo)
        span.append(hi - lo)
    scale = torch.maximum(torch.maximum(span[0], span[1]), span[2])
    code = [((p - s[cid]) / scale[cid] * 536870912.0).to(torch.int64) for p, s in zip(pos, shift)]
    high = sum(_spread(c >> 8) << a for a, c in enumerate(code))
    low = sum(_spread(c & 255) << a for a, c in enumerate(code))
    o = torch.argsort(low, stable=True)
    o = o[torch.argsort(high[o], stable=True)]
    return o[torch.argsort(cid[o], stable=True)], cid


def _sums(col, cid, at):
    """density and force of the cells `at`, from all cells, by binning"""
    h = torch.tensor(REACH, dtype=torch.float64, device="cuda")[col["ctype"].long()]
    hm = float(h.max())
    pos = torch.stack([col["x"], col["y"], col["z"]], 1)
    b = torch.floor((pos - pos.min(0).values) / (hm * (1 + 1e-9))).to(torch.int64) + 1
    m = (b.max(0).values + 2).tolist()
    key = ((cid * m[0] + b[:, 0]) * m[1] + b[:, 1]) * m[2] + b[:, 2]
    skey, o = torch.sort(key)
    P, S = pos[o], col["size"][o]
    dim3 = col["dim"] == 3
    ty = _types(2)
    col_of = lambda f: torch.tensor([f(t) for t in ty], dtype=torch.float64, device="cuda")  # noqa: E731
    kd = col_of(lambda t: (t["h3"] if dim3 else t["h2"]) / t["size"] * (8 / (math.pi * t["h3"]) if dim3 else 40 / (7 * math.pi * t["h2"])))
    kf = col_of(lambda t: 48 / (math.pi * t["h4"]) if dim3 else 320 / (7 * math.pi * t["h3"]))
    out = torch.zeros(4, len(at), dtype=torch.float64, device="cuda")
    for c0 in range(0, len(at), 1 << 21):
        cells = at[c0:c0 + (1 << 21)]
        for dx in (-1, 0, 1):
            for dy in (-1, 0, 1):
                k = key[cells] + (dx * m[1] + dy) * m[2]
                lo = torch.searchsorted(skey, k - 1)
                hi = torch.searchsorted(skey, k + 1, right=True)
                me = torch.arange(len(cells), device="cuda")
                while True:
                    keep = lo < hi
                    lo, hi, me = lo[keep], hi[keep], me[keep]
                    if not len(me):
                        break
                    c = cells[me]
                    d = P[lo] - pos[c]
                    dist = torch.sqrt((d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1]) + d[:, 2] * d[:, 2])
                    near = (dist <= h[c]) & (o[lo] != c)
                    i, ci, q, r = me[near], c[near], lo[near], dist[near]
                    u = r / h[ci]
                    w = torch.where(u <= 0.5, 1 - 6 * u * u + 6 * u ** 3, 2 * (1 - u) ** 3)
                    g = torch.where(u <= 0.5, -2 * u + 3 * u * u, -(1 - u) ** 2) / r
                    t = col["ctype"][ci].long()
                    out[0, c0 + i] += kd[t] * S[q] * w
                    for a in range(3 if dim3 else 2):
                        out[1 + a, c0 + i] += kf[t] * g * d[near, a]
                    lo = lo + 1
    return out


def _axis(p, lower, res):
    """corner index and the weights of it and the next node (the reference
    forms the corner's offset in 32 bits)"""
    i = ((p - lower) / res).to(torch.int64)
    d = (p - (lower + (i.float() * res).double())) / res
    return i, (1.0 - d, d)


def _corners(col, grid):
    res = float(grid["resolution"])
    ax = [_axis(col[k], float(grid["lower"][a]), res) for a, k in enumerate("xyz")]
    ls = grid["localsize"]
    for a in (0, 1):
        for b in (0, 1):
            for c in (0, 1):
                yield (((ax[0][0] + a) * ls[1] + ax[1][0] + b) * ls[2] + ax[2][0] + c,
                       ax[0][1][a] * ax[1][1][b] * ax[2][1][c])


def _modes(n):
    k = torch.arange(1, n + 1, dtype=torch.float64, device="cuda")
    return torch.sin(math.pi * k[:, None] * k[None, :] / (n + 1)) * math.sqrt(2.0 / (n + 1)), \
        2.0 - 2.0 * torch.cos(math.pi * k / (n + 1))


def _transform(u, V):
    u = torch.matmul(V[0], u.reshape(len(V[0]), -1)).reshape(u.shape)
    u = torch.matmul(u, V[2])
    return torch.matmul(u.transpose(1, 2).contiguous(), V[1]).transpose(1, 2).contiguous()


def exact(case, seed):
    kind = case["kind"]
    if kind == "solve":
        grid, u, src, par = _solve_inputs(case, seed)
        ls = grid["localsize"]
        z = par.diffusion * par.dt / float(grid["resolution"] * grid["resolution"])
        VM = [_modes(v) for v in ls]
        V, lam = [m[0] for m in VM], [m[1] for m in VM]
        den = 1.0 + z * (lam[0][:, None, None] + lam[1][None, :, None] + lam[2][None, None, :])
        u = u.reshape(ls)
        for _ in range(case["substeps"]):
            b = u.clone()
            for a in range(3):
                for e in (0, ls[a] - 1):
                    b.select(a, e).add_(z * par.boundary)
            if src is not None:
                b += src.reshape(ls)
            u = _transform(_transform(b, V) / den, V)
        return {"field": u.reshape(-1)}
    col = _colony(case, seed)
    if kind in ("step", "host"):
        order, cid = _order(col)
        if kind == "host":
            order = torch.arange(col["n"], device="cuda")
        r = _sums(col, cid, order)
        if kind == "host":
            return {"density": r[0], "v": None, "mindist": None, "force": r[1:].T.contiguous()}
        return {"density": r[0], "v": None, "mindist": None, "fx": r[1], "fy": r[2], "fz": r[3], "order": None}
    grid = _box_grid(col, case["nodes"])
    total = case["nodes"] ** 3
    if kind == "deposit":
        if case["weight"] == "volume":
            w = 4.0 / 3.0 * math.pi * col["size"] ** 3
        else:
            w = torch.ones(col["n"], dtype=torch.float64, device="cuda")
            w[col["phase"] == 0] = 0.75
        w = torch.where(col["phase"] == 5, torch.zeros_like(w), w) if case["weight"] == "phase" else w
        out = torch.zeros(total, dtype=torch.float64, device="cuda")
        for node, c in _corners(col, grid):
            out.index_add_(0, node, w * c)
        return {"production": out}
    f = _field(grid, seed, torch.float32 if case["field"] == "f32" else torch.float64).double()
    u = f.reshape(grid["localsize"])
    grad = torch.empty(*grid["localsize"], 3, dtype=torch.float64, device="cuda")
    for a in range(3):
        n = u.shape[a]
        i = torch.arange(n, device="cuda")
        d = u.index_select(a, (i + 1).clamp(max=n - 1)) - u.index_select(a, (i - 1).clamp(min=0))
        grad[..., a] = d / float(grid["resolution"])
    four = torch.cat([f[:, None], grad.reshape(-1, 3)], 1)
    out = torch.zeros(col["n"], 4, dtype=torch.float64, device="cuda")
    for node, c in _corners(col, grid):
        out += four[node] * c[:, None]
    return {"gradient": grad.reshape(-1), "values": out.reshape(-1)}
