"""The work that users of this package have it do, as timed cases.

Every case goes through the Python binding of the C ABI (hpcscan_amd.capi), as a
user's program does: the Propa loop (free surface, then the fused Ac2 step), its
split variant (Laplacian, then the pressure update), the FD_D2 and FD_D1 axis
derivatives with their error sums, the grid operations, one shot's forward
modeling, its misfit gradient, and a batch of uneven shots.

listed() holds named cases, draw() one more of the same ranges: grids from the
61-point default side to 1000^3 inner points, ragged and odd sides, two and three
dimensions, FD orders 2-16, FP32, FP64 and FP32 storage with FP64 arithmetic.
"""
import math

import numpy as np
import torch

from hpcscan_amd import capi
from hpcscan_amd.layout import make_layout

DEV = "cuda"
PREC = {"fp32": (False, False), "fp64": (True, True), "fp32c64": (False, True)}   # storage, compute in 64 bits
CAP_BYTES = 4.1e9          # largest grid: 1000^3 in FP32


def listed():
    return [
        # the harness's default run: 61^3, order 8, 20 steps (launches and latency)
        {"name": "propa_default_61", "kind": "propa", "n1": 61, "n2": 61, "n3": 61, "order": 8, "prec": "fp32",
         "steps": 20},
        # the headline size: Propa Ac2Standard at 1000^3, order 8
        {"name": "propa_1000", "kind": "propa", "n1": 1000, "n2": 1000, "n3": 1000, "order": 8, "prec": "fp32",
         "steps": 2},
        # a model cut to its target area: three odd, unequal sides
        {"name": "propa_ragged", "kind": "propa", "n1": 403, "n2": 307, "n3": 255, "order": 4, "prec": "fp32",
         "steps": 4},
        # the double-precision matrix run, high order
        {"name": "propa_fp64_500", "kind": "propa", "n1": 500, "n2": 500, "n3": 500, "order": 12, "prec": "fp64",
         "steps": 2},
        # a 2D section (-dim 2)
        {"name": "propa_2d", "kind": "propa", "n1": 1501, "n2": 2001, "n3": 0, "order": 8, "prec": "fp32",
         "steps": 20},
        # Propa Ac2SplitComp of the matrix, highest order
        {"name": "split_500", "kind": "split", "n1": 500, "n2": 500, "n3": 500, "order": 16, "prec": "fp32",
         "steps": 2},
        # the FD_D2 test case: three axes, Laplacian, their L1 error sums
        {"name": "fd_d2_500", "kind": "fd_d2", "n1": 500, "n2": 500, "n3": 500, "order": 8, "prec": "fp32"},
        # the FD_D1 test case on a ragged grid, odd stencil half-width
        {"name": "fd_d1_ragged", "kind": "fd_d1", "n1": 251, "n2": 199, "n3": 333, "order": 6, "prec": "fp32"},
        # the Grid test case: fills, array operations and the error reductions
        {"name": "grid_ops_300", "kind": "grid", "n1": 300, "n2": 300, "n3": 300, "order": 8, "prec": "fp32"},
        # one shot of forward modeling, a receiver line (traces out)
        {"name": "shot_200", "kind": "shot", "n1": 200, "n2": 200, "n3": 200, "order": 8, "prec": "fp32", "nt": 100},
        # one shot's misfit gradient from a plan, 16-bit checkpoints every 20 steps
        {"name": "gradient_200", "kind": "grad", "n1": 200, "n2": 200, "n3": 200, "order": 8, "prec": "fp32",
         "nt": 100, "every": 20, "ckpt": "fp16"},
        # 32 uneven shots in one batch, the time loop in one graph
        {"name": "batch_32", "kind": "batch", "shots": 32, "lo": 192, "hi": 320, "order": 8, "prec": "fp32", "nt": 60},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _sides(rng, lo, hi, points):
    """three unequal sides, spread over their logarithm, at most `points` together"""
    while True:
        base = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        n = [min(hi, max(lo, int(round(base * rng.uniform(0.7, 1.4))))) for _ in range(3)]
        if rng.random() < 0.4:                       # sizes that people choose: whole tens
            n = [max(lo, v // 10 * 10) for v in n]
        if n[0] * n[1] * n[2] <= points:
            return n


def draw(rng):
    kind = rng.choice(["propa", "propa", "propa", "propa2d", "split", "fd_d2", "fd_d1", "grid", "shot", "grad",
                       "batch"])
    order = rng.choice([2, 4, 4, 6, 8, 8, 8, 10, 12, 12, 14, 16])
    prec = rng.choice(["fp32", "fp32", "fp32", "fp64", "fp32c64"])
    es = 8 if PREC[prec][0] else 4
    c = {"kind": kind, "order": order, "prec": prec}
    if kind == "propa2d":
        c.update(kind="propa", n1=_log(rng, 201, 6000), n2=_log(rng, 201, 6000), n3=0, steps=20)
    elif kind in ("propa", "split"):
        n = _sides(rng, 61, 1000, CAP_BYTES / es / (1 if kind == "propa" else 2))
        p = n[0] * n[1] * n[2]
        c.update(n1=n[0], n2=n[1], n3=n[2], steps=20 if p < 2e6 else 4 if p < 1e8 else 2)
    elif kind in ("fd_d2", "fd_d1", "grid"):
        n = _sides(rng, 61, 700, 3.5e8 if es == 4 else 1.5e8)
        c.update(n1=n[0], n2=n[1], n3=n[2])
    elif kind == "shot":
        n = _sides(rng, 61, 320, 2e7)
        c.update(n1=n[0], n2=n[1], n3=n[2], nt=rng.choice([60, 100, 150]))
    elif kind == "grad":
        n = _sides(rng, 61, 260, 1e7)
        every = rng.choice([0, 10, 20])
        c.update(n1=n[0], n2=n[1], n3=n[2], nt=rng.choice([45, 60, 100]), every=every,
                 ckpt=rng.choice(["fp16", "bf16"]) if every and prec == "fp32" else "full")
    else:
        # a batch takes one precision and rows that are whole 16-byte groups
        lo = _log(rng, 96, 220)
        c.update(prec="fp64" if es == 8 else "fp32", order=rng.choice([4, 8, 8, 12]), shots=rng.choice([4, 8, 16]),
                 lo=lo, hi=lo + rng.choice([32, 64, 100]), nt=60)
    return c


# ---- inputs -----------------------------------------------------------------------------
def _layout(c, n=None):
    n = n or ([c["n1"], c["n2"], c["n3"]] if c["n3"] else [c["n1"], c["n2"]])
    return make_layout(len(n), n, c["order"], fp64=PREC[c["prec"]][0])


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _dtype(c):
    return torch.float64 if PREC[c["prec"]][0] else torch.float32


def _weights(order):
    """centred second-derivative weights A0..AR"""
    R = order // 2
    f = math.factorial
    a = [2.0 * (-1) ** (j + 1) * f(R) ** 2 / (j * j * f(R - j) * f(R + j)) for j in range(1, R + 1)]
    return [-2.0 * sum(a)] + a


def _weights1(order):
    """staggered first-derivative weights A1..AR"""
    R = order // 2
    dd = 1
    for k in range(1, 2 * R, 2):
        dd *= k
    f = math.factorial
    return [(-1) ** (j + 1) * dd * dd / (2.0 ** (2 * R - 2) * f(R + j - 1) * f(R - j) * (2 * j - 1) ** 2)
            for j in range(1, R + 1)]


def _smooth(p, g, lo, hi, dt):
    """smooth random field in [lo, hi] over the whole grid (n3, n2, n1): noise on a coarse grid, interpolated"""
    shape = p.shape3()
    coarse = [max(2, s // 24 + 2) if s > 1 else 1 for s in shape]
    x = torch.rand([1, 1] + coarse, generator=g, device=DEV, dtype=torch.float32)
    x = torch.nn.functional.interpolate(x, size=shape, mode="trilinear", align_corners=True)
    return x[0, 0].to(dt).mul_(hi - lo).add_(lo)


def _modes(p, g, dt, amps):
    """sums of three sine modes over the whole grid (antisymmetric about the inner box's faces), one field per
    row of `amps` (3 amplitudes each)"""
    m = torch.randint(1, 5, (3, 3), generator=g, device=DEV).double()
    out = [torch.zeros(p.shape3(), dtype=dt, device=DEV) for _ in amps]
    for k in range(3):
        t = []
        for a in range(3):
            if a >= p.dim:
                t.append(torch.ones(1, dtype=torch.float64, device=DEV))
                continue
            x = p.axes[a]
            i = torch.arange(x.n, device=DEV, dtype=torch.float64) - x.inner_start
            t.append(torch.sin(math.pi * m[k, a] * i / (x.inner_end - x.inner_start)))
        plane = (t[1][:, None] * t[0][None, :]).to(dt)
        for f, am in zip(out, amps):
            f.addcmul_((float(am[k]) * t[2]).to(dt)[:, None, None].expand(p.shape3()), plane[None].expand(p.shape3()))
    return out


def _dt(c, p, vmax):
    A = _weights(c["order"])
    s = abs(A[0]) + 2 * sum(abs(a) for a in A[1:])
    return 0.8 * math.sqrt(4.0 / (p.dim * s)) * min(p.d[:p.dim]) / vmax


def _coef(p, v, dt):
    c = torch.zeros(p.shape3(), dtype=v.dtype, device=DEV)
    b = _box(p)
    c[b] = (v[b] * dt) ** 2
    return c


def _box(p):
    r = p.inner()
    return (slice(r[4], r[5] + 1), slice(r[2], r[3] + 1), slice(r[0], r[1] + 1))


def _ricker(nt, dt, f0):
    a = (math.pi * f0 * (np.arange(nt) * dt - 1.5 * math.sqrt(6.0) / (math.pi * f0))) ** 2
    return (1.0 - 2.0 * a) * np.exp(-a)


def _shot_inputs(c, p, g, nrec):
    """coef, wavelet, source and receiver indices of one shot: v 2000-4000 m/s, 10 m spacing, source one
    point below the top in the middle, a receiver line on the same depth"""
    p.d = [10.0] * 3
    v = _smooth(p, g, 2000.0, 4000.0, torch.float64)
    dt = _dt(c, p, 4000.0)
    nt = c["nt"]
    wav = torch.tensor(_ricker(nt, dt, 2.0 / (nt * dt)) * float(0.5 + torch.rand(1, generator=g, device=DEV)),
                       dtype=_dtype(c), device=DEV)
    r = p.inner()
    at = lambda i1, i2, i3: i1 + i2 * p.n1 + i3 * p.n1 * p.n2
    src = torch.tensor([at(r[0] + 1, (r[2] + r[3]) // 2, (r[4] + r[5]) // 2)], dtype=torch.int64, device=DEV)
    i2 = np.unique(np.round(np.linspace(r[2], r[3], min(nrec, r[3] - r[2] + 1))).astype(np.int64))
    rec = torch.tensor([at(r[0] + 1, int(j), (r[4] + r[5]) // 2) for j in i2], dtype=torch.int64, device=DEV)
    return {"v": v, "dt": dt, "coef": _coef(p, v, dt).to(_dtype(c)), "wav": wav.reshape(nt, 1).contiguous(),
            "src": src, "rec": rec}


def _cubes(c):
    """sides of a batch's cubes, uneven between lo and hi in no order, whole 16-byte rows"""
    n = np.random.RandomState(c["lo"]).randint(c["lo"] // 4, c["hi"] // 4 + 1, c["shots"]) * 4
    n[0], n[-1] = c["lo"] // 4 * 4, c["hi"] // 4 * 4
    return [int(m) for m in n]


def _inputs(case, seed):
    c, g = case, _gen(seed)
    k = c["kind"]
    if k == "batch":
        n = _cubes(c)
        ps = [_layout(c, [m] * 3) for m in n]
        return {"p": ps, "shots": [_shot_inputs(c, p, g, m) for p, m in zip(ps, n)]}
    p = _layout(c)
    t = _dtype(c)
    s = {"p": p}
    if k in ("propa", "split"):
        v = _smooth(p, g, 0.5, 1.0, t)
        s["coef"] = _coef(p, v, _dt(c, p, 1.0))
        am = torch.randn(3, generator=g, device=DEV).tolist()
        s["prc"], s["prn"] = _modes(p, g, t, [am, [0.999 * x for x in am]])
        if k == "split":
            s["lap"] = torch.zeros(p.shape3(), dtype=t, device=DEV)
    elif k in ("fd_d2", "fd_d1"):
        am = torch.randn(3, generator=g, device=DEV).tolist()
        s["u"], s["ref"] = _modes(p, g, t, [am, [30.0 * x for x in am]])
        s["w"] = [torch.zeros(p.shape3(), dtype=t, device=DEV) for _ in range(4 if k == "fd_d2" else 3)]
    elif k == "grid":
        x = [np.arange(a.halo2_end - a.halo1_start + 1) for a in p.axes]
        ph = torch.rand(7, generator=g, device=DEV).tolist()
        s["t"] = [np.sin(0.05 * (1 + ph[a]) * x[a] + ph[3 + a]) for a in range(3)]
        s["amp"], s["val"] = 1.0 + ph[6], 0.25 + ph[0]
        s["u"], s["v"], s["w"], s["z"] = (torch.zeros(p.shape3(), dtype=t, device=DEV) for _ in range(4))
    else:
        s.update(_shot_inputs(c, p, g, 200))
        if k == "shot":
            s["traces"] = torch.zeros((c["nt"], s["rec"].numel()), dtype=t, device=DEV)
        else:
            # observed data: the traces' order of magnitude, smooth in time
            s["obs"] = torch.cumsum(torch.randn((c["nt"], s["rec"].numel()), generator=g, device=DEV,
                                                dtype=torch.float64), 0).mul_(2e-3).to(t)
            s["grad"] = torch.zeros(p.npoint, dtype=torch.float64, device=DEV)
    return s


# ---- what a user's program has in hand, and one pass --------------------------------------
def _desc(c, s, p):
    return capi.make_shot(c["nt"], s["dt"], (s["src"], s["src"].numel()), s["wav"], (s["rec"], s["rec"].numel()))


def prepare(case, seed):
    c = case
    capi.init(0)
    s = _inputs(c, seed)
    s["case"] = c
    cf = PREC[c["prec"]][1]
    if c["kind"] == "batch":
        s["g"] = [capi.hsx_grid(p, cf) for p in s["p"]]
        for x in s["shots"]:
            del x["v"]
            x["traces"] = torch.zeros((c["nt"], x["rec"].numel()), dtype=_dtype(c), device=DEV)
        torch.cuda.synchronize()
        s["batch"] = capi.Batch(s["g"], [x["coef"] for x in s["shots"]],
                                [_desc(c, x, p) for x, p in zip(s["shots"], s["p"])],
                                [x["traces"] for x in s["shots"]])
        return s
    s["g"] = capi.hsx_grid(s["p"], cf)
    if c["kind"] in ("shot", "grad"):
        del s["v"]
        s["desc"] = _desc(c, s, s["p"])
    if c["kind"] == "grad":
        fmt = {"full": capi.HSX_CKPT_FP32, "fp16": capi.HSX_CKPT_FP16, "bf16": capi.HSX_CKPT_BF16}[c["ckpt"]]
        s["stream"] = torch.cuda.Stream()
        s["plan"] = capi.AdjointPlan(s["g"], c["nt"], s["rec"].numel(), c["every"], fmt)
    torch.cuda.synchronize()
    return s


def run(s):
    c, g = s["case"], s["g"]
    k = c["kind"]
    if k == "propa":
        prn, prc, coef = s["prn"], s["prc"], s["coef"]
        for _ in range(c["steps"]):
            capi.free_surface(g, prc)
            capi.ac2_step(g, prn, prc, coef)
            prn, prc = prc, prn
        return [prn, prc]
    if k == "split":
        prn, prc, coef, lap = s["prn"], s["prc"], s["coef"], s["lap"]
        for _ in range(c["steps"]):
            capi.free_surface(g, prc)
            capi.laplacian(g, prc, lap)
            capi.update_pressure(g, prn, prc, coef, lap)
            prn, prc = prc, prn
        return [prn, prc, lap]
    if k == "fd_d2":
        r = s["p"].inner()
        err = []
        for a in range(4):
            if a < 3:
                capi.fd_d2(g, a, s["u"], s["w"][a])
            else:
                capi.laplacian(g, s["u"], s["w"][a])
            err.append(list(capi.l1_sums(g, s["w"][a], s["ref"], r)))
        return [s["w"], err]
    if k == "fd_d1":
        for a in range(3):
            capi.fd_d1(g, a, s["u"], s["w"][a])
        return s["w"]
    if k == "grid":
        r, q = s["p"].all_points(), s["p"].inner()
        u, v, w, z = s["u"], s["v"], s["w"], s["z"]
        capi.fill_const(g, u, q, s["val"])
        capi.fill_separable(g, v, r, *s["t"], s["amp"])
        capi.array_op(g, capi.HSX_ARRAY_ADD, w, u, v)
        capi.array_op(g, capi.HSX_ARRAY_MULTIPLY, z, w, v)
        capi.free_surface(g, w)
        num = [capi.sum_abs(g, v, q), capi.sum_abs_diff(g, w, v, q), *capi.l1_sums(g, z, v, q),
               capi.max_err(g, w, u, q, 1e-5), *capi.min_max(g, z, q)]
        return [u, v, w, z, num]
    if k == "shot":
        capi.forward(g, s["coef"], s["desc"], s["traces"])
        return s["traces"]
    if k == "grad":
        with torch.cuda.stream(s["stream"]):
            s["grad"].zero_()
        m = s["plan"].gradient(g, s["coef"], s["desc"], s["obs"], s["grad"], stream=s["stream"].cuda_stream)
        return [s["grad"], m]
    s["batch"].run(use_graph=True)
    return [x["traces"] for x in s["shots"]]


def work(case):
    c = case
    es = 8 if PREC[c["prec"]][0] else 4
    R = c["order"] // 2
    k = c["kind"]
    if k == "batch":
        pts = float(sum(m ** 3 for m in _cubes(c)))
        return {"bytes": c["nt"] * pts * 4 * es, "flops": c["nt"] * pts * (9 * R + 9)}
    dim = 3 if c["n3"] else 2
    pts = float(c["n1"]) * c["n2"] * max(1, c["n3"])
    if k == "propa":       # prc, prn, coef in, prn out
        return {"bytes": c["steps"] * pts * 4 * es, "flops": c["steps"] * pts * (dim * (3 * R + 2) + 3)}
    if k == "split":       # u in, lap out; four in, one out
        return {"bytes": c["steps"] * pts * 7 * es, "flops": c["steps"] * pts * (dim * (3 * R + 2) + 3)}
    if k == "fd_d2":       # u in, w out four times; w and ref in for each error
        return {"bytes": pts * 16 * es, "flops": pts * (6 * (3 * R + 2) + 4 * 5)}
    if k == "fd_d1":
        return {"bytes": pts * 6 * es, "flops": pts * 9 * R}
    if k == "grid":        # two fills, two array operations, five reductions of 1 or 2 grids
        return {"bytes": pts * (2 + 6 + 8) * es, "flops": pts * 16}
    if k == "shot":
        return {"bytes": c["nt"] * pts * 4 * es, "flops": c["nt"] * pts * (9 * R + 9)}
    # gradient: forward and adjoint steps, the recomputation where there are checkpoints; per reverse step
    # three wavefields read, the gradient (64 bits) read and written
    steps = (3 if c["every"] else 2) * 4 * es + 3 * es + 16
    return {"bytes": c["nt"] * pts * steps, "flops": c["nt"] * pts * (3 if c["every"] else 2) * (9 * R + 9)}


# ---- the same in 64 bits, with plain tensor operations -------------------------------------
def _views(p, u, dim, off):
    """u shifted by `off` along tensor dim `dim`, on the inner box"""
    b = list(_box(p))
    b[dim] = slice(b[dim].start + off, b[dim].stop + off)
    return u[tuple(b)]


def _x_bc(p, u):
    for a in range(p.dim):
        dim, x = 2 - a, p.axes[a]
        v = u[tuple(slice(None) if d == dim else s for d, s in enumerate(_box(p)))]
        R = x.halo1_end - x.halo1_start + 1
        lo, hi = x.inner_start, x.inner_end
        v.select(dim, lo).zero_()
        v.narrow(dim, lo - R, R).copy_(-v.narrow(dim, lo + 1, R).flip(dim))
        v.select(dim, hi).zero_()
        v.narrow(dim, hi + 1, R).copy_(-v.narrow(dim, hi - R, R).flip(dim))


def _x_d2(p, u, a, A):
    acc = A[0] * _views(p, u, 2 - a, 0)
    for j in range(1, len(A)):
        acc.add_(_views(p, u, 2 - a, j) + _views(p, u, 2 - a, -j), alpha=A[j])
    return acc.mul_((1.0 / p.d[a]) ** 2)


def _x_lap(p, u, A):
    out = _x_d2(p, u, 0, A)
    for a in range(1, p.dim):
        out.add_(_x_d2(p, u, a, A))
    return out


def _x_step(p, prn, prc, coef, A):
    b = _box(p)
    lap = _x_lap(p, prc, A)
    prn[b] = 2.0 * prc[b] - prn[b] + coef[b] * lap
    return lap


def _x_forward(p, s, A, nt, keep=None):
    coef = s["coef"].double()
    prn, prc = (torch.zeros(p.shape3(), dtype=torch.float64, device=DEV) for _ in range(2))
    wav, tr = s["wav"].double(), []
    if keep is not None:
        keep.append(prc.clone())
    for n in range(nt):
        _x_bc(p, prc)
        _x_step(p, prn, prc, coef, A)
        prn.view(-1)[s["src"]] += wav[n]
        tr.append(prn.view(-1)[s["rec"]])
        if keep is not None:
            keep[-1] = prc.clone()
            keep.append(prn.clone())
        prn, prc = prc, prn
    return torch.stack(tr)


def exact(case, seed):
    c = case
    s = _inputs(c, seed)
    p, A, k = s["p"], _weights(c["order"]), c["kind"]
    if k == "batch":
        return [_x_forward(q, x, A, c["nt"]) for q, x in zip(p, s["shots"])]
    b = _box(p)
    if k in ("propa", "split"):
        prn, prc, coef = (s[n].double() for n in ("prn", "prc", "coef"))
        full = torch.zeros_like(prc) if k == "split" else None
        for _ in range(c["steps"]):
            _x_bc(p, prc)
            lap = _x_step(p, prn, prc, coef, A)
            if full is not None:
                full[b] = lap
            prn, prc = prc, prn
        return [prn, prc] if full is None else [prn, prc, full]
    if k == "fd_d2":
        u, w = s["u"].double(), []
        for a in range(4):
            w.append(torch.zeros_like(u))
            w[-1][b] = _x_d2(p, u, a, A) if a < 3 else _x_lap(p, u, A)
        ref = float(s["ref"][b].double().abs().sum())
        # the difference's sum is in 32 bits mostly the rounding of the derivatives
        return [w, [[None, ref]] * 4]
    if k == "fd_d1":
        u, w, A1 = s["u"].double(), [], _weights1(c["order"])
        for a in range(3):
            acc = torch.zeros_like(u)
            acc[b] = sum(x * (_views(p, u, 2 - a, j) - _views(p, u, 2 - a, -j - 1)) for j, x in enumerate(A1)) / p.d[a]
            w.append(acc)
        return w
    if k == "grid":
        t = _dtype(c)
        r = p.all_points()
        u, v = (torch.zeros(p.shape3(), dtype=torch.float64, device=DEV) for _ in range(2))
        u[b] = torch.tensor(s["val"], dtype=t).double().item()
        t1, t2, t3 = (torch.tensor(x, device=DEV) for x in s["t"])
        v[r[4]:r[5] + 1, r[2]:r[3] + 1, r[0]:r[1] + 1] = s["amp"] * t1[None, None, :] * t2[None, :, None] * t3[:, None, None]
        w = u + v
        z = w * v
        _x_bc(p, w)
        num = [v[b].abs().sum(), (w[b] - v[b]).abs().sum(), (z[b] - v[b]).abs().sum(), v[b].abs().sum(),
               ((w[b] - u[b]).abs() / u[b].abs()).max(), z[b].min(), z[b].max()]
        return [u, v, w, z, [float(x) for x in num]]
    if k == "shot":
        return _x_forward(p, s, A, c["nt"])
    # the adjoint recursion mu^k = 2 mu^{k+1} - (mu^{k+2} - c e^k) + c Lap mu^{k+1} and its imaging sum
    nt, q = c["nt"], []
    e = _x_forward(p, s, A, nt, keep=q) - s["obs"].double()
    coef, wav = s["coef"].double(), s["wav"].double()
    q = [torch.zeros_like(q[0])] + q                     # q[k + 1] = q^k, k = -1 .. nt
    box = tuple(slice(x.start + 1, x.stop - 1) for x in b)
    mu1, mu2, g = (torch.zeros(p.shape3(), dtype=torch.float64, device=DEV) for _ in range(3))
    scale = -1.0 / s["dt"] ** 2
    r = p.inner()
    j = int(s["src"][0])
    i3, i2, i1 = j // (p.n1 * p.n2), j // p.n1 % p.n2, j % p.n1
    inside = r[0] < i1 < r[1] and r[2] < i2 < r[3] and r[4] < i3 < r[5]
    for n in range(nt, 0, -1):
        mu2.view(-1)[s["rec"]] -= coef.view(-1)[s["rec"]] * e[n - 1]
        _x_bc(p, mu1)
        _x_step(p, mu2, mu1, coef, A)
        g[box] += scale * mu2[box] * (q[n + 1][box] - 2.0 * q[n][box] + q[n - 1][box])
        if inside:
            g.view(-1)[j] -= scale * mu2.view(-1)[j] * wav[n - 1, 0]
        mu1, mu2 = mu2, mu1
    return [g.reshape(-1), 0.5 * float((e * e).sum())]
