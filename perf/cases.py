"""Performance cases of the framework: the calls that stencil programs make, through the public
Python binding of the C ABI, over the sizes, element types and forms they use.

A case names one application loop ("op"), its grid, its number of sweeps and its form.  The state
is what such a program keeps between calls: the fields on the device (allocated by the library's
own allocator), the double buffer's current side, and the one context of the process, whose
tuning decisions and workspaces later calls reuse.  Each pass advances the fields further, as a
program's time loop does.
"""
import math

import numpy as np
import torch

from appfis_amd import hip

_TORCH = {hip.U8: torch.uint8, hip.F32: torch.float32, hip.F64: torch.float64, hip.F16: torch.float16,
          hip.BF16: torch.bfloat16}
_CODE = {"u8": hip.U8, "f32": hip.F32, "f64": hip.F64, "f16": hip.F16, "bf16": hip.BF16}
_SIZE = {"u8": 1, "f16": 2, "bf16": 2, "f32": 4, "f64": 8}
_FORM = {"plain": hip.PLAIN, "chosen": hip.CHOSEN}

HEAT_C = 0.1
# c0 = 0.5, c_r = 0.125 / r on three axes, divided by their growth of 2.0625 per step so that a
# long run stays in the range of every storage type
FDTD_C = [c / 2.0625 for c in (0.5, 0.125, 0.125 / 2, 0.125 / 3, 0.125 / 4)]
OMEGA = 0.8
DX, CFL, HEXTRA, RAIN, MANNING2, WALL = 10.0, 0.5, 1e-3, 50e-3 / 3600.0, 0.035 ** 2, 1e6

_ctx = None


def context():
    """The process's context: one device, one stream, one host thread."""
    global _ctx
    if _ctx is None:
        torch.cuda.init()
        _ctx = hip.Context(0)
    return _ctx


# ---- the cases -----------------------------------------------------------------------------------


def listed():
    return [
        # a small plate, the kind a unit test or a parameter study runs in its thousands: 50
        # sweeps and the field's checksum, all launch latency
        {"name": "heat_small", "op": "heat", "nx": 96, "ny": 80, "dtype": "f64", "form": "chosen", "iters": 50},
        # the ordinary heat run: 1024 x 1024 in FP64, 500 explicit sweeps
        {"name": "heat_1024", "op": "heat", "nx": 1024, "ny": 1024, "dtype": "f64", "form": "chosen", "iters": 500},
        # many independent plates of uneven sizes advanced together
        {"name": "heat_ensemble", "op": "heat_ens", "grids": 64, "lo": 128, "hi": 1024, "pick": 1006,
         "dtype": "f64", "iters": 200},
        # a Life board whose width is no multiple of anything, and its live-cell count
        {"name": "gol_ragged", "op": "gol", "nx": 1000, "ny": 777, "form": "chosen", "iters": 100},
        # the large board: 1000 generations of 8192 x 8192
        {"name": "gol_8192", "op": "gol", "nx": 8192, "ny": 8192, "form": "chosen", "iters": 1000},
        # wave propagation in FP64 on a middling box with odd sides, called with the default form
        {"name": "fdtd_f64_odd", "op": "fdtd", "nx": 255, "ny": 201, "nz": 179, "dtype": "f64", "form": "plain",
         "iters": 10},
        # the large box in FP32
        {"name": "fdtd_f32_512", "op": "fdtd", "nx": 512, "ny": 512, "nz": 512, "dtype": "f32", "form": "chosen",
         "iters": 20},
        # fields stored in 16 bits to halve the traffic
        {"name": "fdtd_bf16_256", "op": "fdtd", "nx": 256, "ny": 256, "nz": 256, "dtype": "bf16", "form": "chosen",
         "iters": 20},
        # the Poisson solve: FP32 sweeps with the residual of each, the default form
        {"name": "himeno_f32", "op": "himeno", "nx": 257, "ny": 257, "nz": 513, "dtype": "f32", "form": "plain",
         "iters": 50},
        # an FP64 Poisson solve by defect correction on a middling grid
        {"name": "himeno_dc", "op": "himeno", "nx": 129, "ny": 129, "nz": 257, "dtype": "f64", "form": "chosen",
         "iters": 48},
        # one catchment in FP64, the default form
        {"name": "flood_f64", "op": "flood", "sides": "785", "dtype": "f64", "form": "plain", "iters": 40},
        # a flood ensemble of uneven catchments in FP32
        {"name": "flood_ens_f32", "op": "flood_ens",
         "sides": "3851,1405,2125,870,1740,2278,1101,2204,985,1182,2958,785", "dtype": "f32", "iters": 20},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["heat", "heat_ens", "gol", "gol", "fdtd", "fdtd", "himeno", "flood", "flood_ens"])
    form = rng.choice(["plain", "chosen"])
    if op == "heat":
        return {"op": op, "nx": _log(rng, 48, 2048), "ny": _log(rng, 48, 2048), "dtype": rng.choice(["f64", "f32"]),
                "form": form, "iters": _log(rng, 20, 500)}
    if op == "heat_ens":
        return {"op": op, "grids": rng.randint(4, 64), "lo": 64, "hi": rng.choice([256, 512, 1024]),
                "pick": rng.randrange(1 << 20), "dtype": rng.choice(["f64", "f32"]), "iters": _log(rng, 20, 200)}
    if op == "gol":
        nx = _log(rng, 64, 8192)
        align = rng.choice([1, 1, 32, 2048])  # boards are as often round in binary as not
        nx = max(align, nx // align * align)
        return {"op": op, "nx": nx, "ny": _log(rng, 64, 8192), "form": form if rng.random() < 0.5 else "chosen",
                "iters": _log(rng, 10, 300)}
    if op == "fdtd":
        return {"op": op, "nx": _log(rng, 32, 512), "ny": _log(rng, 32, 512), "nz": _log(rng, 32, 512),
                "dtype": rng.choice(["f32", "f64", "f16", "bf16"]), "form": form, "iters": rng.randint(2, 20)}
    if op == "himeno":
        return {"op": op, "nx": _log(rng, 33, 257), "ny": _log(rng, 33, 257), "nz": _log(rng, 33, 513),
                "dtype": "f64" if form == "chosen" else rng.choice(["f32", "f64"]), "form": form,
                "iters": rng.randint(4, 48)}
    if op == "flood":
        return {"op": op, "sides": str(_log(rng, 64, 2048)), "dtype": rng.choice(["f64", "f32"]), "form": form,
                "iters": _log(rng, 10, 80)}
    return {"op": op, "sides": ",".join(str(_log(rng, 128, 2048)) for _ in range(rng.randint(3, 12))),
            "dtype": rng.choice(["f64", "f32"]), "iters": rng.randint(10, 40)}


# ---- inputs --------------------------------------------------------------------------------------


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _rand(shape, seed):
    return torch.rand(shape, generator=_gen(seed), dtype=torch.float64, device="cuda")


def _sizes(case):
    """(nx, ny) of every grid of a heat ensemble."""
    r = np.random.RandomState(case["pick"])
    n = r.randint(case["lo"], case["hi"] + 1, size=(case["grids"], 2))
    return [(int(a), int(b)) for a, b in n]


def _plate(nx, ny, dtype, seed):
    """Uniform [0, 1) interior, Dirichlet 0 in the ghost ring."""
    u = torch.zeros((ny + 2, nx + 2), dtype=_TORCH[_CODE[dtype]], device="cuda")
    u[1:-1, 1:-1] = _rand((ny, nx), seed).to(u.dtype)
    return u


def _box(case, seed):
    """Uniform [0, 1) interior in the storage type, 4 ghost cells of 0."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    u = torch.zeros((nz + 8, ny + 8, nx + 8), dtype=_TORCH[_CODE[case["dtype"]]], device="cuda")
    u[4:-4, 4:-4, 4:-4] = _rand((nz, ny, nx), seed).to(u.dtype)
    return u


def _board(case, seed):
    """Cells alive with probability 1/4."""
    b = torch.zeros((case["ny"] + 2, case["nx"] + 2), dtype=torch.uint8, device="cuda")
    b[1:-1, 1:-1] = (torch.rand((case["ny"], case["nx"]), generator=_gen(seed), device="cuda") < 0.25).to(torch.uint8)
    return b


def _poisson(case, seed):
    """The 14 arrays p0, p1, a0..a3, b0..b2, c0..c2, bnd, wrk1: p = (k/(nz-1))^2, a0..a2 uniform
    in [0.9, 1.1], a3 = 1/6, b = 0, c = bnd = 1, wrk1 = 0."""
    shape, dt = (case["nz"], case["ny"], case["nx"]), _TORCH[_CODE[case["dtype"]]]
    k = torch.arange(shape[0], dtype=torch.float64, device="cuda") / (shape[0] - 1)
    p = (k * k).view(-1, 1, 1).expand(shape).to(dt)

    def full(v):
        return torch.full(shape, v, dtype=dt, device="cuda")

    a = [(0.9 + 0.2 * _rand(shape, 3 * seed + i)).to(dt) for i in range(3)]
    return [p, p, *a, full(1 / 6), full(0), full(0), full(0), full(1), full(1), full(1), full(1), full(0)]


def _catchment(n, dtype, seed):
    """h, qx, qy, z, n2 of an n x n catchment of 10 m cells: 20 Gaussian hills (5-50 m high, 200-2000 m
    wide) on a slope of 0.001 behind a wall, water at rest in the lowest tenth, and patches of
    sheet water centimetres deep with dry ground between them."""
    r = np.random.RandomState(seed % (1 << 31))
    x = (torch.arange(n, dtype=torch.float64, device="cuda") + 0.5) * DX
    z = (0.001 * x).view(1, -1).repeat(n, 1)
    for _ in range(20):
        amp, sigma, cx, cy = 5 + 45 * r.rand(), 200 + 1800 * r.rand(), r.rand() * n * DX, r.rand() * n * DX
        gx, gy = torch.exp(-(x - cx) ** 2 / (2 * sigma ** 2)), torch.exp(-(x - cy) ** 2 / (2 * sigma ** 2))
        z += amp * gy.view(-1, 1) * gx.view(1, -1)
    wave = [2 * math.pi * x / (DX * (40 + 40 * r.rand())) + 6 * r.rand() for _ in range(2)]
    sheet = 0.1 * torch.clamp(torch.sin(wave[1]).view(-1, 1) * torch.sin(wave[0]).view(1, -1) + 0.3, min=0)
    low, high = z.min(), z.max()
    lake = torch.clamp(low + 0.1 * (high - low) - z, min=0)
    dt = _TORCH[_CODE[dtype]]

    def padded(inner, edge):
        f = torch.full((n + 2, n + 2), edge, dtype=dt, device="cuda")
        f[1:-1, 1:-1] = inner.to(dt) if isinstance(inner, torch.Tensor) else inner
        return f

    return [padded(torch.maximum(lake, sheet), 0.0), padded(0.0, 0.0), padded(0.0, 0.0), padded(z, WALL),
            padded(MANNING2, MANNING2)]


def _catchments(case, seed):
    return [_catchment(int(n), case["dtype"], 1000 * seed + i) for i, n in enumerate(case["sides"].split(","))]


# ---- device fields -------------------------------------------------------------------------------


class _Memory:
    """A library allocation as torch sees it (no copy)."""

    def __init__(self, arr):
        kind = {hip.U8: "|u1", hip.F32: "<f4", hip.F64: "<f8", hip.F16: "<f2", hip.BF16: "<i2"}[arr.dtype]
        self.__cuda_array_interface__ = {"shape": arr.shape, "typestr": kind, "data": (arr.ptr, False), "version": 2}


class Field:
    """A field in the library's memory and the same memory as a tensor.  The tensor keeps the
    allocation, so that a result outlives the state that it was computed in."""

    def __init__(self, values, dtype):
        self.arr = context().array(tuple(values.shape), _CODE[dtype])
        t = torch.as_tensor(_Memory(self.arr), device="cuda")
        self.tensor = t.view(torch.bfloat16) if dtype == "bf16" else t
        self.tensor.allocation = self.arr
        self.tensor.copy_(values)


def prepare(case, seed):
    op, s = case["op"], {"case": case, "ctx": context()}
    if op == "heat":
        u = _plate(case["nx"], case["ny"], case["dtype"], seed)
        s["buf"] = [Field(u, case["dtype"]), Field(torch.zeros_like(u), case["dtype"])]
    elif op == "heat_ens":
        s["grids"] = []
        for i, (nx, ny) in enumerate(_sizes(case)):
            u = _plate(nx, ny, case["dtype"], 1000 * seed + i)
            s["grids"].append([Field(u, case["dtype"]), Field(torch.zeros_like(u), case["dtype"]), nx, ny])
    elif op == "gol":
        b = _board(case, seed)
        s["buf"] = [Field(b, "u8"), Field(torch.zeros_like(b), "u8")]
    elif op == "fdtd":
        u = _box(case, seed)
        s["buf"] = [Field(u, case["dtype"]), Field(torch.zeros_like(u), case["dtype"])]
    elif op == "himeno":
        s["arrays"] = [Field(a, case["dtype"]) for a in _poisson(case, seed)]
    else:
        s["scen"] = [[Field(f, case["dtype"]) for f in c] for c in _catchments(case, seed)]
        s["params"] = hip.FloodParams(DX, CFL, HEXTRA, 1.0, 0.0, RAIN, 0.0)
    torch.cuda.synchronize()
    return s


# ---- one pass ------------------------------------------------------------------------------------


def run(state):
    case, ctx = state["case"], state["ctx"]
    op, n = case["op"], case["iters"]
    if op in ("heat", "gol", "fdtd"):
        a, b = state["buf"]
        if op == "heat":
            ctx.heat2d(a.arr, b.arr, case["nx"], case["ny"], HEAT_C, n, _FORM[case["form"]])
        elif op == "gol":
            ctx.gol(a.arr, b.arr, case["nx"], case["ny"], n, _FORM[case["form"]])
        else:
            ctx.fdtd3d(a.arr, b.arr, case["nx"], case["ny"], case["nz"], FDTD_C, n, _FORM[case["form"]])
        if n % 2:  # the field is in the second buffer: it is the current one from here on
            state["buf"] = [b, a]
        now, other = state["buf"]
        if op == "fdtd":
            return now.tensor
        total = ctx.reduce_sum_wide(now.arr, [1, case["nx"] + 1, 1, case["ny"] + 1, 0, 1])
        # a Life call leaves the last two generations, a heat call the field; both programs
        # report a sum over the interior
        return [now.tensor, other.tensor, total] if op == "gol" else [now.tensor, total]
    if op == "heat_ens":
        ctx.heat2d_ensemble([(g[0].arr, g[1].arr, g[2], g[3]) for g in state["grids"]], HEAT_C, n)
        if n % 2:
            for g in state["grids"]:
                g[0], g[1] = g[1], g[0]
        return [g[0].tensor for g in state["grids"]]
    if op == "himeno":
        f = state["arrays"]
        gosa = ctx.himeno([x.arr for x in f], case["nx"], case["ny"], case["nz"], OMEGA, n, _FORM[case["form"]])
        if n % 2:
            f[0], f[1] = f[1], f[0]
        return [f[0].tensor, gosa]
    scen, prm = state["scen"], state["params"]
    if op == "flood":
        f = scen[0]
        side = int(case["sides"])
        t, v = ctx.flood_run(*[x.arr for x in f], side, side, prm, n, _FORM[case["form"]])
    else:
        keys = ("h", "qx", "qy", "z", "n2")
        sides = [int(x) for x in case["sides"].split(",")]
        t, v = ctx.flood_ensemble_run([{"nx": m, "ny": m, **{k: x.arr for k, x in zip(keys, f)}}
                                       for m, f in zip(sides, scen)], prm, n, _CODE[case["dtype"]])
    return [[x.tensor for x in f[:3]] for f in scen] + [t, v]


def work(case):
    """Bytes that go in and come out once, and the arithmetic of the update formulas (integer
    operations for Life; about 360 for a flood cell: two edge solves and the friction update)."""
    op, n = case["op"], case["iters"]
    if op == "heat":
        cells = case["nx"] * case["ny"]
        return {"bytes": 2 * cells * _SIZE[case["dtype"]], "flops": 7 * cells * n}
    if op == "heat_ens":
        cells = sum(nx * ny for nx, ny in _sizes(case))
        return {"bytes": 2 * cells * _SIZE[case["dtype"]], "flops": 7 * cells * n}
    if op == "gol":
        cells = case["nx"] * case["ny"]
        return {"bytes": 3 * cells, "flops": 10 * cells * n}
    if op == "fdtd":
        cells = case["nx"] * case["ny"] * case["nz"]
        return {"bytes": 2 * cells * _SIZE[case["dtype"]], "flops": 29 * cells * n}
    if op == "himeno":
        cells = case["nx"] * case["ny"] * case["nz"]
        return {"bytes": 14 * cells * _SIZE[case["dtype"]], "flops": 34 * cells * n}
    cells = sum(int(m) ** 2 for m in case["sides"].split(","))
    return {"bytes": 8 * cells * _SIZE[case["dtype"]], "flops": 360 * cells * n}


# ---- the same results in 64 bits -----------------------------------------------------------------


def _heat64(u, n):
    u = u.double()
    for _ in range(n):
        c = u[1:-1, 1:-1]
        v = u.clone()
        v[1:-1, 1:-1] = c + HEAT_C * (u[:-2, 1:-1] + u[2:, 1:-1] + u[1:-1, 2:] + u[1:-1, :-2] - 4 * c)
        u = v
    return u


def _fdtd64(u, n):
    u = u.double()
    inner = slice(4, -4)
    for _ in range(n):
        v = torch.zeros_like(u)
        acc = FDTD_C[0] * u[inner, inner, inner]
        for r in range(1, 5):
            lo, hi = slice(4 - r, -4 - r), slice(4 + r, -4 + r or None)
            acc = acc + FDTD_C[r] * (u[inner, inner, lo] + u[inner, inner, hi] + u[inner, lo, inner] +
                                     u[inner, hi, inner] + u[lo, inner, inner] + u[hi, inner, inner])
        v[inner, inner, inner] = acc
        u = v
    return u


def _himeno64(arrays, n):
    p, _, a0, a1, a2, a3, b0, b1, b2, c0, c1, c2, bnd, wrk1 = [x.double() for x in arrays]
    m, gosa = slice(1, -1), []

    def at(f, k, j, i):
        return f[1 + k:f.shape[0] - 1 + k, 1 + j:f.shape[1] - 1 + j, 1 + i:f.shape[2] - 1 + i]

    for _ in range(n):
        s0 = (at(a0, 0, 0, 0) * at(p, 0, 0, 1) + at(a1, 0, 0, 0) * at(p, 0, 1, 0) + at(a2, 0, 0, 0) * at(p, 1, 0, 0)
              + at(b0, 0, 0, 0) * (at(p, 0, 1, 1) - at(p, 0, -1, 1) - at(p, 0, 1, -1) + at(p, 0, -1, -1))
              + at(b1, 0, 0, 0) * (at(p, 1, 1, 0) - at(p, 1, -1, 0) - at(p, -1, 1, 0) + at(p, -1, -1, 0))
              + at(b2, 0, 0, 0) * (at(p, 1, 0, 1) - at(p, 1, 0, -1) - at(p, -1, 0, 1) + at(p, -1, 0, -1))
              + at(c0, 0, 0, 0) * at(p, 0, 0, -1) + at(c1, 0, 0, 0) * at(p, 0, -1, 0)
              + at(c2, 0, 0, 0) * at(p, -1, 0, 0) + at(wrk1, 0, 0, 0))
        ss = (s0 * at(a3, 0, 0, 0) - at(p, 0, 0, 0)) * at(bnd, 0, 0, 0)
        p = p.clone()
        p[m, m, m] += OMEGA * ss
        gosa.append(ss.square().sum())
    return [p, torch.stack(gosa)]


def _edge64(h1, h2, q1, q2, s1, s2, z1, z2, hn1, hn2, dt):
    """Roe flux across an edge with entropy fix, bed slope and wet/dry treatment.  q: momentum along
    the edge's normal, s: across it.  Returns what the two cells lose, as (h, normal, across)."""
    g, tiny = 9.81, 1e-12
    sq1, sq2 = torch.sqrt(torch.clamp(h1, min=0)), torch.sqrt(torch.clamp(h2, min=0))
    zero = torch.zeros_like(h1)
    (u1, v1), (u2, v2) = [(torch.where(w, a / h, zero), torch.where(w, b / h, zero))
                          for a, b, h, w in ((q1, s1, h1, hn1), (q2, s2, h2, hn2))]
    dh, c = h2 - h1, torch.sqrt(g * 0.5 * (h1 + h2))
    u, v = (u1 * sq1 + u2 * sq2) / (sq1 + sq2), (v1 * sq1 + v2 * sq2) / (sq1 + sq2)
    lam, fix = [u - c, u, u + c], [zero, zero, zero]
    rg = 3.132091953
    for i, sign in ((0, -1.0), (2, 1.0)):
        e1, e2 = u1 + sign * rg * sq1, u2 + sign * rg * sq2
        fan = (e1 < 0) & (e2 > 0)
        new = e1 * (e2 - lam[0]) / (e2 - e1) if i == 0 else e2 * (lam[2] - e1) / (e2 - e1)
        fix[i] = torch.where(fan, lam[i] - new, zero)
        lam[i] = torch.where(fan, new, lam[i])
    jump = ((q2 - q1) - u * dh) / c
    alpha = [0.5 * (dh - jump), ((s2 - s1) - v * dh) / c, 0.5 * (dh + jump)]
    vec = [(1.0, u - c, v), (0.0, 0.0, c), (1.0, u + c, v)]
    dz = z2 - z1
    up = dz >= 0
    dzp = torch.where(up & (z1 + h1 < z2), h1, torch.where(~up & (z2 + h2 < z1), -h2, dz))
    beta = 0.5 * g * (torch.where(up, h1, h2) - 0.5 * dzp.abs()) * dzp / c
    hs = h1 + alpha[0]
    sub = (lam[0] * lam[2] < 0) & (hs > 0) & (h1 > 0) & (h2 > 0)
    capped = torch.minimum(torch.maximum(beta, alpha[0] * lam[0] - h1 * DX * 0.5 / dt),
                           -alpha[2] * lam[2] + h2 * DX * 0.5 / dt)
    beta = torch.where(sub, capped, beta)
    betas = [beta, zero, -beta]
    l1, l2 = hs - beta / lam[0], hs - beta / lam[2]
    only1 = (l2 < -tiny) & (h2 < tiny)
    only2 = ~only1 & (l1 < -tiny) & (h1 < tiny)
    mass = (lam[0] * alpha[0] - betas[0]) + (lam[2] * alpha[2] - betas[2])
    out = []
    wet = (h1 > 0) | (h2 > 0)
    for first in (True, False):
        d = []
        for k in range(3):
            t = zero
            for i in range(3):
                side = (lam[i] <= 0) if first else (lam[i] > 0)
                t = t + torch.where(side, (lam[i] * alpha[i] - betas[i]) * vec[i][k], zero)
            t = torch.where(only1 | only2, zero, t)
            if k == 0:
                t = torch.where(only1 if first else only2, mass, t)
            for i in (0, 2):
                side = (fix[i] <= 0) if first else (fix[i] > 0)
                t = t + torch.where(side, fix[i] * alpha[i] * vec[i][k], zero)
            d.append(torch.where(wet & (t.abs() >= tiny), t, zero))
        out.append(d)
    return out


def _flood64(fields, n):
    # the fields are compared with the threshold as their type holds it
    hx = float(torch.tensor(HEXTRA, dtype=fields[0].dtype))
    h, qx, qy, z, n2 = [f.double() for f in fields]
    g, tiny, m, time, times, volumes = 9.81, 1e-12, slice(1, -1), 0.0, [], []
    for _ in range(n):
        hi, xi, yi = h[m, m], qx[m, m], qy[m, m]
        deep, root = hi > hx, torch.sqrt(g * hi)
        step = CFL * torch.minimum(DX / ((xi / hi).abs() + root), DX / ((yi / hi).abs() + root))
        step = torch.where(deep, step, torch.full_like(step, math.inf)).min()
        dt = torch.where(torch.isinf(step), torch.ones_like(step), step)
        wet = h >= hx
        a, b = (m, slice(None, -1)), (m, slice(1, None))
        d1, d2 = _edge64(h[a], h[b], qx[a], qx[b], qy[a], qy[b], z[a], z[b], wet[a], wet[b], dt)
        loss = [d2[k][:, :-1] + d1[k][:, 1:] for k in range(3)]
        a, b = (slice(1, None), m), (slice(None, -1), m)  # the normal points from row j to row j - 1's side
        d1, d2 = _edge64(h[a], h[b], qy[a], qy[b], qx[a], qx[b], z[a], z[b], wet[a], wet[b], dt)
        # the second eigenvector and its strength both change sign between the directions: the same product
        loss = [loss[0] + d1[0][:-1] + d2[0][1:], loss[1] + d1[2][:-1] + d2[2][1:], loss[2] + d1[1][:-1] + d2[1][1:]]
        f = dt / DX
        hn = torch.clamp(hi - f * loss[0], min=0)
        mx, my = xi - f * loss[1], yi - f * loss[2]
        mod = torch.sqrt(mx * mx + my * my)
        rub = (n2[m, m] > tiny) & (hi >= hx) & (mod > tiny)
        tt = dt * g * n2[m, m] * mod / hi ** (7.0 / 3.0)
        slow = torch.sqrt(1.0 + 4.0 * tt)
        mx = torch.where(rub, 2.0 * mx / (1.0 + slow), mx)
        my = torch.where(rub, 2.0 * my / (1.0 + slow), my)
        still = hn < hx
        zero = torch.zeros_like(mx)
        h, qx, qy = h.clone(), qx.clone(), qy.clone()
        h[m, m], qx[m, m], qy[m, m] = hn + RAIN * dt, torch.where(still, zero, mx), torch.where(still, zero, my)
        hi, top = h[m, m], h[m, m] + z[m, m]

        def bank(dj, di):
            at = (slice(1 + dj, h.shape[0] - 1 + dj), slice(1 + di, h.shape[1] - 1 + di))
            return (hi > hx) & (top < z[at]) & (h[at] < tiny)

        qx[m, m] = torch.where(bank(0, 1) | bank(0, -1), zero, qx[m, m])
        qy[m, m] = torch.where(bank(-1, 0) | bank(1, 0), zero, qy[m, m])
        time += float(dt)
        times.append(time)
        volumes.append(float(h[m, m].sum()) * DX * DX)
    return [h, qx, qy], times, volumes


def exact(case, seed):
    op, n = case["op"], case["iters"]
    if op == "heat":
        u = _heat64(_plate(case["nx"], case["ny"], case["dtype"], seed), n)
        return [u, np.float64(float(u[1:-1, 1:-1].sum()))]
    if op == "heat_ens":
        return [_heat64(_plate(nx, ny, case["dtype"], 1000 * seed + i), n) for i, (nx, ny) in enumerate(_sizes(case))]
    if op == "fdtd":
        return _fdtd64(_box(case, seed), n)
    if op == "himeno":
        return _himeno64(_poisson(case, seed), n)
    if op == "gol":
        return None  # whole numbers
    done = [_flood64(f, n) for f in _catchments(case, seed)]
    times, volumes = np.array([d[1] for d in done]), np.array([d[2] for d in done])
    if op == "flood":
        times, volumes = times[0], volumes[0]
    return [d[0] for d in done] + [times, volumes]
