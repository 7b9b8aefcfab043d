"""GPU parity of the Triton flood step chain (fused flux/update/rain + fix/CFL/volume).

FP64 without friction touches only + - * / sqrt, all correctly rounded on both sides,
so h, qx, qy, the dt sequence and the simulated time are bit-exact against the oracle.
With Manning friction the GPU's cbrt may differ from glibc's by an ulp, so FP64 is held
to FLOOD_F64_RTOL.  The FP32 bulk form is checked against the FP64 oracle with the
stated FLOOD_F32_H_RTOL (relative L2 of h) and its FP64 Kahan volume against the
mass balance.  The batched ensemble (tile work-list, graph-captured step chunks) must
reproduce single-scenario runs bit for bit.
"""
import numpy as np
import pytest

import oracle
from appfis_amd import hip

pytestmark = pytest.mark.gpu

FLOOD_F64_RTOL = 1e-9
FLOOD_F32_H_RTOL = 1e-3
# Stated accuracy of the FP32 bulk form on the config workload (2000 steps from a dry
# start under rain) against the FP64 oracle: relative L2 of h and of the Kahan volume.
# The FP32 error depends on the scenario: 9e-6 on scenario 23, 1.7e-3 on scenario 4, where
# water collects in a fast jet along the west wall and the jet's cells differ by up to
# 3.5 cm.  That is the cost of FP32 storage, not of the kernel's arithmetic: the oracle's
# own FP32 restatement (libm-accurate operations) is off by 1.6e-3, and FP64 arithmetic
# with h, qx, qy rounded to FP32 after every step by 5.3e-4 (both measured with the oracle
# on the CPU; too slow to repeat in this test).
FLOOD_F32_CONFIG_H_RTOL = 5e-3
FLOOD_F32_CONFIG_VOL_RTOL = 1e-4
DX, CN, HEXTRA, DT_FALLBACK, RAIN = 10.0, 0.5, 1e-3, 1.0, 50e-3 / 3600.0


def scenario(n, seed, dtype=np.float64, wet=0.0):
    z = oracle.flood_dem(n, n, DX, seed)
    h = np.zeros_like(z)
    if wet:
        h[1:-1, 1:-1] = np.maximum(np.percentile(z[1:-1, 1:-1], 40) - z[1:-1, 1:-1], 0.0) + wet
    n2 = np.full_like(z, 0.035 ** 2)
    return [a.astype(dtype) for a in (h, np.zeros_like(z), np.zeros_like(z), z, n2)]


def params(print_interval=0.0):
    return hip.FloodParams(DX, CN, HEXTRA, DT_FALLBACK, print_interval, RAIN, 0.0)


def gpu_run(ctx, arrs, steps, variant=hip.PLAIN, print_interval=0.0):
    dt = hip.F64 if arrs[0].dtype == np.float64 else hip.F32
    d = [ctx.from_numpy(a, dt) for a in arrs]
    n = arrs[0].shape[0] - 2
    t, v = ctx.flood_run(d[0], d[1], d[2], d[3], d[4], n, n, params(print_interval), steps, variant)
    return [x.download() for x in d[:3]], t, v


def cpu_run(arrs, steps, print_interval=0.0):
    a = [x.copy() for x in arrs]
    n = a[0].shape[0] - 2
    t, v, dt = oracle.flood_run(a[0], a[1], a[2], a[3], a[4], n, n, DX, CN, HEXTRA, DT_FALLBACK, print_interval,
                                RAIN, 0.0, steps)
    return a[:3], t, v


@pytest.mark.parametrize("n,wet,steps", [(48, 0.0, 60), (100, 0.2, 40), (67, 0.5, 25)])
def test_flood_f64_frictionless_bit_exact(ctx, n, wet, steps):
    arrs = scenario(n, 3000 + n, wet=wet)
    arrs[4][:] = 0.0
    g, tg, vg = gpu_run(ctx, arrs, steps)
    c, tc, vc = cpu_run(arrs, steps)
    for a, b in zip(g, c):
        assert np.array_equal(a, b)
    assert np.array_equal(tg, tc)
    assert np.allclose(vg, vc, rtol=1e-13, atol=0)


@pytest.mark.parametrize("n", [1, 2, 61, 62, 63, 125, 311, 500])
def test_flood_strip_heights_bit_exact(ctx, n):
    # the strips' height follows the grid (1 row up to 5 at these sizes): one cell, strips one
    # column short of, equal to and one past their width, and last strips with fewer rows
    arrs = scenario(n, 3200 + n, wet=0.1)
    arrs[4][:] = 0.0
    g, tg, vg = gpu_run(ctx, arrs, 7)
    c, tc, vc = cpu_run(arrs, 7)
    for a, b in zip(g, c):
        assert np.array_equal(a, b)
    assert np.array_equal(tg, tc)
    assert np.allclose(vg, vc, rtol=1e-13, atol=0)


# A call's strips have one height, which follows the sum of its grids: beside a dry grid of these
# sides (0: alone) a small grid is marched in strips of 1, 2, 3, 5, 14 and 32 rows (on 256 CUs).
FLOOD_BESIDE = {hip.F64: [0, 465, 713, 1240, 1581, 2387], hip.F32: [0, 775, 1426, 1674, 1581, 2387]}
FLOOD_HEIGHTS = [1, 2, 3, 5, 14, 32]


def _strip_rows(dt, sides):
    """The height by the rule of csrc/flood_impl.hpp on 256 CUs, for grids of (nx, ny)."""
    few, more = (2.1, 0.4) if dt == hip.F64 else (2.2, 0.2)

    def cost(rows):
        strips = sum(-(-nx // 62) * -(-ny // rows) for nx, ny in sides)
        return max(-(-(-(-strips // 4)) // 256), few) * (rows + more)

    return min([32, 28, 24, 20, 16, 14, 12, 10, 8, 7, 6, 5, 4, 3, 2, 1], key=cost)


@pytest.mark.parametrize("dt", [hip.F64, hip.F32])
def test_flood_strips_of_every_height(ctx, dt):
    # 70 x 67 cells: two strips wide, and the last strip of each height but 1 has fewer rows.  FP64
    # without friction equals the oracle bit for bit at every height; FP32 gives the bits of the
    # strips of one row
    nx, ny, steps = 70, 67, 9
    npdt = np.float64 if dt == hip.F64 else np.float32
    z = oracle.flood_dem(nx, ny, DX, 3300)
    h = np.zeros_like(z)
    h[1:-1, 1:-1] = np.maximum(np.percentile(z[1:-1, 1:-1], 40) - z[1:-1, 1:-1], 0.0) + 0.1
    h[20:30, 10:40] = 0.0
    arrs = [x.astype(npdt) for x in (h, np.zeros_like(z), np.zeros_like(z), z, np.zeros_like(z))]
    c = [x.astype(np.float64) for x in arrs]
    tc, vc, _ = oracle.flood_run(*c, nx, ny, DX, CN, HEXTRA, DT_FALLBACK, 0.0, RAIN, 0.0, steps)
    keys = ("h", "qx", "qy", "z", "n2")
    first = None
    for side, height in zip(FLOOD_BESIDE[dt], FLOOD_HEIGHTS):
        sides = [(nx, ny)] + ([(side, side)] if side else [])
        assert _strip_rows(dt, sides) == height
        scen = [{"nx": nx, "ny": ny, **{k: ctx.from_numpy(x, dt) for k, x in zip(keys, arrs)}}]
        if side:
            scen.append({"nx": side, "ny": side, **{k: ctx.array((side + 2, side + 2), dt) for k in keys}})
        t, v = ctx.flood_ensemble_run(scen, params(), steps, dt)
        got = [scen[0][k].download() for k in keys[:3]] + [t[0]]
        first = first or got
        for x, y in zip(got, c[:3] + [tc] if dt == hip.F64 else first):
            assert np.array_equal(x, y), height
        assert np.allclose(v[0], vc, rtol=1e-13 if dt == hip.F64 else 1e-4, atol=0)


# dx on both sides of the range in which dt * d / dx is taken by the reciprocal and its remainder,
# some with inexact reciprocals; a dam breaks onto shallow and onto dry ground, so edges with the
# entropy fix and with a dry side meet edges without in one wave
@pytest.mark.parametrize("dx", [0.75, 1.0, 3.0000000000000004, 7.7, 2.0 ** 61])
def test_flood_f64_cell_sizes_bit_exact(ctx, dx):
    n, steps = 90, 12
    h = np.full((n + 2, n + 2), 0.05)
    h[:, :30] = 10.0
    h[40:60, 50:] = 0.0
    zero = np.zeros_like(h)
    arrs = [h, zero, zero.copy(), np.linspace(0.0, 3.0, n + 2) * np.ones_like(h), zero.copy()]
    d = [ctx.from_numpy(x, hip.F64) for x in arrs]
    t, v = ctx.flood_run(*d, n, n, hip.FloodParams(dx, CN, HEXTRA, DT_FALLBACK, 0.0, RAIN, 0.0), steps)
    c = [x.copy() for x in arrs]
    tc, vc, _ = oracle.flood_run(*c, n, n, dx, CN, HEXTRA, DT_FALLBACK, 0.0, RAIN, 0.0, steps)
    for a, b in zip(d[:3], c[:3]):
        assert np.array_equal(a.download(), b)
    assert np.array_equal(t, tc)
    assert np.allclose(v, vc, rtol=1e-13, atol=0)


@pytest.mark.parametrize("n,wet,steps", [(64, 0.0, 80), (90, 0.3, 50)])
def test_flood_f64_with_friction(ctx, n, wet, steps):
    arrs = scenario(n, 3100 + n, wet=wet)
    g, tg, vg = gpu_run(ctx, arrs, steps)
    c, tc, vc = cpu_run(arrs, steps)
    scale = np.max(np.abs(c[0])) + 1e-30
    assert np.max(np.abs(g[0] - c[0])) <= FLOOD_F64_RTOL * scale
    qs = max(np.max(np.abs(c[1])), np.max(np.abs(c[2])), 1e-30)
    assert np.max(np.abs(g[1] - c[1])) <= FLOOD_F64_RTOL * qs * 10
    assert np.allclose(tg, tc, rtol=1e-12)
    assert np.allclose(vg, vc, rtol=1e-10)


def test_flood_graph_form_matches_direct_launches(ctx):
    arrs = scenario(80, 3201, wet=0.1)
    steps = 45  # two captured chunks of 20 plus 5 direct steps
    a, ta, va = gpu_run(ctx, arrs, steps, hip.PLAIN)
    b, tb, vb = gpu_run(ctx, arrs, steps, hip.CHOSEN)
    for x, y in zip(a, b):
        assert np.array_equal(x, y)
    assert np.array_equal(ta, tb) and np.array_equal(va, vb)


def test_flood_graph_replays_repeatedly(ctx):
    # 5 replays of the captured 20-step chunk per call, four calls in a row with eager
    # work and synchronisation between them: every per-step record of every call must
    # equal the direct-launch run.  The chunk is captured once and cached: later calls
    # with the same shape and parameters replay it on their own (new) buffers, the last
    # one on another scenario of the same size
    runs = [scenario(64, 3211, wet=0.2)] * 3 + [scenario(64, 3212, wet=0.4)]
    refs = {}
    for call, arrs in enumerate(runs):
        if id(arrs) not in refs:
            refs[id(arrs)] = gpu_run(ctx, arrs, 100, hip.PLAIN)
        ref, tr, vr = refs[id(arrs)]
        scratch = ctx.array((1000,), hip.F64)
        ctx.fill_value(scratch, float(call))
        ctx.sync()
        got, tg, vg = gpu_run(ctx, arrs, 100, hip.CHOSEN)
        for x, y in zip(ref, got):
            assert np.array_equal(x, y), call
        assert np.array_equal(tr, tg) and np.array_equal(vr, vg), call
        scratch.free()
    a, b = (refs[id(r)][0][0] for r in (runs[0], runs[3]))
    assert not np.array_equal(a, b)  # the two scenarios differ


def test_flood_print_interval_clamp(ctx):
    arrs = scenario(40, 3301, wet=0.3)
    arrs[4][:] = 0.0
    g, tg, _ = gpu_run(ctx, arrs, 30, print_interval=7.0)
    c, tc, _ = cpu_run(arrs, 30, print_interval=7.0)
    assert np.array_equal(tg, tc)
    assert np.any(np.isclose(tg, 7.0, rtol=0, atol=1e-12))


def test_flood_f32_against_f64(ctx):
    n, steps = 128, 200
    a64 = scenario(n, 3401)
    c, tc, vc = cpu_run(a64, steps)
    a32 = [x.astype(np.float32) for x in a64]
    g, tg, vg = gpu_run(ctx, a32, steps, hip.CHOSEN)
    rel = np.linalg.norm(g[0].astype(np.float64) - c[0]) / np.linalg.norm(c[0])
    vmass = RAIN * n * n * DX * DX * tg
    print(f"[flood f32] rel-L2(h) {rel:.3e}; volume vs rain*A*t {np.max(np.abs(vg - vmass) / vmass):.3e}")
    assert rel < FLOOD_F32_H_RTOL
    assert np.max(np.abs(vg - vmass) / vmass) < 1e-5


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_flood_ensemble_matches_single_runs(ctx, dtype):
    sizes = [33, 64, 17, 100, 48]
    steps = 44
    dt = hip.F64 if dtype == np.float64 else hip.F32
    scen, singles = [], []
    for k, n in enumerate(sizes):
        arrs = scenario(n, 3500 + k, dtype, wet=0.2 if k % 2 else 0.0)
        d = [ctx.from_numpy(a, dt) for a in arrs]
        scen.append({"nx": n, "ny": n, "h": d[0], "qx": d[1], "qy": d[2], "z": d[3], "n2": d[4]})
        singles.append(gpu_run(ctx, arrs, steps, hip.PLAIN))
    t, v = ctx.flood_ensemble_run(scen, params(), steps, dt)
    for k, s in enumerate(scen):
        for x, y in zip((s["h"], s["qx"], s["qy"]), singles[k][0]):
            assert np.array_equal(x.download(), y), k
        assert np.array_equal(t[k], singles[k][1]) and np.array_equal(v[k], singles[k][2])


def test_flood_dem_device_matches_oracle(ctx):
    z = ctx.array((258, 258), hip.F64)
    ctx.flood_dem(z, 256, 256, DX, 77)
    ref = oracle.flood_dem(256, 256, DX, 77)
    # device exp vs glibc exp: a few ulps
    assert np.allclose(z.download(), ref, rtol=1e-14, atol=1e-12)


# ---------------------------------------------------------------------------------
# The config workload itself: scenarios of the 24-scenario ensemble (sides drawn from
# [512, 4096] by splitmix64 seed 1005, DEM seed 1005 + s), 2000 steps from a dry start
# under 50 mm/h of rain, against the FP64 oracle.  The two smallest sides (785 and 870,
# scenarios 23 and 4) keep the oracle to seconds.  Perturbing n^2 by a few ulps moves the
# oracle's fields by at most 3e-13 on these runs, so the FP64 bar is FLOOD_F64_RTOL.
# ---------------------------------------------------------------------------------
CONFIG_STEPS = 2000
CONFIG_SCEN = [(23, 785), (4, 870)]
_oracle_cache = {}


def config_scenario(s, n):
    z = oracle.flood_dem(n, n, DX, 1005 + s)
    return [np.zeros_like(z), np.zeros_like(z), np.zeros_like(z), z, np.full_like(z, 0.035 ** 2)]


def config_oracle(s, n):
    if (s, n) not in _oracle_cache:
        print(f"[flood config] oracle scenario {s} ({n}^2) x {CONFIG_STEPS} steps", flush=True)
        _oracle_cache[(s, n)] = cpu_run(config_scenario(s, n), CONFIG_STEPS)
    return _oracle_cache[(s, n)]


def test_flood_config_scenario_fp64_against_oracle(ctx):
    s, n = CONFIG_SCEN[0]
    (h, qx, qy), tc, vc = config_oracle(s, n)
    for variant in (hip.PLAIN, hip.CHOSEN):
        print(f"[flood config] GPU FP64 scenario {s} ({n}^2) variant {variant}", flush=True)
        g, tg, vg = gpu_run(ctx, config_scenario(s, n), CONFIG_STEPS, variant)
        for a, b in zip(g, (h, qx, qy)):
            assert np.abs(a - b).max() <= FLOOD_F64_RTOL * max(1.0, float(np.abs(b).max()))
        assert np.allclose(tg, tc, rtol=1e-12, atol=0) and np.allclose(vg, vc, rtol=1e-12, atol=0)
    assert h.max() > 0.1 and np.abs(qx).max() > 1e-3  # 2000 steps of rain made runoff


def test_flood_config_ensemble_against_oracle(ctx):
    """Config-range scenarios batched in one ensemble call (tile work-list over both,
    graph-captured step chunks), FP64 and the FP32 bulk form, each against the FP64
    oracle of its scenario."""
    refs = [config_oracle(s, n) for s, n in CONFIG_SCEN]
    for dtype in (np.float64, np.float32):
        dt = hip.F64 if dtype == np.float64 else hip.F32
        scen = []
        for s, n in CONFIG_SCEN:
            d = [ctx.from_numpy(a.astype(dtype), dt) for a in config_scenario(s, n)]
            scen.append({"nx": n, "ny": n, "h": d[0], "qx": d[1], "qy": d[2], "z": d[3], "n2": d[4]})
        print(f"[flood config] GPU ensemble dtype {dt}: {[n for _, n in CONFIG_SCEN]}", flush=True)
        t, v = ctx.flood_ensemble_run(scen, params(), CONFIG_STEPS, dt)
        for k, ((h, qx, qy), tc, vc) in enumerate(refs):
            gh = scen[k]["h"].download().astype(np.float64)
            if dtype == np.float64:
                for a, b in zip((gh, scen[k]["qx"].download(), scen[k]["qy"].download()), (h, qx, qy)):
                    assert np.abs(a - b).max() <= FLOOD_F64_RTOL * max(1.0, float(np.abs(b).max()))
                assert np.allclose(v[k], vc, rtol=1e-12, atol=0)
            else:
                rel = float(np.linalg.norm(gh - h) / np.linalg.norm(h))
                vrel = float(abs(v[k][-1] - vc[-1]) / vc[-1])
                print(f"[flood config] FP32 scenario {CONFIG_SCEN[k]}: h rel-L2 {rel:.3e}, "
                      f"volume rel {vrel:.3e}, simulated time {t[k][-1]:.3f} s (FP64 {tc[-1]:.3f} s)", flush=True)
                assert rel <= FLOOD_F32_CONFIG_H_RTOL and vrel <= FLOOD_F32_CONFIG_VOL_RTOL
