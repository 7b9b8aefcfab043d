"""GPU parity of the hand-written config kernels against the oracle.

Heat2D, GameOfLife and FDTD3d are integer work or fixed-order floating point with no
FMA contraction on either side, so the bar is bit-exact: the PLAIN and CHOSEN forms
must reproduce the oracle's bytes.  Full config sizes are covered through the oracle
for a few sweeps plus size-independent properties for the full sweep count.
"""
import hashlib
import json
import os
import time

import numpy as np
import pytest

import oracle
from appfis_amd import hip

pytestmark = pytest.mark.gpu

FDTD_COEFF = [0.5, 0.125, 0.0625, 0.125 / 3, 0.03125]


def _heat_pair(ctx, nx, ny, dt, seed=1001):
    a = np.zeros((ny + 2, nx + 2), dtype=np.float64 if dt == hip.F64 else np.float32)
    oracle.fill_uniform(a, 1, seed)
    return a, ctx.from_numpy(a, dt), ctx.array(a.shape, dt)


@pytest.mark.parametrize("dt", [hip.F64, hip.F32])
@pytest.mark.parametrize("nx,ny,iters", [(37, 29, 11), (64, 64, 16), (130, 67, 9), (1, 5, 3), (300, 250, 37)])
@pytest.mark.parametrize("variant", [hip.PLAIN, hip.CHOSEN])
def test_heat2d_bit_exact(ctx, dt, nx, ny, iters, variant):
    a, d0, d1 = _heat_pair(ctx, nx, ny, dt)
    ctx.heat2d(d0, d1, nx, ny, 0.1, iters, variant)
    ref = oracle.heat2d(a.copy(), np.zeros_like(a), nx, ny, 0.1, iters)
    got = (d0, d1)[iters % 2].download()
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("tsteps", [1, 3, 4, 8, 11, 16])
def test_heat2d_chosen_depths(ctx, tsteps):
    nx, ny, iters = 200, 150, 23
    a, d0, d1 = _heat_pair(ctx, nx, ny, hip.F64)
    ctx.heat2d(d0, d1, nx, ny, 0.1, iters, hip.CHOSEN, tsteps)
    ref = oracle.heat2d(a.copy(), np.zeros_like(a), nx, ny, 0.1, iters)
    assert np.array_equal((d0, d1)[iters % 2].download(), ref)


@pytest.mark.parametrize("dt", [hip.F64, hip.F32])
@pytest.mark.parametrize("nx,ny,iters", [(200, 150, 37), (5, 300, 19), (1030, 9, 21)])
def test_heat2d_every_candidate_bit_exact(ctx, dt, nx, ny, iters):
    # every temporal-blocking candidate the autotuner may pick, forced one at a time
    # (partial tiles in both axes; a grid narrower and one shorter than any tile)
    a, d0, d1 = _heat_pair(ctx, nx, ny, dt)
    ref = oracle.heat2d(a.copy(), np.zeros_like(a), nx, ny, 0.1, iters)
    names = hip.heat2d_candidates(dt)
    assert len(names) >= 2
    for i, name in enumerate(names):
        d0.upload(a)
        ctx.heat2d(d0, d1, nx, ny, 0.1, iters, hip.CANDIDATE0 + i)
        assert np.array_equal((d0, d1)[iters % 2].download(), ref), name


# 62 x 78 fills the window of the one-block form, 63 x 78 and 62 x 79 are the first that do not;
# at 400 x 420 every tiling has blocks with and without a side of the grid
@pytest.mark.parametrize("dt", [hip.F64, hip.F32])
@pytest.mark.parametrize("nx,ny", [(62, 78), (63, 78), (62, 79), (1, 1), (400, 420)])
@pytest.mark.parametrize("iters", [1, 2, 37])
def test_heat2d_windows(ctx, dt, nx, ny, iters):
    a, d0, d1 = _heat_pair(ctx, nx, ny, dt, seed=nx + ny)
    ref = oracle.heat2d(a.copy(), np.zeros_like(a), nx, ny, 0.1, iters)
    for variant in (hip.CHOSEN, *(hip.CANDIDATE0 + i for i in range(len(hip.heat2d_candidates(dt))))):
        d0.upload(a)
        d1.upload(np.zeros_like(a))
        ctx.heat2d(d0, d1, nx, ny, 0.1, iters, variant)
        assert np.array_equal((d0, d1)[iters % 2].download(), ref), variant


def test_heat2d_whole_grid_launch_split(ctx):
    # more sweeps than one launch of the one-block form takes
    nx, ny, iters = 30, 41, 2311
    a, d0, d1 = _heat_pair(ctx, nx, ny, hip.F64)
    ctx.heat2d(d0, d1, nx, ny, 0.1, iters, hip.CANDIDATE0 + len(hip.heat2d_candidates(hip.F64)) - 1)
    assert np.array_equal(d1.download(), oracle.heat2d(a.copy(), np.zeros_like(a), nx, ny, 0.1, iters))


# infinities, NaN and magnitudes of which four are (or grow to be) past the type's largest: every
# form has to give what the one-sweep form does, near them and in the tiles that hold none
@pytest.mark.parametrize("dt", [hip.F64, hip.F32])
@pytest.mark.parametrize("c", [0.1, 0.4, -3.0])
def test_heat2d_extreme_values(ctx, dt, c):
    nx, ny, iters = 150, 140, 19
    a, d0, d1 = _heat_pair(ctx, nx, ny, dt, seed=77)
    top = np.finfo(a.dtype).max
    a[30, 40], a[31, 90], a[100, 20], a[120, 130] = top / 2, top / 5, -top / 3, top / 1e5
    for special in (None, np.inf, np.nan):
        if special is not None:
            a[60, 145] = special
        d0.upload(a)
        d1.upload(np.zeros_like(a))
        ctx.heat2d(d0, d1, nx, ny, c, iters, hip.PLAIN)
        ref = d1.download()
        for variant in (hip.CHOSEN, *(hip.CANDIDATE0 + i for i in range(len(hip.heat2d_candidates(dt))))):
            d0.upload(a)
            d1.upload(np.zeros_like(a))
            ctx.heat2d(d0, d1, nx, ny, c, iters, variant)
            got = d1.download()
            assert np.array_equal(got[1:-1, 1:-1], ref[1:-1, 1:-1], equal_nan=True), (special, variant)
        d0.upload(a)
        d1.upload(np.zeros_like(a))
        ctx.heat2d_ensemble([(d0, d1, nx, ny)], c, iters)
        assert np.array_equal(d1.download()[1:-1, 1:-1], ref[1:-1, 1:-1], equal_nan=True), special


@pytest.mark.parametrize("dt", [hip.F64, hip.F32])
@pytest.mark.parametrize("iters", [1, 8, 23, 64])
def test_heat2d_ensemble_matches_oracle(ctx, dt, iters):
    # uneven grids advanced together (one launch per chunk over all grids, graph-replayed)
    sizes = [(1, 5), (37, 29), (130, 67), (300, 250), (64, 64), (2, 1), (513, 31)]
    grids, refs = [], []
    for k, (nx, ny) in enumerate(sizes):
        a, d0, d1 = _heat_pair(ctx, nx, ny, dt, seed=2000 + k)
        grids.append((d0, d1, nx, ny))
        refs.append(oracle.heat2d(a.copy(), np.zeros_like(a), nx, ny, 0.1, iters))
    ctx.heat2d_ensemble(grids, 0.1, iters)
    for (d0, d1, nx, ny), ref in zip(grids, refs):
        assert np.array_equal((d0, d1)[iters % 2].download(), ref), (nx, ny)


# ensembles for which the cost rule takes each of its tilings (most grids of the larger ones are
# uneven by a cell, so all have partial tiles)
@pytest.mark.parametrize("dt", [hip.F64, hip.F32])
@pytest.mark.parametrize("ngrid,side,iters", [(3, 70, 15), (3, 70, 16), (24, 143, 15), (24, 200, 16)])
def test_heat2d_ensemble_tilings(ctx, dt, ngrid, side, iters):
    grids, refs = [], []
    for k in range(ngrid):
        nx, ny = side + k % 3, side - k % 5
        a, d0, d1 = _heat_pair(ctx, nx, ny, dt, seed=2500 + k)
        grids.append((d0, d1, nx, ny))
        refs.append(oracle.heat2d(a.copy(), np.zeros_like(a), nx, ny, 0.1, iters))
    ctx.heat2d_ensemble(grids, 0.1, iters)
    for (d0, d1, nx, ny), ref in zip(grids, refs):
        assert np.array_equal((d0, d1)[iters % 2].download(), ref), (nx, ny)


def test_heat2d_ensemble_repeated_calls(ctx):
    # each call captures and replays its launch chain as a graph; three calls in a row on
    # the same grids (eager reductions between them) continue the same trajectory
    sizes = [(40, 33), (129, 70), (7, 200)]
    grids, arrs = [], []
    for k, (nx, ny) in enumerate(sizes):
        a, d0, d1 = _heat_pair(ctx, nx, ny, hip.F64, seed=2100 + k)
        grids.append((d0, d1, nx, ny))
        arrs.append(a)
    done, prev = 0, 0
    for call, iters in enumerate((9, 16, 7)):
        if prev % 2:  # the last call left the field in buffer 1: bring it to buffer 0
            for d0, d1, _, _ in grids:
                d0.upload(d1.download())
        ctx.heat2d_ensemble(grids, 0.1, iters)
        done += iters
        prev = iters
        for (d0, d1, nx, ny), a in zip(grids, arrs):
            ref = oracle.heat2d(a.copy(), np.zeros_like(a), nx, ny, 0.1, done)
            got = (d0, d1)[iters % 2].download()
            assert np.array_equal(got, ref), (call, nx, ny)
            ctx.reduce_sum_wide(d0, [1, nx + 1, 1, ny + 1])


def test_heat2d_ensemble_graph_reuse():
    # the launch chain is captured on the first call and replayed by later calls with
    # the same shapes and sweep count: a second set of grids (new buffers, new values)
    # must be advanced, not the first; after the context workspace is reallocated (a
    # flood run in between, on a fresh context whose workspace only held the heat
    # table) the chain is captured again
    sizes = [(40, 33), (129, 70), (7, 200)]
    iters = 16
    keep = []

    def one_set(c, seed):
        grids, arrs = [], []
        for k, (nx, ny) in enumerate(sizes):
            a, d0, d1 = _heat_pair(c, nx, ny, hip.F64, seed=seed + k)
            grids.append((d0, d1, nx, ny))
            arrs.append(a)
            keep.extend((d0, d1))
        return grids, arrs

    def check(c, grids, arrs, tag):
        c.heat2d_ensemble(grids, 0.1, iters)
        for (d0, d1, nx, ny), a in zip(grids, arrs):
            ref = oracle.heat2d(a.copy(), np.zeros_like(a), nx, ny, 0.1, iters)
            assert np.array_equal((d0, d1)[iters % 2].download(), ref), (tag, nx, ny)

    with hip.Context(0) as c:
        check(c, *one_set(c, 2200), "first")
        check(c, *one_set(c, 2300), "same shapes, new buffers")
        # grow the workspace: a flood run keeps three field copies of its grid there
        n = 300
        z = oracle.flood_dem(n, n, 10.0, 2400)
        zero = np.zeros_like(z)
        d = [c.from_numpy(x, hip.F64) for x in (zero, zero, zero, z, np.full_like(z, 0.035 ** 2))]
        keep.extend(d)
        c.flood_run(d[0], d[1], d[2], d[3], d[4], n, n, hip.FloodParams(10.0, 0.5, 1e-3, 1.0, 0.0, 1e-5, 0.0), 2,
                    hip.PLAIN)
        check(c, *one_set(c, 2500), "after the workspace grew")
        for x in keep:
            x.free()


def test_heat2d_full_config(ctx):
    # 1024^2 FP64, 500 sweeps: the whole config against the oracle
    nx = ny = 1024
    a, d0, d1 = _heat_pair(ctx, nx, ny, hip.F64)
    ref = oracle.heat2d(a.copy(), np.zeros_like(a), nx, ny, 0.1, 500)
    for variant in (hip.PLAIN, hip.CHOSEN):
        d0.upload(a)
        ctx.heat2d(d0, d1, nx, ny, 0.1, 500, variant)
        got = d0.download()
        assert np.array_equal(got, ref), variant
    print(f"[heat2d] checksum {ref.sum():.17g}")


def _gol_pair(ctx, nx, ny, seed=1002, p=0.25):
    a = np.zeros((ny + 2, nx + 2), dtype=np.uint8)
    oracle.fill_bernoulli(a, 1, seed, p)
    return a, ctx.from_numpy(a), ctx.array(a.shape, hip.U8)


@pytest.mark.parametrize("nx,ny,gens", [(14, 9, 5), (62, 40, 13), (64, 64, 10), (94, 33, 7), (126, 77, 21),
                                        (253, 101, 6), (1000, 19, 4), (510, 257, 31)])
def test_gol_plain_bit_exact(ctx, nx, ny, gens):
    # widths cover W = nx + 2 = 0 .. 15 mod 16 across the cases
    a, d0, d1 = _gol_pair(ctx, nx, ny)
    ctx.gol(d0, d1, nx, ny, gens, hip.PLAIN)
    ref = oracle.gol_u8(a.copy(), np.zeros_like(a), nx, ny, gens)
    assert np.array_equal((d0, d1)[gens % 2].download(), ref)


@pytest.mark.parametrize("nx", list(range(14, 30)))
def test_gol_plain_all_residues(ctx, nx):
    ny, gens = 23, 9
    a, d0, d1 = _gol_pair(ctx, nx, ny, seed=nx)
    ctx.gol(d0, d1, nx, ny, gens, hip.PLAIN)
    ref = oracle.gol_u8(a.copy(), np.zeros_like(a), nx, ny, gens)
    assert np.array_equal((d0, d1)[gens % 2].download(), ref)
    # the other buffer holds generation gens-1 with its ring exchanged
    prev = oracle.gol_u8(a.copy(), np.zeros_like(a), nx, ny, gens - 1)
    assert np.array_equal((d0, d1)[(gens + 1) % 2].download(), prev)


# rows of 16 bytes and less (cell by cell), the narrowest that are computed by chunks, boards of
# two rows (every chunk touches a ghost row), and chunks that end a ghost row and start the next
@pytest.mark.parametrize("nx,ny", [(2, 2), (14, 2), (15, 2), (15, 40), (16, 3), (17, 2), (30, 2), (45, 4), (1021, 2)])
def test_gol_plain_ghost_chunks(ctx, nx, ny):
    gens = 12
    a, d0, d1 = _gol_pair(ctx, nx, ny, seed=nx + ny, p=0.4)
    ctx.gol(d0, d1, nx, ny, gens, hip.PLAIN)
    assert np.array_equal(d0.download(), oracle.gol_u8(a.copy(), np.zeros_like(a), nx, ny, gens))
    assert np.array_equal(d1.download(), oracle.gol_u8(a.copy(), np.zeros_like(a), nx, ny, gens - 1))


def test_gol_full_config_prefix(ctx):
    # 8192^2 config: the first 12 generations against the oracle bit for bit
    nx = ny = 8192
    a, d0, d1 = _gol_pair(ctx, nx, ny)
    ctx.gol(d0, d1, nx, ny, 12, hip.PLAIN)
    ref = oracle.gol_u8(a.copy(), np.zeros_like(a), nx, ny, 12)
    assert np.array_equal(d0.download(), ref)


@pytest.mark.parametrize("nx,ny,gens", [(32, 2, 3), (32, 9, 1), (64, 64, 10), (96, 7, 13), (160, 33, 21),
                                        (256, 100, 2), (2048, 17, 5), (94, 33, 7), (50, 40, 6),
                                        (2048, 3, 40), (2048, 130, 37), (4096, 50, 33), (16384, 20, 19),
                                        (8192, 9, 2), (2048, 64, 1)])
def test_gol_chosen_both_buffers(ctx, nx, ny, gens):
    # bit-packed form (nx % 32 == 0; other widths take the byte kernel; nx % 2048 == 0
    # also runs the temporally blocked kernel): buf[gens % 2] holds generation gens and
    # the other buffer generation gens-1, rings exchanged
    a, d0, d1 = _gol_pair(ctx, nx, ny, seed=nx * 7 + ny)
    ctx.gol(d0, d1, nx, ny, gens, hip.CHOSEN)
    ref = oracle.gol_u8(a.copy(), np.zeros_like(a), nx, ny, gens)
    assert np.array_equal((d0, d1)[gens % 2].download(), ref)
    prev = oracle.gol_u8(a.copy(), np.zeros_like(a), nx, ny, gens - 1)
    assert np.array_equal((d0, d1)[(gens + 1) % 2].download(), prev)


@pytest.mark.parametrize("nx,ny,gens", [(2048, 45, 17), (4096, 30, 9), (8192, 21, 6),
                                        (8192, 32, 9), (8192, 64, 20), (8192, 96, 27)])
def test_gol_every_blocked_candidate(ctx, nx, ny, gens):
    # every blocked kernel of the bit-packed form, forced one at a time (candidates whose
    # block does not span nx refuse with an error); the 8192-cell rows with ny of one,
    # two and three 32-row bands put a band's periodic neighbours on itself or on the
    # same other band
    a, d0, d1 = _gol_pair(ctx, nx, ny, seed=nx + gens)
    ref = oracle.gol_u8(a.copy(), np.zeros_like(a), nx, ny, gens)
    prev = oracle.gol_u8(a.copy(), np.zeros_like(a), nx, ny, gens - 1)
    ran = []
    for i, name in enumerate(hip.gol_candidates()):
        d0.upload(a)
        try:
            ctx.gol(d0, d1, nx, ny, gens, hip.CANDIDATE0 + i)
        except hip.AppfisError as e:
            assert "spanned" in str(e) or "needs nx" in str(e), e
            continue
        ran.append(name)
        assert np.array_equal((d0, d1)[gens % 2].download(), ref), name
        assert np.array_equal((d0, d1)[(gens + 1) % 2].download(), prev), name
    assert len(ran) >= 3


@pytest.mark.parametrize("nx,ny,gens", [(32, 3, 20), (33, 5, 9), (40, 2, 26), (63, 64, 17), (64, 97, 33), (65, 17, 25),
                                        (1000, 77, 49), (1983, 40, 20), (1984, 33, 9), (1985, 50, 18), (2016, 20, 17),
                                        (4031, 49, 34), (6144, 30, 19), (8191, 100, 33), (31, 12, 9)])
def test_gol_windows_of_any_width(ctx, nx, ny, gens):
    # every window shape forced, and the one the rule takes, where the row ends inside, at and
    # just past a word and a window (62 stored words), in boards narrower than a window and
    # lower than a block (both wrap around several times); 31 cells run the byte kernel
    a, d0, d1 = _gol_pair(ctx, nx, ny, seed=nx * 11 + gens)
    ref = oracle.gol_u8(a.copy(), np.zeros_like(a), nx, ny, gens)
    prev = oracle.gol_u8(a.copy(), np.zeros_like(a), nx, ny, gens - 1)
    wins = [hip.CANDIDATE0 + i for i, name in enumerate(hip.gol_candidates()) if name.startswith("win ")]
    assert len(wins) >= 3
    for variant in [hip.CHOSEN] + (wins if nx >= 32 else []):
        d0.upload(a)
        ctx.gol(d0, d1, nx, ny, gens, variant)
        assert np.array_equal((d0, d1)[gens % 2].download(), ref), variant
        assert np.array_equal((d0, d1)[(gens + 1) % 2].download(), prev), variant


@pytest.mark.parametrize("nx,ny,gens", [(32, 3, 20), (33, 5, 9), (63, 64, 17), (65, 17, 25), (1000, 77, 49),
                                        (1984, 33, 9), (1985, 50, 18), (4031, 49, 34), (6144, 30, 19)])
def test_gol_windows_write_every_cell(ctx, nx, ny, gens):
    # as above with both buffers filled anew before each form: a cell left out, in either buffer or
    # its ring, keeps a value that no board holds
    a, d0, d1 = _gol_pair(ctx, nx, ny, seed=nx * 13 + gens)
    ref = oracle.gol_u8(a.copy(), np.zeros_like(a), nx, ny, gens)
    prev = oracle.gol_u8(a.copy(), np.zeros_like(a), nx, ny, gens - 1)
    wins = [hip.CANDIDATE0 + i for i, name in enumerate(hip.gol_candidates()) if name.startswith("win ")]
    b = a.copy()
    b[[0, -1], :] = b[:, [0, -1]] = 9
    for variant in [hip.PLAIN, hip.CHOSEN] + wins:
        d0.upload(a if variant == hip.PLAIN else b)  # the packed forms read no ring
        d1.upload(np.full_like(a, 7))
        ctx.gol(d0, d1, nx, ny, gens, variant)
        assert np.array_equal((d0, d1)[gens % 2].download(), ref), variant
        assert np.array_equal((d0, d1)[(gens + 1) % 2].download(), prev), variant


@pytest.mark.parametrize("gens", [2, 7, 8, 9, 16, 17, 24, 25])
def test_gol_full_row_launch_split(ctx, gens):
    # the full-row form runs a call's generations in at least two launches, the first
    # packing and the last unpacking the uint8 field (up to G = 8 generations: n-1 and 1;
    # beyond: G per launch and the rest in the last): generation counts around G and 2G,
    # both buffers against the oracle
    nx, ny = 2048, 40
    names = hip.gol_candidates()
    a, d0, d1 = _gol_pair(ctx, nx, ny, seed=gens + 500)
    ctx.gol(d0, d1, nx, ny, gens, hip.CANDIDATE0 + names.index("tw1 k3 g8 w16"))
    ref = oracle.gol_u8(a.copy(), np.zeros_like(a), nx, ny, gens)
    prev = oracle.gol_u8(a.copy(), np.zeros_like(a), nx, ny, gens - 1)
    assert np.array_equal((d0, d1)[gens % 2].download(), ref)
    assert np.array_equal((d0, d1)[(gens + 1) % 2].download(), prev)


def test_gol_chosen_glider_period(ctx):
    # a glider on an N x N torus returns to its start after 4N generations
    n = 64
    a = np.zeros((n + 2, n + 2), dtype=np.uint8)
    for x, y in [(2, 1), (3, 2), (1, 3), (2, 3), (3, 3)]:
        a[y + 1, x + 1] = 1
    d0, d1 = ctx.from_numpy(a), ctx.array(a.shape, hip.U8)
    ctx.gol(d0, d1, n, n, 4 * n, hip.CHOSEN)
    got = d0.download()
    assert np.array_equal(got[1:-1, 1:-1], a[1:-1, 1:-1])
    ctx.gol(d0, d1, n, n, 2 * n, hip.CHOSEN)
    assert not np.array_equal(d0.download()[1:-1, 1:-1], a[1:-1, 1:-1])


def test_gol_chosen_full_config_prefix(ctx):
    # 8192^2 config: 12 generations of the bit-packed form against the oracle, and
    # 100 generations against the byte kernel
    nx = ny = 8192
    a, d0, d1 = _gol_pair(ctx, nx, ny)
    ctx.gol(d0, d1, nx, ny, 12, hip.CHOSEN)
    ref = oracle.gol_u8(a.copy(), np.zeros_like(a), nx, ny, 12)
    assert np.array_equal(d0.download(), ref)
    del ref
    d0.upload(a)
    ctx.gol(d0, d1, nx, ny, 100, hip.CHOSEN)
    c0, c1 = d0.download(), d1.download()
    d0.upload(a)
    ctx.gol(d0, d1, nx, ny, 100, hip.PLAIN)
    assert np.array_equal(d0.download(), c0) and np.array_equal(d1.download(), c1)


def test_gol_full_config_every_100th_generation(ctx):
    # the 8192^2 config for 1000 generations, checked at every 100th generation against
    # the oracle: tests/golden/gol_8192.json holds the SHA-256 of the oracle's interior and
    # its live count at generations 100..1000 (tests/golden/make_gol_golden.py); both the
    # byte kernel and the bit-packed kernel must hit every digest, and agree on both
    # buffers (the other one holds the previous generation with its ring)
    gold = json.load(open(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "gol_8192.json")))
    nx, ny = gold["nx"], gold["ny"]
    a = np.zeros((ny + 2, nx + 2), dtype=np.uint8)
    oracle.fill_bernoulli(a, 1, gold["seed"], gold["p"])
    p0, p1 = ctx.from_numpy(a), ctx.array(a.shape, hip.U8)
    c0, c1 = ctx.from_numpy(a), ctx.array(a.shape, hip.U8)
    for rec in gold["records"]:
        ctx.gol(p0, p1, nx, ny, 100, hip.PLAIN)
        ctx.gol(c0, c1, nx, ny, 100, hip.CHOSEN)
        got_p, got_c = p0.download(), c0.download()
        gen = rec["generation"]
        for form, got in (("plain", got_p), ("chosen", got_c)):
            interior = np.ascontiguousarray(got[1:-1, 1:-1])
            assert int(interior.sum(dtype=np.int64)) == rec["live"], (form, gen)
            assert hashlib.sha256(interior.tobytes()).hexdigest() == rec["sha256"], (form, gen)
        assert np.array_equal(got_p, got_c), gen
        assert np.array_equal(p1.download(), c1.download()), gen
        print(f"[gol] generation {gen}: live {rec['live']} (both forms match the oracle)", flush=True)


def _fdtd_pair(ctx, n, dt, seed=1004):
    npdt = {hip.F32: np.float32, hip.F64: np.float64, hip.F16: np.float16, hip.BF16: np.uint16}[dt]
    shape = tuple(x + 8 for x in n[::-1])
    a = np.zeros(shape, dtype=npdt)
    oracle.fill_uniform(a, 4, seed, bf16=(dt == hip.BF16))
    return a, ctx.from_numpy(a, dt), ctx.array(shape, dt)


@pytest.mark.parametrize("variant", [hip.PLAIN, hip.CHOSEN])
@pytest.mark.parametrize("dt", [hip.F32, hip.F64, hip.F16, hip.BF16])
@pytest.mark.parametrize("n,steps", [((37, 29, 23), 4), ((64, 64, 64), 3), ((70, 17, 130), 2), ((130, 66, 70), 3)])
def test_fdtd3d_bit_exact(ctx, dt, n, steps, variant):
    nx, ny, nz = n
    coeff = FDTD_COEFF if dt not in (hip.F16,) else [c / 2.0625 for c in FDTD_COEFF]
    a, d0, d1 = _fdtd_pair(ctx, n, dt)
    ctx.fdtd3d(d0, d1, nx, ny, nz, coeff, steps, variant)
    ref = oracle.fdtd3d(a.copy(), np.zeros_like(a), nx, ny, nz, coeff, steps, bf16=(dt == hip.BF16))
    got = (d0, d1)[steps % 2].download()
    assert np.array_equal(got.view(np.uint8), ref.view(np.uint8))


@pytest.mark.parametrize("dt", [hip.F32, hip.F64, hip.F16, hip.BF16])
@pytest.mark.parametrize("n", [(70, 33, 40), (68, 21, 37), (71, 30, 19), (68, 9, 259), (68, 1, 1), (68, 2, 3)])
def test_fdtd3d_every_candidate_bit_exact(ctx, dt, n):
    # every tiling the autotuner may pick, forced one at a time; nx = 70, 68, 71 covers
    # x points per lane (1, 2, 4) that do and do not divide nx, nz = 259 gives the
    # 64- to 256-plane z-chunks a last chunk of 3 planes (fewer than a prefetch ring),
    # and one plane of one row / three planes of two rows leave every prefetch short
    coeff = FDTD_COEFF if dt != hip.F16 else [c / 2.0625 for c in FDTD_COEFF]
    a, d0, d1 = _fdtd_pair(ctx, n, dt)
    ref = oracle.fdtd3d(a.copy(), np.zeros_like(a), *n, coeff, 3, bf16=(dt == hip.BF16))
    names = hip.fdtd3d_candidates(dt)
    assert len(names) >= 2
    ran = 0
    for i, name in enumerate(names):
        d0.upload(a)
        try:
            ctx.fdtd3d(d0, d1, *n, coeff, 3, hip.CANDIDATE0 + i)
        except hip.AppfisError as e:
            if name.startswith("dma "):  # direct-to-LDS rows: whole 16-byte chunks per row
                assert "needs nx + 8 divisible" in str(e) and (n[0] + 8) * np.dtype(a.dtype).itemsize % 16, e
            else:  # a candidate whose x points per lane do not divide nx
                assert "needs nx" in str(e) and int(name.split()[0][2:]) > 1 and n[0] % int(name.split()[0][2:]), e
            continue
        ran += 1
        assert np.array_equal(d1.download().view(np.uint8), ref.view(np.uint8)), name
    assert ran >= 2


@pytest.mark.parametrize("dt", [hip.F64, hip.F32])
@pytest.mark.parametrize("nx,ny", [(40, 33), (96, 80), (333, 250)])
def test_heat2d_chosen_calls_of_few_sweeps(ctx, dt, nx, ny):
    # one and two sweeps one by one, up to 16 in shallow tiles where these need no more launches
    for it in range(1, 20):
        a, d0, d1 = _heat_pair(ctx, nx, ny, dt)
        ctx.heat2d(d0, d1, nx, ny, 0.1, it, hip.CHOSEN)
        ref = oracle.heat2d(a.copy(), np.zeros_like(a), nx, ny, 0.1, it)
        assert np.array_equal((d0, d1)[it % 2].download(), ref), it


def test_heat2d_call_of_one_sweep_loads_no_halo(ctx):
    # one sweep of 2048 x 2048 in FP32 takes 8 us without a halo, 12 in tiles with one of 12 cells
    n = 2048
    d0, d1 = (ctx.array((n + 2, n + 2), hip.F32) for _ in range(2))
    ms = {}
    for v in (hip.PLAIN, hip.CHOSEN, hip.PLAIN, hip.CHOSEN):
        for _ in range(8):
            ctx.timer_start()
            for _ in range(20):
                ctx.heat2d(d0, d1, n, n, 0.1, 1, v)
            ms[v] = min(ms.get(v, 1e9), ctx.timer_stop())
    assert ms[hip.CHOSEN] < 1.25 * ms[hip.PLAIN], ms


@pytest.mark.parametrize("nx", [2, 3, 5, 12, 13, 14, 15, 16, 17, 30])
def test_gol_byte_kernel_on_narrow_boards(ctx, nx):
    # padded rows shorter than the kernel's 16-byte chunk, equal to it and longer; both buffers with
    # their rings: generation n and, in the other, n - 1
    for ny in (2, 3, 21, 700):
        a = np.zeros((ny + 2, nx + 2), dtype=np.uint8)
        oracle.fill_bernoulli(a, 1, 73 + nx, 0.4)
        d = [ctx.from_numpy(a), ctx.from_numpy(np.full_like(a, 1))]
        ctx.gol(d[0], d[1], nx, ny, 3, hip.PLAIN)
        for gens, got in ((3, d[1]), (2, d[0])):
            ref = oracle.gol_u8(a.copy(), np.zeros_like(a), nx, ny, gens)[1:-1, 1:-1]
            assert np.array_equal(got.download(), np.pad(ref, 1, mode="wrap")), (ny, gens)


# board, generations, launches of the packed generations: two generations and tall boards of few
# words go one by one (all but the last, which unpacks), short calls of 2048 cells a row run in
# full-row waves (8 generations a launch, conversions included), all others in windows
@pytest.mark.parametrize("nx,ny,gens,launches", [
    (32, 3, 2, 1), (32, 5, 3, 1), (96, 96, 2, 1), (96, 97, 3, 1), (64, 300001, 2, 1), (64, 300001, 5, 4),
    (2048, 7, 2, 2), (2048, 65, 8, 2), (2048, 65, 9, 2), (2048, 300, 19, 3)])
def test_gol_short_calls_and_tall_boards(ctx, nx, ny, gens, launches):
    a = np.zeros((ny + 2, nx + 2), dtype=np.uint8)
    oracle.fill_bernoulli(a, 1, 71, 0.3)
    d0, d1 = ctx.from_numpy(a), ctx.from_numpy(np.full_like(a, 1))
    ctx.gol(d0, d1, nx, ny, gens, hip.CHOSEN)  # tunes the shape
    d0.upload(a)
    d1.upload(np.full_like(a, 1))
    ctx.kernel_timing(True)
    ctx.gol(d0, d1, nx, ny, gens, hip.CHOSEN)
    got = ctx.kernel_time()[1]
    ctx.kernel_timing(False)
    e = [ctx.from_numpy(a), ctx.from_numpy(np.full_like(a, 1))]
    ctx.gol(e[0], e[1], nx, ny, gens, hip.PLAIN)
    ref = oracle.gol_u8(a.copy(), np.zeros_like(a), nx, ny, gens)
    assert np.array_equal((d0, d1)[gens % 2].download()[1:-1, 1:-1], ref[1:-1, 1:-1])
    for x, y in zip((d0, d1), e):  # both buffers, rings included
        assert np.array_equal(x.download(), y.download())
    assert got == launches


@pytest.mark.parametrize("dt", [hip.F32, hip.F64, hip.F16, hip.BF16])
@pytest.mark.parametrize("n", [(5, 3, 1), (66, 9, 2), (100, 101, 103), (127, 131, 140), (162, 161, 163), (257, 257, 260),
                               (256, 264, 260), (301, 330, 340), (321, 330, 640)])
def test_fdtd3d_tilings_by_size(ctx, dt, n):
    # the fixed tiling and the planes per block follow the grid: one plane, chunks of two, and
    # sizes on either side of 1, 2, 4, 16, 24, 32 and 64 million points, even and odd widths
    nx, ny, nz = n
    if nx * ny * nz > 60e6 and dt == hip.F64:
        pytest.skip("the FP64 lines all lie below")
    coeff = FDTD_COEFF if dt != hip.F16 else [c / 2.0625 for c in FDTD_COEFF]
    a, d0, d1 = _fdtd_pair(ctx, n, dt)
    ref = oracle.fdtd3d(a.copy(), np.zeros_like(a), nx, ny, nz, coeff, 1, bf16=(dt == hip.BF16))
    for variant in (hip.PLAIN, hip.CHOSEN):
        ctx.fdtd3d(d0, d1, nx, ny, nz, coeff, 1, variant)
        assert np.array_equal(d1.download(), ref)


@pytest.mark.parametrize("dt", [hip.F32, hip.F64, hip.F16, hip.BF16])
@pytest.mark.parametrize("n", [(5, 3, 1), (64, 32, 2), (66, 9, 3), (40, 33, 61), (100, 101, 103), (127, 131, 140),
                               (162, 161, 163), (257, 130, 301), (256, 264, 260), (321, 330, 340)])
def test_fdtd3d_tilings_write_every_point(ctx, dt, n):
    # NaN in the target before each form: a point that a dropped plane, chunk or tile leaves out
    # stays one.  One plane, two, odd counts that the chunks do not divide, the sizes between which
    # PLAIN's tilings change
    nx, ny, nz = n
    coeff = FDTD_COEFF if dt != hip.F16 else [c / 2.0625 for c in FDTD_COEFF]
    a, d0, d1 = _fdtd_pair(ctx, n, dt)
    ref = oracle.fdtd3d(a.copy(), np.zeros_like(a), nx, ny, nz, coeff, 1, bf16=(dt == hip.BF16))
    blank = np.zeros_like(a)
    blank[4:-4, 4:-4, 4:-4] = 0x7FC0 if dt == hip.BF16 else np.nan
    for variant in (hip.PLAIN, hip.CHOSEN):
        d1.upload(blank)
        ctx.fdtd3d(d0, d1, nx, ny, nz, coeff, 1, variant)
        assert np.array_equal(d1.download().view(np.uint8), ref.view(np.uint8)), variant


def test_fdtd3d_chosen_call_costs_the_host_no_tuning(ctx):
    # a call on a tuned shape launches its kernel and no more, whatever the number of planes:
    # preparing the tuning took this column 100 ms and more of the host's time, a launch takes
    # some 10 us
    n = (1, 1, 1000000)
    _, d0, d1 = _fdtd_pair(ctx, n, hip.F32)
    ctx.fdtd3d(d0, d1, *n, FDTD_COEFF, 1, hip.CHOSEN)
    ctx.sync()
    t = []
    for _ in range(3):
        t0 = time.perf_counter()
        ctx.fdtd3d(d0, d1, *n, FDTD_COEFF, 1, hip.CHOSEN)
        t.append(time.perf_counter() - t0)
        ctx.sync()
    assert min(t) < 5e-3, t


def test_fdtd3d_plain_call_costs_the_host_no_loop_over_planes(ctx):
    # the planes of a block are chosen from a few dozen counts: trying every one took this column
    # some 30 ms of the host's time in each call, a launch takes some 10 us
    n = (1, 1, 4000000)
    _, d0, d1 = _fdtd_pair(ctx, n, hip.F16)
    ctx.fdtd3d(d0, d1, *n, FDTD_COEFF, 1, hip.PLAIN)
    ctx.sync()
    t = []
    for _ in range(3):
        t0 = time.perf_counter()
        ctx.fdtd3d(d0, d1, *n, FDTD_COEFF, 1, hip.PLAIN)
        t.append(time.perf_counter() - t0)
        ctx.sync()
    assert min(t) < 5e-3, t


@pytest.mark.parametrize("dt", [hip.F32, hip.F64, hip.BF16])
def test_fdtd3d_more_rows_than_low_tiles_reach(ctx, dt):
    # 540000 rows are 67500 tiles of 8 rows, over a launch's 65536: taller tiles take them
    n = (1, 540000, 1)
    a, d0, d1 = _fdtd_pair(ctx, n, dt)
    ref = oracle.fdtd3d(a.copy(), np.zeros_like(a), *n, FDTD_COEFF, 1, bf16=(dt == hip.BF16))
    for variant in (hip.PLAIN, hip.CHOSEN):
        d1.upload(np.zeros_like(a))
        ctx.fdtd3d(d0, d1, *n, FDTD_COEFF, 1, variant)
        assert np.array_equal(d1.download(), ref), variant


def test_fdtd3d_streaming_tilings_keep_long_blocks(ctx):
    # 512^3 in FP32: the direct-to-LDS tilings, one block to a CU, march 256 planes each (128 in two
    # rounds take 241 us a sweep for 212)
    n = (512, 512, 512)
    d0, d1 = (ctx.array(tuple(x + 8 for x in n), hip.F32) for _ in range(2))
    ctx.fdtd3d(d0, d1, *n, FDTD_COEFF, 2, hip.CHOSEN)
    report = [x for x in ctx.tune_report().splitlines() if "kernel 3 dtype 2 shape 512x512x512" in x][-1]
    for tiling in ("dma ty16 ry2 zc256 d2", "dma ty16 ry2 zc256 d3", "dma ty8 ry4 zc256 d2"):
        assert tiling in report, report


@pytest.mark.parametrize("dt,off", [(hip.F32, 4), (hip.F64, 8), (hip.F16, 2), (hip.BF16, 2)])
def test_fdtd3d_on_unaligned_buffers(ctx, dt, off):
    # buffers that start `off` bytes into an allocation, so that the preferred tilings'
    # alignment fails (16 bytes for the direct-to-LDS rows, 4 for the 16-bit pairs):
    # PLAIN and CHOSEN fall back to tilings that fit and stay bit-exact (nx + 8 = 72 and
    # an even nx would otherwise admit them)
    from types import SimpleNamespace
    n = (64, 20, 17)
    coeff = FDTD_COEFF if dt != hip.F16 else [c / 2.0625 for c in FDTD_COEFF]
    a, d0, d1 = _fdtd_pair(ctx, n, dt)
    ref = oracle.fdtd3d(a.copy(), np.zeros_like(a), *n, coeff, 3, bf16=(dt == hip.BF16))
    big = [ctx.array((a.nbytes + 64,), hip.U8) for _ in range(2)]
    bufs = [SimpleNamespace(ptr=b.ptr + off, dtype=dt) for b in big]
    for variant in (hip.PLAIN, hip.CHOSEN):
        print(f"[fdtd unaligned] dtype {dt} offset {off} variant {variant}", flush=True)
        hip.check(hip.lib().appfis_memcpy_h2d(ctx.handle, bufs[0].ptr, a.ctypes.data, a.nbytes), "h2d")
        ctx.fdtd3d(bufs[0], bufs[1], *n, coeff, 3, variant)
        got = np.empty_like(a)
        hip.check(hip.lib().appfis_memcpy_d2h(ctx.handle, got.ctypes.data, bufs[1].ptr, a.nbytes), "d2h")
        assert np.array_equal(got.view(np.uint8), ref.view(np.uint8)), variant


# unit roundoff of the storage formats: every sweep rounds each stored value once
FDTD_UNIT_ROUNDOFF = {hip.F32: 2.0 ** -24, hip.F16: 2.0 ** -11, hip.BF16: 2.0 ** -8}


def test_fdtd3d_full_config(ctx):
    """512^3, 100 sweeps.  FP32 two sweeps bit-exact against the oracle; FP64 (the
    reference dtype) all 100 sweeps bit-exact against the oracle's FP64; FP32, FP16 and
    BF16 storage (CHOSEN tiling) against that FP64 field, on normalised fields
    u / 2.0625^n (FP16 runs with the coefficients divided by 2.0625, so its field is
    already normalised).

    Bound: the seeded input is rounded to the storage type once and every sweep rounds
    each stored value once (relative error <= u, the unit roundoff, each time); the
    normalised operator has non-negative weights summing to 1 with a zero halo, so it
    does not amplify earlier errors in the max norm or the L2 norm.  After n sweeps the
    normalised max-abs error is at most (n + 1) * u * max|u0| (max|u0| < 1) and the
    relative L2 error at most (n + 1) * u * |u0| / |u_n|, asserted as 2 (n + 1) u after
    checking |u_n| / |u0| > 0.5 (the mean 0.5 of the seeded field survives 100 sweeps in
    the interior)."""
    n = (512, 512, 512)
    steps = 100
    scale = 2.0625 ** steps
    a, d0, d1 = _fdtd_pair(ctx, n, hip.F32)
    ctx.fdtd3d(d0, d1, *n, FDTD_COEFF, 2)
    ref = oracle.fdtd3d(a.copy(), np.zeros_like(a), *n, FDTD_COEFF, 2)
    assert np.array_equal(d0.download(), ref)
    del ref, d0, d1
    # FP64: the oracle for all 100 sweeps, and the GPU bit-identical to it
    a64 = np.zeros(a.shape)
    oracle.fill_uniform(a64, 4, 1004)
    f64 = oracle.fdtd3d(a64.copy(), np.zeros_like(a64), *n, FDTD_COEFF, steps)
    assert np.linalg.norm(f64.ravel()) / np.linalg.norm(a64.ravel()) / scale > 0.5
    e0, e1 = ctx.from_numpy(a64), ctx.array(a64.shape, hip.F64)
    ctx.fdtd3d(e0, e1, *n, FDTD_COEFF, steps, hip.CHOSEN)
    assert np.array_equal(e0.download(), f64)
    print(f"[fdtd3d] FP64 512^3 x {steps}: bit-identical to the oracle", flush=True)
    del e0, e1
    f64 /= scale
    norm64 = np.linalg.norm(f64.ravel())
    for dt in (hip.F32, hip.F16, hip.BF16):
        coeff = FDTD_COEFF if dt != hip.F16 else [c / 2.0625 for c in FDTD_COEFF]
        b, b0, b1 = _fdtd_pair(ctx, n, dt)
        ctx.fdtd3d(b0, b1, *n, coeff, steps, hip.CHOSEN)
        raw = b0.download()
        del b, b0, b1
        if dt == hip.BF16:
            got = (raw.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
        else:
            got = raw.astype(np.float64)
        if dt != hip.F16:
            got /= scale
        diff = got - f64
        max_abs = float(np.abs(diff).max())
        rel_l2 = float(np.linalg.norm(diff.ravel()) / norm64)
        bound = (steps + 1) * FDTD_UNIT_ROUNDOFF[dt]
        print(f"[fdtd3d] dtype {dt} vs FP64 after {steps} sweeps (normalised): max-abs {max_abs:.3e} "
              f"rel-L2 {rel_l2:.3e} (bound {bound:.3e})", flush=True)
        assert max_abs <= bound and rel_l2 <= 2 * bound
        del got, diff, raw