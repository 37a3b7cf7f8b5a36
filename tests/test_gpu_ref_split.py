"""Sweeps on the caller's layout by the lane-split kernel (tuning key ref_split, on by default for
tsw_sweep_apply and tsw_sweep_apply_multi with the staggered pattern's default tuning): the oracle's
sweep (FP64 within 1e-12, FP32 within 2e-6, TSW_MIXED as FP64), the same bits as the diagonal-layout
path (ref_split -1), row bands with exchange records (meshes taller than one workgroup's rows), many
right-hand sides against single sweeps, misaligned device arrays through the conversions, and the
forced stall path."""
import math

import numpy as np
import pytest

import tsw
from _common import ls_ordinates, orc_sweep, random_problem, rel_err

pytestmark = pytest.mark.gpu


def _ctx(g, o, ref_split=1):
    c = tsw.Context(0)
    c.problem_set(g.nx, g.ny, g.p, o.xi, o.eta, o.w, o.quad_off, g.ax, g.bx, g.ay, g.by)
    c.set_pattern("hip-staggered")
    c.set_tuning("ref_split", ref_split)
    return c


# (nx, ny, p): one band; two bands at degree 1 (256 rows per workgroup) and 2-3 (128 rows)
SHAPES = [(17, 23, 1), (11, 300, 1), (21, 40, 2), (13, 150, 2), (9, 31, 3), (12, 170, 3)]


@pytest.mark.parametrize("dt", [math.inf, 0.3])
@pytest.mark.parametrize("shape", SHAPES)
def test_ref_split_sweep_matches_oracle_and_diagonal_path(shape, dt):
    nx, ny, p = shape
    o = ls_ordinates(6)
    g, st, _, src = random_problem(nx, ny, p, o, seed=900 + nx + p, materials=3)
    print("ref split", shape, dt, flush=True)
    ref = orc_sweep(g, o, st, src, dt)
    outs = {}
    for rs in (1, -1):
        with _ctx(g, o, rs) as c:
            for prec in (tsw.FP64, tsw.FP32, tsw.MIXED):
                out = src.copy()
                c.sweep(out, st, dt, precision=prec)
                outs[rs, prec] = out
                if rs == 1:
                    assert c.get_tuning("lane_split") == 1
    for prec, tol in ((tsw.FP64, 1e-12), (tsw.FP32, 2e-6), (tsw.MIXED, 1e-12)):
        assert rel_err(outs[1, prec], ref) <= tol, prec
        np.testing.assert_array_equal(outs[1, prec][0], src[0])
        np.testing.assert_array_equal(outs[1, prec][:, -1], src[:, -1])
    # the same arithmetic as the diagonal-layout kernels (TSW_MIXED there refines an FP32 sweep)
    np.testing.assert_array_equal(outs[1, tsw.FP64], outs[-1, tsw.FP64])
    np.testing.assert_array_equal(outs[1, tsw.FP32], outs[-1, tsw.FP32])
    np.testing.assert_array_equal(outs[1, tsw.MIXED], outs[1, tsw.FP64])


def test_ref_split_multi_equals_single_sweeps_and_misaligned_fallback():
    import torch
    o = ls_ordinates(8)
    g, st, _, src = random_problem(14, 160, 2, o, seed=911, materials=4)
    rng = np.random.default_rng(5)
    srcs = [src + rng.uniform(0, 1, size=src.shape) * (k % 2) for k in range(5)]
    dev = torch.device("cuda:0")
    with _ctx(g, o) as c:
        st_d = torch.from_numpy(st).to(dev)
        for prec in (tsw.FP64, tsw.FP32):
            one = []
            for s_ in srcs:
                a = torch.from_numpy(s_).to(dev)
                c.sweep(a, st_d, math.inf, precision=prec)
                one.append(a)
            many = [torch.from_numpy(s_).to(dev) for s_ in srcs]
            c.sweep_multi(many, st_d, math.inf, precision=prec)
            big = torch.zeros(src.size + 1, dtype=torch.float64, device=dev)
            shifted = big[1:].view(src.shape)  # 8 bytes off a 16-byte boundary: the conversions
            shifted.copy_(torch.from_numpy(srcs[0]))
            c.sweep(shifted, st_d, math.inf, precision=prec)
            torch.cuda.synchronize()
            for a, b in zip(one, many):
                assert torch.equal(a, b), prec
            assert torch.equal(one[0], shifted), prec
        assert rel_err(one[0].cpu().numpy(), orc_sweep(g, o, st, srcs[0], math.inf)) <= 2e-6


def test_ref_split_band_stall_is_reported_and_recovered():
    o = ls_ordinates(4)
    g, st, _, src = random_problem(30, 140, 2, o, seed=812, materials=3)
    ref = orc_sweep(g, o, st, src)
    with _ctx(g, o) as c:
        for prec, tol in ((tsw.FP64, 1e-12), (tsw.FP32, 2e-6)):
            out = src.copy()
            c.sweep(out, st, precision=prec)
            assert rel_err(out, ref) <= tol
            c.set_tuning("stall_test", 1)
            with pytest.raises(tsw.TswError) as ei:
                c.sweep(src.copy(), st, precision=prec)
            assert ei.value.code == tsw.TSW_E_HIP and "stalled" in str(ei.value)
            for _ in range(2):
                out = src.copy()
                c.sweep(out, st, precision=prec)
                assert rel_err(out, ref) <= tol, prec


# rows at the wave (16 or 32 row slots), workgroup (192, 64, 96) and band edges, columns below and at the prefetch
# ring and the halo ring (rows of a wave), one ordinate per quadrant and more than a workgroup per XCD
EDGES = [(1, 1, 1, 2), (3, 33, 1, 8), (33, 192, 1, 2), (31, 193, 1, 4), (2, 385, 1, 4), (1, 16, 2, 2), (15, 17, 2, 8),
         (17, 64, 2, 2), (16, 65, 2, 4), (5, 129, 2, 12), (4, 15, 3, 4), (18, 96, 3, 2), (7, 97, 3, 8), (33, 193, 3, 4)]


@pytest.mark.parametrize("persistent", [1, 0])
@pytest.mark.parametrize("shape", EDGES)
def test_ref_split_edges_match_the_diagonal_path(shape, persistent):
    nx, ny, p, order = shape
    o = ls_ordinates(order)
    g, st, _, src = random_problem(nx, ny, p, o, seed=40 + nx + ny, materials=2)
    print("ref split edges", shape, persistent, flush=True)
    for prec, tol in ((tsw.FP64, 1e-12), (tsw.FP32, 2e-6)):
        a, b, c2 = src.copy(), src.copy(), src.copy()
        with _ctx(g, o, 1) as c:
            c.set_tuning("batch_persistent", persistent)
            c.sweep(a, st, 0.7, precision=prec)
            c.sweep(c2, st, 0.7, precision=prec)  # the other set of counters
        with _ctx(g, o, -1) as c:
            c.sweep(b, st, 0.7, precision=prec)
        assert rel_err(a, orc_sweep(g, o, st, src, 0.7)) <= tol, prec
        np.testing.assert_array_equal(a, b)
        np.testing.assert_array_equal(a, c2)


# the lane-split kernel itself (batch_split_rows set), with storer waves in bands of up to 192, 96 and 96 rows, and without
# in bands of up to 256, 128 and 128
@pytest.mark.parametrize("persistent", [1, 0])
@pytest.mark.parametrize("storers", [1, -1])
@pytest.mark.parametrize("shape", EDGES + [(3, 256, 1, 2), (2, 257, 1, 2), (5, 128, 2, 2), (3, 97, 2, 4), (6, 128, 3, 2)])
def test_ref_split_with_and_without_storers(shape, storers, persistent):
    nx, ny, p, order = shape
    o = ls_ordinates(order)
    g, st, _, src = random_problem(nx, ny, p, o, seed=60 + nx + ny, materials=2)
    print("ref split storers", shape, storers, persistent, flush=True)
    for prec, tol in ((tsw.FP64, 1e-12), (tsw.FP32, 2e-6)):
        outs = []
        with _ctx(g, o, 1) as c:
            c.set_tuning("batch_split_rows", (192 if p == 1 else 96) if storers > 0 else (256 if p == 1 else 128))
            c.set_tuning("batch_split_storers", storers)
            c.set_tuning("batch_persistent", persistent)
            for _ in range(2):
                a = src.copy()
                c.sweep(a, st, 0.7, precision=prec)
                outs.append(a)
            assert (c.get_tuning("lane_split"), c.get_tuning("lane_coefficient")) == (1, 0)
        with _ctx(g, o, -1) as c:
            b = src.copy()
            c.sweep(b, st, 0.7, precision=prec)
        assert rel_err(b, orc_sweep(g, o, st, src, 0.7)) <= tol, prec
        np.testing.assert_array_equal(outs[0], b)
        np.testing.assert_array_equal(outs[1], b)


# the lane-per-coefficient kernel: rows of a wave (4; 16 at degree 1), of a workgroup (56, 224) and of a band (24, 64),
# columns below, at and past the 16 that its feeder holds, against the lane-split kernel (batch_split_rows set)
WIDE_EDGES = [(1, 1, 2, 2), (2, 3, 2, 4), (15, 4, 2, 2), (16, 5, 2, 6), (17, 56, 2, 4), (33, 57, 2, 4), (40, 121, 2, 8),
              (1, 57, 3, 2), (16, 56, 3, 4), (18, 73, 3, 6), (35, 200, 3, 4), (17, 15, 1, 2), (16, 17, 1, 4),
              (9, 224, 1, 2), (30, 225, 1, 6), (3, 300, 1, 12)]


@pytest.mark.parametrize("shape", WIDE_EDGES)
def test_ref_wide_edges_match_the_lane_split_kernel(shape):
    nx, ny, p, order = shape
    o = ls_ordinates(order)
    g, st, _, src = random_problem(nx, ny, p, o, seed=400 + nx + ny, materials=3)
    print("ref wide edges", shape, flush=True)
    for prec, tol in ((tsw.FP64, 1e-12), (tsw.FP32, 2e-6)):
        outs = []
        for rows in (0, 0, 32):
            with _ctx(g, o, 1) as c:
                if rows:
                    c.set_tuning("batch_split_rows", rows)
                a = src.copy()
                for _ in range(2):  # a sweep leaves the exchange records empty for the next
                    a[1:-1, 1:-1] = src[1:-1, 1:-1]
                    c.sweep(a, st, 0.4, precision=prec)
                outs.append(a)
        assert rel_err(outs[0], orc_sweep(g, o, st, src, 0.4)) <= tol, prec
        np.testing.assert_array_equal(outs[0], outs[2])
        np.testing.assert_array_equal(outs[0], outs[1])


@pytest.mark.parametrize("prec", [tsw.FP64, tsw.FP32])
def test_ref_sweeps_of_few_and_many_rows_alternate(prec):
    """Single sweeps (a lane per coefficient) between calls with many sources (lane-split, taking items from counters)."""
    import torch
    o = ls_ordinates(8)
    g, st, _, src = random_problem(6, 90, 2, o, seed=12, materials=2)
    dev = torch.device("cuda:0")
    with _ctx(g, o) as c:
        st_d = torch.from_numpy(st).to(dev)
        one = torch.from_numpy(src).to(dev)
        c.sweep(one, st_d, math.inf, precision=prec)
        for singles in (0, 1, 2, 3):
            for _ in range(singles):
                a = torch.from_numpy(src).to(dev)
                c.sweep(a, st_d, math.inf, precision=prec)
                assert torch.equal(a, one)
            many = [torch.from_numpy(src).to(dev) for _ in range(7)]  # 25,200 rows
            c.sweep_multi(many, st_d, math.inf, precision=prec)
            for k, a in enumerate(many):
                assert torch.equal(a, one), (singles, k)


@pytest.mark.parametrize("p,rows", [(1, 48), (2, 32), (3, 32)])
def test_ref_split_persistent_switched_on_and_off(p, rows):
    """A launch with one workgroup per item leaves the item counters alone: whichever launch follows takes every item."""
    o = ls_ordinates(6)
    g, st, _, src = random_problem(10, 100, p, o, seed=50 + p, materials=3)
    print("ref split persistent on and off", p, flush=True)
    with _ctx(g, o) as c:
        c.set_tuning("batch_split_rows", rows)  # the lane-split kernel
        first = None
        for persistent in (1, 0, 1, 0, 0, 1, 1, 0, 1):
            c.set_tuning("batch_persistent", persistent)
            a = src.copy()
            c.sweep(a, st, 0.7)
            if first is None:
                first = a
                assert rel_err(a, orc_sweep(g, o, st, src, 0.7)) <= 1e-12
            np.testing.assert_array_equal(a, first)


# sources of one launch by their rows (of all ordinates): which kernel takes them in FP64 and in FP32 (1: a lane per
# coefficient).  Past 100 columns it gives way at 20,000 rows at degrees 1 and 2 and, with few materials, between 30,000
# and 60,000 at degree 3, where 13 sources of 112 rows in one band go without storers; the line is another on few columns
@pytest.mark.parametrize("prec", [tsw.FP64, tsw.FP32])
@pytest.mark.parametrize("shape,kernel", [((101, 60, 1, 8, 9), (0, 0)), ((101, 60, 2, 8, 9), (0, 0)), ((101, 60, 2, 8, 8), (1, 1)),
                                          ((101, 112, 3, 8, 7), (1, 1)), ((101, 112, 3, 8, 13), (0, 0)),
                                          ((30, 100, 1, 8, 21), (0, 0)), ((20, 32, 2, 8, 33), (1, 0)),
                                          ((50, 40, 2, 8, 13), (1, 0)), ((40, 60, 3, 8, 13), (1, 0)),
                                          ((40, 200, 2, 8, 3), (1, 1)), ((40, 201, 2, 8, 3), (1, 0)),
                                          ((12, 100, 3, 8, 14), (1, 1)), ((50, 60, 2, 8, 20), (1, 0))])
def test_ref_sweeps_of_many_sources_equal_single_sweeps(shape, kernel, prec):
    import torch
    nx, ny, p, order, n = shape
    o = ls_ordinates(order)
    g, st, _, src = random_problem(nx, ny, p, o, seed=20 + nx + ny + p, materials=2)
    print("ref many sources", shape, prec, flush=True)
    dev = torch.device("cuda:0")
    with _ctx(g, o) as c:
        st_d = torch.from_numpy(st).to(dev)
        one = [torch.from_numpy(src * (1 + k)).to(dev) for k in range(2)]
        many = [one[k % 2].clone() for k in range(n)]
        for a in one:
            c.sweep(a, st_d, 0.5, precision=prec)
        assert c.get_tuning("lane_coefficient") == 1
        c.sweep_multi(many, st_d, 0.5, precision=prec)
        assert c.get_tuning("lane_split") == 1
        assert c.get_tuning("lane_coefficient") == kernel[0 if prec == tsw.FP64 else 1]
        for k, a in enumerate(many):
            assert torch.equal(a, one[k % 2]), k
    assert rel_err(one[0].cpu().numpy(), orc_sweep(g, o, st, src, 0.5)) <= (1e-12 if prec == tsw.FP64 else 2e-6)


def test_ref_split_more_sources_than_one_launch_takes():
    import torch
    o = ls_ordinates(4)
    g, st, _, src = random_problem(6, 70, 2, o, seed=3, materials=2)
    dev = torch.device("cuda:0")
    with _ctx(g, o) as c:
        st_d = torch.from_numpy(st).to(dev)
        many = [torch.from_numpy(src * (1 + k % 3)).to(dev) for k in range(33)]
        one = [torch.from_numpy(src * (1 + k)).to(dev) for k in range(3)]
        for a in one:
            c.sweep(a, st_d, math.inf)
        c.sweep_multi(many, st_d, math.inf)
        torch.cuda.synchronize()
        for k, a in enumerate(many):
            assert torch.equal(a, one[k % 3]), k


@pytest.mark.parametrize("p", [1, 2, 3])
def test_ref_split_follows_changes_of_the_inputs(p):
    """The sweep queued behind the check of the cross sections leaves the array alone when they have changed (also
    in one halo-side value, to more than 64 values and back), and each sweep is counted once."""
    o = ls_ordinates(4)
    g, st, _, src = random_problem(9, 35, p, o, seed=70 + p, materials=3)
    one = st.copy()
    one[g.nx, g.ny] *= 1.5
    many = random_problem(9, 35, p, o, seed=71 + p)[1]
    with _ctx(g, o) as c:
        c.sweep_timing(reset=True)
        seq = [(st, 0.3), (st, 0.3), (one, 0.3), (one, math.inf), (st, 0.3), (many, 0.3), (st, 0.3), (2 * st, 0.3)]
        for k, (sig, dt) in enumerate(seq):
            for prec, tol in ((tsw.FP64, 1e-12), (tsw.FP32, 2e-6)):
                out = src.copy()
                c.sweep(out, sig, dt, precision=prec)
                assert rel_err(out, orc_sweep(g, o, sig, src, dt)) <= tol, (k, prec)
                assert c.sweep_timing(reset=True)[0] == 1 or sig is many, (k, prec)


@pytest.mark.parametrize("rows", [0, 32])
def test_ref_split_and_diagonal_path_follow_the_same_changes(rows):
    """Sweeps on either layout by turns on one context, with other cross sections each time: the kernels read the material
    index in different layouts (rows 0: the cells', 32: the diagonals' in both)."""
    o = ls_ordinates(4)
    g, st, _, src = random_problem(12, 40, 2, o, seed=77, materials=3)
    sigs = [st, st[::-1, ::-1].copy(), 1.5 * st, np.where(st > st.mean(), 0.7, st)]
    with _ctx(g, o) as c:
        c.set_tuning("batch_split_rows", rows)
        for k in range(12):
            c.set_tuning("ref_split", (1, 1, -1)[k % 3])
            out = src.copy()
            c.sweep(out, sigs[k % 4], 0.3)
            assert rel_err(out, orc_sweep(g, o, sigs[k % 4], src, 0.3)) <= 1e-12, k


def test_ref_split_tuning_key():
    o = ls_ordinates(4)
    g, st, _, src = random_problem(5, 5, 1, o, seed=1)
    with _ctx(g, o) as c:
        for bad in (-2, 2):
            with pytest.raises(tsw.TswError):
                c.set_tuning("batch_split_storers", bad)
        assert c.get_tuning("ref_split") == 1
        for bad in (0, 2):
            with pytest.raises(tsw.TswError):
                c.set_tuning("ref_split", bad)
