"""GPU parity of pipelined stripe jobs: a 64-lane stripe job whose stripes P
wavefronts share, handing the boundary column over through device memory.

A round with fewer work items than the forward launch's wavefront slots pipes
its stripe jobs, P a job by its size (MH_DP_PIPE sets one P for the first
jobs; 0 or 1 keeps one wavefront a job).
Bar: bit-exact paths and scores against the oracle (full DP: NWSmall; banded:
the region DP at the stripe width used), and identical output for every P.
"""
import os

import numpy as np
import pytest

import mauvehip
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


@pytest.fixture
def dp_env():
    keys = ("MH_DP_PIPE", "MH_DP_COLS", "MH_DP_BAND_KIND")
    old = {k: os.environ.get(k) for k in keys}
    yield
    for k, v in old.items():
        if v is None:
            os.environ.pop(k, None)
        else:
            os.environ[k] = v


def _related(rng, la, lb, div=0.1):
    a = rng.integers(0, 4, la, dtype=np.uint8)
    b = a.copy() if lb <= la else np.concatenate([a, rng.integers(0, 4, lb - la, dtype=np.uint8)])
    b = b[:lb].copy()
    hit = rng.random(lb) < div
    b[hit] = rng.integers(0, 4, int(hit.sum()), dtype=np.uint8)
    return a, b


def _batch(pairs):
    A = np.concatenate([p[0] for p in pairs])
    B = np.concatenate([p[1] for p in pairs])
    la = np.array([len(p[0]) for p in pairs], dtype=np.int64)
    lb = np.array([len(p[1]) for p in pairs], dtype=np.int64)
    ao = np.concatenate([[0], np.cumsum(la)[:-1]])
    bo = np.concatenate([[0], np.cumsum(lb)[:-1]])
    return A, B, mauvehip.make_jobs(ao, la, bo, lb)


# shapes: one row, a row per chunk edge, many stripes at every width
SHAPES = [(1, 3000), (2, 1100), (63, 700), (64, 2000), (65, 1300), (500, 2600), (1500, 3100),
          (3000, 900), (700, 5000), (129, 257)]


def _pipe_parts(ctx):
    ms, n = ctx.kernel_time("dp_pipe_jobs")
    return int(round(ms * n))


@pytest.mark.parametrize("cols", ["4", "8", "16"])
def test_pipelined_full_dp_matches_oracle(ctx, dp_env, cols):
    rng = np.random.default_rng(700 + int(cols))
    pairs = [_related(rng, la, lb) for la, lb in SHAPES]
    A, B, jobs = _batch(pairs)
    os.environ["MH_DP_COLS"] = cols
    want = [po.nwsmall(a, b) for a, b in pairs]
    outs = {}
    for P in ("1", "2", "3", "5", "auto"):
        if P == "auto":
            os.environ.pop("MH_DP_PIPE", None)
        else:
            os.environ["MH_DP_PIPE"] = P
        ctx.set_timing(True)
        ctx.reset_kernel_times()
        paths, res = mauvehip.global_align(ctx, A, B, jobs)
        npiped = _pipe_parts(ctx)
        ctx.set_timing(False)
        if P == "1":
            assert npiped == 0
        elif P == "auto":
            # ten items, far fewer than the slots: the large jobs get up to eight parts
            assert npiped > 0
        else:
            # every job with at least P stripes of 64*cols columns runs pipelined
            sw = 64 * int(cols)
            assert npiped == sum((lb + sw - 1) // sw >= int(P) for _, lb in SHAPES), P
        got = [(mauvehip.path_of(paths, res, k), int(res[k]["score"])) for k in range(len(pairs))]
        for k, (p, sc) in enumerate(got):
            assert p == want[k][0] and sc == int(want[k][1]), (P, k, SHAPES[k])
        outs[P] = got
    assert all(v == outs["1"] for v in outs.values())


@pytest.mark.parametrize("cols", ["4", "16"])
def test_pipelined_banded_matches_region_oracle(ctx, dp_env, cols):
    rng = np.random.default_rng(710 + int(cols))
    shapes = SHAPES + [(4000, 3000), (2500, 4100)]
    pairs = [_related(rng, la, lb, 0.05) for la, lb in shapes]
    A, B, jobs = _batch(pairs)
    bands = rng.choice([3, 17, 64, 300], size=len(pairs)).astype(np.uint32)
    os.environ["MH_DP_COLS"] = cols
    os.environ["MH_DP_BAND_KIND"] = "stripes"
    ref = None
    for P in ("1", "2", "4", "auto"):
        if P == "auto":
            os.environ.pop("MH_DP_PIPE", None)
        else:
            os.environ["MH_DP_PIPE"] = P
        paths, res, dev, st = mauvehip.global_align_banded(ctx, A, B, jobs, bands, flags=mauvehip.BAND_NO_FALLBACK)
        got = [(mauvehip.path_of(paths, res, k), int(res[k]["score"]), int(dev[k]), int(res[k]["path_len"]))
               for k in range(len(pairs))]
        if ref is None:
            ref = got
            for k, (a, b) in enumerate(pairs):
                eff, kind, width = mauvehip.band_region(len(a), len(b), 2 * int(bands[k]))
                p, sc, dv = po.nwsmall_region(a, b, eff, width if kind == mauvehip.REGION_STRIPES else 0)
                if p is None:
                    assert got[k][3] == 0
                    continue
                assert got[k][0] == p and got[k][1] == sc and got[k][2] == dv, (k, shapes[k], int(bands[k]))
        assert got == ref, P


def test_narrow_banded_stripes_over_all_lanes(ctx, dp_env):
    """Jobs of 16-lane stripes that the round spreads take all 64 lanes, one or
    two columns a lane, over the same stripes: columns at a stripe's edges, one
    row, rows at the chunks' edges, operands far from square."""
    rng = np.random.default_rng(730)
    shapes = [(1, 300), (15, 129), (16, 128), (17, 65), (400, 63), (900, 64), (1023, 1025), (700, 641), (1600, 1500),
              (2100, 1000), (1000, 2300)]
    pairs = [_related(rng, la, lb, 0.05) for la, lb in shapes for _ in range(3)]
    bands = np.array([2, 9, 40] * len(shapes), dtype=np.uint32)
    A, B, jobs = _batch(pairs)
    os.environ.pop("MH_DP_COLS", None)
    os.environ["MH_DP_BAND_KIND"] = "stripes"
    got = {}
    for P in ("1", "auto"):
        if P == "auto":
            os.environ.pop("MH_DP_PIPE", None)
        else:
            os.environ["MH_DP_PIPE"] = P
        ctx.set_timing(True)
        ctx.reset_kernel_times()
        paths, res, dev, st = mauvehip.global_align_banded(ctx, A, B, jobs, bands, flags=mauvehip.BAND_NO_FALLBACK)
        assert (_pipe_parts(ctx) > 0) == (P == "auto")
        ctx.set_timing(False)
        got[P] = [(mauvehip.path_of(paths, res, k), int(res[k]["score"]), int(dev[k]), int(res[k]["path_len"]))
                  for k in range(len(pairs))]
    narrow = 0
    for k, (a, b) in enumerate(pairs):
        eff, kind, width = mauvehip.band_region(len(a), len(b), 2 * int(bands[k]))
        narrow += kind == mauvehip.REGION_STRIPES and width <= 128 and len(b) > width
        p, sc, dv = po.nwsmall_region(a, b, eff, width if kind == mauvehip.REGION_STRIPES else 0)
        if p is None:
            assert got["auto"][k][3] == 0
        else:
            assert got["auto"][k][:3] == (p, sc, dv), (k, len(a), len(b), int(bands[k]))
    assert narrow > 10
    assert got["1"] == got["auto"]


@pytest.mark.parametrize("n,length,band,spread", [(8, 3000, 50, True), (4000, 300, 32, False), (60, 1000, 4, False)])
def test_narrow_banded_jobs_spread_where_it_gains(ctx, dp_env, n, length, band, spread):
    """Jobs of 16-lane stripes are spread over all lanes where SIMDs would be
    idle, and left four a wavefront where the round has enough of them or their
    bands are so narrow that a stripe waits for the one before it; either way
    the paths, scores and deviations of one wavefront a job."""
    rng = np.random.default_rng(n)
    pairs = [_related(rng, length, length, 0.05) for _ in range(n)]
    A, B, jobs = _batch(pairs)
    bands = np.full(n, band, dtype=np.uint32)
    os.environ.pop("MH_DP_COLS", None)
    os.environ["MH_DP_BAND_KIND"] = "stripes"
    got = {}
    for P in ("1", "auto"):
        if P == "auto":
            os.environ.pop("MH_DP_PIPE", None)
        else:
            os.environ["MH_DP_PIPE"] = P
        ctx.set_timing(True)
        ctx.reset_kernel_times()
        paths, res, dev, st = mauvehip.global_align_banded(ctx, A, B, jobs, bands, flags=mauvehip.BAND_NO_FALLBACK)
        assert _pipe_parts(ctx) == (n if spread and P == "auto" else 0)
        ctx.set_timing(False)
        got[P] = [(mauvehip.path_of(paths, res, k), int(res[k]["score"]), int(dev[k])) for k in range(n)]
    assert got["1"] == got["auto"]


@pytest.mark.parametrize("budget_gb", ["0.002", "0.004", "0.02"])
def test_rounds_of_spread_banded_jobs_stay_within_the_budget(ctx, dp_env, monkeypatch, budget_gb):
    """A job spread over wavefronts takes more memory (a boundary four times as
    large, a byte a column where a lane has one): a round's trace and boundary
    columns stay within the budget with it, and paths, scores and deviations
    are those of one wavefront a job."""
    rng = np.random.default_rng(740)
    shapes = [(2100, 1000), (1600, 1500), (1000, 2300), (900, 640)] * 15
    pairs = [_related(rng, la, lb, 0.05) for la, lb in shapes]
    bands = rng.choice([2, 9, 40], size=len(pairs)).astype(np.uint32)
    A, B, jobs = _batch(pairs)
    os.environ.pop("MH_DP_COLS", None)
    os.environ["MH_DP_BAND_KIND"] = "stripes"

    def run():
        ctx.set_timing(True)
        ctx.reset_kernel_times()
        paths, res, dev, st = mauvehip.global_align_banded(ctx, A, B, jobs, bands, flags=mauvehip.BAND_NO_FALLBACK)
        arena, piped = ctx.kernel_time("dp_arena_bytes")[0], _pipe_parts(ctx)
        ctx.set_timing(False)
        return [(mauvehip.path_of(paths, res, k), int(res[k]["score"]), int(dev[k]), int(res[k]["path_len"]))
                for k in range(len(pairs))], arena, piped

    os.environ["MH_DP_PIPE"] = "1"
    want, one, piped = run()
    assert piped == 0
    os.environ.pop("MH_DP_PIPE")
    free, most, piped = run()
    assert piped > 0 and most > one and free == want
    monkeypatch.setenv("MH_DP_TB_BUDGET_GB", budget_gb)
    got, arena, piped = run()
    budget = float(budget_gb) * (1 << 30)
    assert 0 < arena <= budget
    if budget > most:
        assert arena == most
    assert got == want


def test_pipelined_prefix_with_many_small_jobs(ctx, dp_env):
    """A round whose work items nearly fill the slots pipes only a prefix of
    its stripe jobs; the output equals the unpipelined one."""
    rng = np.random.default_rng(720)
    pairs = [_related(rng, la, lb) for la, lb in [(2000, 3000)] * 6]
    pairs += [_related(rng, int(x), int(x)) for x in rng.integers(300, 600, 2900)]
    A, B, jobs = _batch(pairs)
    os.environ["MH_DP_COLS"] = "4"
    res_by = {}
    for P in ("1", "2"):
        os.environ["MH_DP_PIPE"] = P
        ctx.set_timing(True)
        ctx.reset_kernel_times()
        paths, res = mauvehip.global_align(ctx, A, B, jobs)
        npiped = _pipe_parts(ctx)
        ctx.set_timing(False)
        res_by[P] = (paths.copy(), res.copy(), npiped)
    assert res_by["1"][2] == 0 and res_by["2"][2] > 0
    assert np.array_equal(res_by["1"][1], res_by["2"][1])
    assert np.array_equal(res_by["1"][0], res_by["2"][0])
    for k in range(6):
        p, sc = po.nwsmall(*pairs[k])
        assert mauvehip.path_of(*res_by["2"][:2], k) == p and int(res_by["2"][1][k]["score"]) == int(sc)
