"""Swaptions (bs_swaptions_host_f64) on the MI355X, through the C ABI, against
the oracle's restatement of HJM_Swaption_Blocking
(parsec-ff/pkgs/apps/swaptions/src/HJM_Swaption_Blocking.cpp:20-222).

The kernel follows the reference's arithmetic step for step (same draws,
same order of every FP64 product and sum); what differs is the device's
exp/log (last-bit differences) and the order of the final sums over paths.
The bar: every price within 1e-12 relative (+1e-13 absolute) of the oracle's
and every standard error within 1e-8 relative, whose formula subtracts two
nearly equal sums (below a noise floor of 8 |price| sqrt(1e-15), where the
payoffs do not vary, both standard errors are rounding noise).  Shapes cover the driver's portfolio, every factor count
1..8, swaptions starting at t = 0 and past the kernel's register form (the
generic form), swap curves past the horizon, compounded strikes, trial
counts that are not multiples of the block size, and the full 128-swaption
1,000,000-trial workload (two swaptions checked against the oracle).
"""
import ctypes
import math
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "oracle"))

import pyswaptions as S  # noqa: E402
from p3arsec_amd import swaptions as W  # noqa: E402

pytestmark = pytest.mark.gpu

YLD = W.parsec_portfolio(1)[0][0]["yield"]


def sw(**kw):
    d = {"strike": 0.1, "compounding": 0.0, "maturity": 1.0, "tenor": 2.0, "interval": 1.0,
         "years": 5.5, "yield": YLD, "factors": W.PARSEC_FACTORS}
    n = kw.pop("n", None)
    F = kw.pop("F", None)
    if n is not None:
        rng = np.random.default_rng(n * 10 + F)
        d["yield"] = 0.05 + 0.004 * np.arange(n)
        d["factors"] = rng.uniform(0.0, 0.01, (F, n - 1))
    d.update(kw)
    return d


def check(got, want, tag):
    (gp, ge), (op, oe) = got, want
    if math.isnan(op) or math.isinf(op):
        assert gp == op or (math.isnan(gp) and math.isnan(op)), (tag, gp, op)
        return 0.0
    assert abs(gp - op) <= 1e-12 * abs(op) + 1e-13, (tag, gp, op)
    # When the payoffs barely vary (a swaption starting at t = 0 pays the same
    # on every path), sumsq - sum^2/n is rounding noise in both, its sign and
    # size set by the order of the sums: at or below this floor (or NaN, the
    # root of a negative noise) the two standard errors are both noise.
    floor = 8 * abs(op) * math.sqrt(1e-15)
    if math.isnan(oe) or oe <= floor:
        assert math.isnan(ge) or ge <= floor, (tag, ge, oe, floor)
    else:
        assert abs(ge - oe) <= 1e-8 * abs(oe) + 1e-15, (tag, ge, oe)
    return abs(gp - op) / max(abs(op), 1e-300)


def test_parsec_portfolio_matches_oracle(gpu):
    sws, base = W.parsec_portfolio(16)
    p, e = W.price(sws, 20000, base)
    worst = 0.0
    for i, s in enumerate(sws):
        worst = max(worst, check((p[i], e[i]), S.price_blocking(s, base + i, 20000), i))
    print(f"16 swaptions x 20000 trials: max relative price difference {worst:.2e}")
    assert np.all(np.isfinite(p)) and np.all(p >= 0)


SHAPES = [   # strikes near the money: 20-40% of paths pay
    dict(strike=0.13),
    dict(years=19.75, strike=0.18),
    dict(years=5.0, strike=0.12, compounding=0.5),
    dict(years=8.0, maturity=2.0, tenor=3.0, interval=0.5, strike=0.19),
    dict(years=10.0, maturity=0.0, tenor=4.0, strike=0.15),               # starts at t = 0
    dict(years=3.0, maturity=2.1, tenor=0.5, interval=0.25, strike=0.19),  # curve past horizon
    dict(years=6.0, factors=W.PARSEC_FACTORS[:1], strike=0.14),            # 1 factor
    dict(n=20, F=5, years=12.0, maturity=4.0, tenor=5.0, strike=0.14),
    dict(n=30, F=2, years=15.0, maturity=3.0, tenor=4.0, strike=0.12),     # start 6: generic
    dict(n=12, F=8, years=6.0, maturity=1.5, tenor=2.0, strike=0.08),      # 8 factors
    dict(n=20, F=8, years=10.0, maturity=4.0, tenor=2.0, strike=0.11),     # 8 x 8 draws
    dict(n=64, F=1, years=16.0, maturity=10.0, tenor=5.0, strike=0.41),    # 64 steps, 40 draws
    dict(n=2, F=3, years=2.0, maturity=0.0, tenor=1.0, strike=0.3,
         factors=W.PARSEC_FACTORS[:, :1]),                                 # smallest curve
    # strongly negative rates: the discount factors past the last cash flow
    # grow, so every path takes the kernel's full computation
    dict(years=11.0, tenor=2.0, strike=-0.3, **{"yield": np.full(11, -0.4)}),
]


@pytest.mark.parametrize("i", range(len(SHAPES)))
def test_shapes_match_oracle(gpu, i):
    s = sw(**SHAPES[i])
    for trials, block in ((1001, 16), (77, 1), (500, 7), (4096, 16)):
        got = W.price([s], trials, 4321 + i, block)
        check((got[0][0], got[1][0]), S.price_blocking(s, 4321 + i, trials, block),
              (i, trials, block))


def test_many_swaptions_mixed_starts(gpu):
    # one launch for swaptions of different horizons, starts and curve lengths
    sws = [sw(years=y, strike=k, maturity=m) for y, k, m in
           ((5.0, 0.11, 1.0), (9.0, 0.13, 2.5), (14.0, 0.2, 3.0), (6.0, 0.1, 0.0),
            (7.5, 0.12, 1.4))] * 7
    p, e = W.price(sws, 3000, 777)
    for i, s in enumerate(sws):
        check((p[i], e[i]), S.price_blocking(s, 777 + i, 3000), i)


def test_bit_reproducible_and_stream(gpu):
    sws, base = W.parsec_portfolio(8)
    a = W.price(sws, 50000, base)
    b = W.price(sws, 50000, base)
    st = gpu.Stream()
    c = W.price(sws, 50000, base, stream=st.handle)
    st.destroy()
    for x, y in ((a, b), (a, c)):
        assert np.array_equal(x[0], y[0]) and np.array_equal(x[1], y[1])


def test_one_trial_and_single_path_blocks(gpu):
    s = sw(years=5.5, strike=0.3)
    for trials, block in ((1, 1), (1, 16), (2, 1)):
        got = W.price([s], trials, 99, block)
        check((got[0][0], got[1][0]), S.price_blocking(s, 99, trials, block), (trials, block))


def test_zero_draw_gives_the_reference_nan_and_inf(gpu):
    """Counter 2^31 - 1 draws u = 0, whose inverse normal is -inf: that path's
    rates become infinite or NaN (0 x inf where a factor is 0).  The map
    follows the reference through it: same price, NaN or inf included."""
    sws, _ = W.parsec_portfolio(4)
    m31 = 2147483647
    for i, s in enumerate(sws):
        for back in (1, 5, 29, 31, 95):
            seed = m31 - back
            got = W.price([s], 64, seed)
            check((got[0][0], got[1][0]), S.price_blocking(s, seed, 64), (i, back))


def test_native_workload(gpu):
    """PARSEC's native run: 128 swaptions x 1,000,000 trials."""
    sws, base = W.parsec_portfolio(128)
    p, e = W.price(sws, 1_000_000, base)
    assert np.all(np.isfinite(p)) and np.all(p >= 0)
    assert np.all(e[p > 0] > 0)
    for i in (0, 127):
        check((p[i], e[i]), S.price_chain(sws[i], base + i, 1_000_000), i)
    print(f"128 x 1M: prices {p.min():.4f} .. {p.max():.4f}")


def test_counters_near_the_limit(gpu):
    """Seeds whose last counters come within a few thousand of 2^42, where
    1513517 c approaches 2^63: the kernel's Mersenne reduction against the
    oracle's literal 64-bit remainders."""
    s = sw(years=5.5, strike=0.13)
    trials = 1000                      # 1008 paths x 30 counters each
    for slack in (5, 1000, 123457):
        seed = 2 ** 42 - 1008 * 30 - slack
        got = W.price([s], trials, seed)
        check((got[0][0], got[1][0]), S.price_blocking(s, seed, trials), slack)
    # one past the limit is refused
    from p3arsec_amd import capi
    with pytest.raises(capi.BSError):
        W.price([s], trials, 2 ** 42 - 1008 * 30 + 1)


@pytest.mark.parametrize("n,F,start,points,every", [
    # draws (start x F) and cash flows (points / every) at the edges of the
    # register form (3, 6 draws; 1-4 flows) and of the wide form's batches of
    # 12 draws and its widths up to 64 flows
    (11, 1, 1, 1, 1), (11, 2, 1, 2, 1), (11, 1, 3, 3, 1), (11, 4, 1, 4, 1), (11, 5, 1, 2, 2),
    (11, 3, 2, 4, 2), (11, 7, 1, 3, 1), (20, 4, 3, 5, 1), (20, 6, 2, 6, 1), (20, 1, 13, 6, 1),
    (30, 8, 3, 7, 1), (30, 5, 5, 8, 1), (40, 7, 7, 9, 1), (40, 2, 12, 12, 1), (40, 8, 8, 13, 1),
    (40, 3, 1, 16, 1), (40, 1, 4, 17, 1), (64, 2, 6, 24, 1), (64, 2, 32, 25, 1), (64, 3, 8, 32, 1),
    (64, 1, 2, 33, 1), (64, 1, 7, 48, 1), (64, 1, 13, 49, 1), (64, 1, 1, 62, 1), (64, 4, 1, 62, 3),
])
def test_draw_and_cash_flow_edges(gpu, n, F, start, points, every):
    """The bar is the file's: about 64 roundings of exponents below 4 in size
    move a payoff by at most 64 x 4 x 2^-53 = 3e-14 relative to the bonds."""
    years = 0.25 * n
    s = sw(n=n, F=F, years=years, maturity=start * 0.25, tenor=points * 0.25,
           interval=every * 0.25, strike=0.13)
    for trials in (1, 255, 5000):
        got = W.price([s], trials, 97 * n + F, 1)
        check((got[0][0], got[1][0]), S.price_blocking(s, 97 * n + F, trials, 1), (n, F, trials))


@pytest.mark.parametrize("count,trials", [(128, 131_073), (128, 524_289)])
def test_more_paths_per_work_item(gpu, count, trials):
    sws, base = W.parsec_portfolio(count)
    p, e = W.price(sws, trials, base)
    for i in (0, count - 1):
        check((p[i], e[i]), S.price_chain(sws[i], base + i, trials), i)


def test_blocks_with_a_zero_draw(gpu):
    """One block of five holds the counter that draws u = 0, in a draw the
    payoff does not read (finite prices) or reads (the reference's NaN or inf);
    its paths take the step-by-step kernel, the others the linear one."""
    m31 = 2147483647
    for s in W.parsec_portfolio(3)[0]:
        for offset in (25, 1):
            seed = m31 - 30 * 2500 - offset
            got = W.price([s], 5000, seed)
            check((got[0][0], got[1][0]), S.price_blocking(s, seed, 5000), offset)


def test_rates_past_the_linear_bound(gpu):
    """A horizon of 2000 years: exponents past the bound that keeps the
    reference's products from underflow, next to an ordinary swaption."""
    wide = sw(years=2000.0, maturity=182.0, tenor=364.0, interval=182.0, strike=0.02)
    p, e = W.price([wide, sw(strike=0.13)], 3000, 31)
    for i, s in enumerate((wide, sw(strike=0.13))):
        check((p[i], e[i]), S.price_blocking(s, 31 + i, 3000), i)


def same_bits(a, b):
    # a trial count that is no multiple of the block makes some of the
    # reference's standard errors the root of a negative number
    return np.array_equal(a.view(np.uint64), b.view(np.uint64))


def test_calls_from_more_threads_than_workspaces(gpu):
    import threading
    sets = [W.parsec_portfolio(8 + k, 1979 + k) for k in range(8)]
    want = [W.price(s, 3000, base) for s, base in sets]
    bad = []

    def work(k):
        st = gpu.Stream()
        for _ in range(20):
            p, e = W.price(sets[k][0], 3000, sets[k][1], stream=st.handle)
            if not (same_bits(p, want[k][0]) and same_bits(e, want[k][1])):
                bad.append(k)
        st.destroy()

    ts = [threading.Thread(target=work, args=(k,)) for k in range(8)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad


def test_parameters_past_a_workspace(gpu):
    """6000 swaptions have more parameters than a workspace's 1 MB: the same
    bits as the call in pieces that fit."""
    sws, base = W.parsec_portfolio(6000)
    p, e = W.price(sws, 64, base)
    for lo in range(0, 6000, 500):
        q, f = W.price(sws[lo:lo + 500], 64, base + lo)
        assert same_bits(p[lo:lo + 500], q) and same_bits(e[lo:lo + 500], f), lo


@pytest.mark.parametrize("count,trials", [(1, 1), (511, 600), (512, 600), (513, 600),
                                          (64, 131_072), (64, 131_200), (65, 131_072)])
def test_both_ends_of_a_launch_give_the_same_bits(gpu, count, trials):
    """A launch whose last blocks form the results (up to 512 swaptions and 8192
    blocks) against the same swaptions one by one and in halves."""
    sws, base = W.parsec_portfolio(count)
    p, e = W.price(sws, trials, base, 1)
    q, f = W.price(sws[:1], trials, base, 1)
    check((p[0], e[0]), (q[0], f[0]), "first")
    half = (count + 1) // 2
    if half < count:
        q, f = W.price(sws[half:], trials, base + half, 1)
        for i in (0, count - half - 1):
            check((p[half + i], e[half + i]), (q[i], f[i]), i)
    again = W.price(sws, trials, base, 1)
    assert same_bits(p, again[0]) and same_bits(e, again[1])


def desk(count):
    """Swaptions with 4 to 40 draws and 2 to 10 cash flows, starts at steps 1-10."""
    return [sw(n=24, F=4, years=6.0, maturity=0.25 * (1 + i % 10), tenor=2.5 - 0.5 * (i % 4),
               interval=0.25, strike=0.11 + 0.002 * i) for i in range(count)]


@pytest.mark.parametrize("sws,trials", [
    # work-items of 2 to 32 rows in the whole call (8 to 125,056 blocks of 1024
    # paths), fewer in its parts; units of 2 and 8 rows
    (lambda: W.parsec_portfolio(600)[0], 600), (lambda: W.parsec_portfolio(70)[0], 16_385),
    (lambda: W.parsec_portfolio(65)[0], 262_145), (lambda: W.parsec_portfolio(128)[0], 524_288),
    (lambda: W.parsec_portfolio(128)[0], 1_000_000), (lambda: desk(40), 30_001),
    (lambda: desk(20) + W.parsec_portfolio(20)[0], 1_000),
    (lambda: [dict(s, factors=s["factors"][:1]) for s in W.parsec_portfolio(9)[0]], 40_000),
])
@pytest.mark.parametrize("seed", [1979, 2147483647 - 30 * 700])
def test_a_swaptions_bits_do_not_depend_on_the_call(gpu, sws, trials, seed):
    """A swaption priced alone, in a shard and in the portfolio: the same bits,
    also where the second seed's zero draw leaves paths to the step-by-step
    kernel, and in launches that end by themselves as in those that don't."""
    sws = sws()
    if len({len(s["factors"]) for s in sws}) > 1:
        sws = [dict(s, factors=s["factors"][:3]) for s in sws]
    p, e = W.price(sws, trials, seed)
    parts = {(0, 1), (len(sws) - 1, len(sws)), (len(sws) // 2, len(sws) // 2 + 1),
             (0, len(sws) // 3), (len(sws) // 3, len(sws))}
    for lo, hi in sorted(parts):
        q, f = W.price(sws[lo:hi], trials, seed + lo)
        assert same_bits(p[lo:hi], q) and same_bits(e[lo:hi], f), (lo, hi)


@pytest.mark.parametrize("F", [1, 3, 4, 5, 8])
@pytest.mark.parametrize("start", [1, 2, 3, 4, 5, 8, 9, 12])
def test_step_by_step_forms(gpu, F, start):
    """At the edges of the step-by-step kernel's forms (starts at up to 2, 4 and 8
    steps, and beyond): path 700's last draw, which no payoff reads, is u = 0, so
    its unit of paths goes to that kernel; beside a swaption that is priced by it
    whole.  The bar is the file's."""
    if start * F > 64:
        pytest.skip("more than 64 draws")
    n = 26
    per_path = (n - 1) * F
    seed = 2147483647 - 700 * per_path - (per_path - 1)
    s = sw(n=n, F=F, years=0.25 * n, maturity=start * 0.25, tenor=1.0, interval=0.25, strike=0.13)
    whole = dict(s, years=400.0 * n, maturity=start * 400.0, tenor=1600.0, interval=400.0,
                 strike=0.01)
    p, e = W.price([s, whole], 3000, seed, 1)
    for i, x in enumerate((s, whole)):
        check((p[i], e[i]), S.price_blocking(x, seed + i, 3000, 1), i)
        q, f = W.price([x], 3000, seed + i, 1)
        assert same_bits(p[i:i + 1], q) and same_bits(e[i:i + 1], f)


@pytest.mark.parametrize("count,trials", [(128, 32_000), (128, 98_300), (128, 262_100)])
@pytest.mark.parametrize("seed", [1979, 2147483647 - 30 * 700, 2147483647 - 30 * 256 - 29])
def test_units_of_two_rows_in_pairs(gpu, count, trials, seed):
    """Work-items of 8, 16 and 32 rows, whose units of 2 are folded in pairs, the
    last pair cut by the end of the paths, against the swaption alone (4 rows or 2):
    the same bits, also where a zero draw takes the first or the second unit of a
    pair away."""
    sws = W.parsec_portfolio(count)[0]
    p, e = W.price(sws, trials, seed, 1)
    for i in (0, 1, 2, count // 2, count - 1):
        q, f = W.price(sws[i:i + 1], trials, seed + i, 1)
        assert same_bits(p[i:i + 1], q) and same_bits(e[i:i + 1], f), i
    check((p[1], e[1]), S.price_chain(sws[1], seed + 1, trials, 1), 1)
