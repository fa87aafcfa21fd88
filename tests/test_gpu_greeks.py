"""The fused adjoint kernel (price + delta, vega, rho, theta) on the MI355X.

Checked against
  * FP64 central finite differences of the A&S price (the quantity the
    adjoint differentiates) with bump 1e-5 relative, and with the 1e-3 bump
    the benchmark spec names, whose truncation error (h S)^2/6 * d3P/dS3
    reaches ~3e-4 on delta when sigma sqrt(T) is near its 0.0112 minimum;
  * the closed-form Greeks with the exact normal CDF (differs from the A&S
    derivatives by at most ~6e-5 of the scale, see test_oracle.py).
Errors are measured as |adjoint - check| / scale with per-Greek scales
  price: S+K, delta: 1, vega: S sqrt(T), rho: K T, theta: S+K,
and as plain relative error over options whose Greek is at least 1% of its
scale.  The price output must equal the price-only kernel bit for bit.
"""
import numpy as np
import pytest

from p3arsec_amd import books

pytestmark = pytest.mark.gpu
NAMES = ("price", "delta", "vega", "rho", "theta")
# scaled-error bounds vs FP64 FD (h=1e-5): float rounding of the adjoint
# sweep, whose d1 path is amplified by 1/(sigma sqrt T) (<= 1/0.0112 here)
BOUND_FD = (1e-6, 1e-4, 2e-5, 1e-4, 1e-5)
# vs FD with h=1e-3: add the FD truncation error
BOUND_FD3 = (1e-6, 6e-4, 5e-5, 1e-4, 2e-5)


def scales(book):
    s, k, t = (a.astype(np.float64) for a in (book.s, book.k, book.t))
    return [s + k, np.ones_like(s), s * np.sqrt(t), k * t, s + k]


def gpu_greeks(capi, book):
    db = capi.DeviceBook(book)
    outs = capi.greeks(db)
    res = np.stack([o.download(np.float32, book.n) for o in outs]).astype(np.float64)
    price = capi.price(db).download(np.float32, book.n)
    for o in outs:
        o.free()
    db.free()
    return res, price


def d12(book):
    s, k, r, v, t = (a.astype(np.float64) for a in book.arrays()[:5])
    den = v * np.sqrt(t)
    d1 = (np.log(s / k) + (r + 0.5 * v * v) * t) / den
    return d1, d1 - den


def report(tag, got, ref, sc, mask=None):
    line = []
    for j, name in enumerate(NAMES):
        scaled = np.abs(got[j] - ref[j]) / sc[j]
        big = np.abs(ref[j]) >= 0.01 * sc[j]
        if mask is not None:
            scaled, big = scaled[mask], big & mask
        rel = np.abs(got[j] - ref[j])[big] / np.abs(ref[j])[big]
        line.append(f"{name}: scaled max {scaled.max():.2e} mean {scaled.mean():.2e}, "
                    f"rel max {rel.max() if rel.size else 0:.2e}")
    print(f"\n{tag}\n  " + "\n  ".join(line))


def test_adjoint_against_fd_and_closed_form(gpu, oracle):
    book = books.make_book(200_000, books.SEED_BASE + 4)
    got, price = gpu_greeks(gpu, book)
    assert np.array_equal(got[0].astype(np.float32).view(np.uint32), price.view(np.uint32))
    sc = scales(book)
    fd3 = oracle.greeks_fd(book, 1e-3)
    fd5 = oracle.greeks_fd(book, 1e-5)
    ex = oracle.greeks_exact(book)
    # The A&S CNDF jumps by 1.05e-9 at 0 (CNDF(0+) = 0.5000000005,
    # CNDF(0-) = 0.4999999995); a 1e-5 bump that straddles it is not a
    # derivative, so that check skips options with |d1| or |d2| < 2e-3.
    d1, d2 = d12(book)
    smooth = (np.abs(d1) > 2e-3) & (np.abs(d2) > 2e-3)
    report("adjoint vs FP64 central FD (h=1e-3)", got, fd3, sc)
    report(f"adjoint vs FP64 central FD (h=1e-5, {int((~smooth).sum())} options near "
           f"the CNDF jump excluded)", got, fd5, sc, smooth)
    report("adjoint vs closed form", got, ex, sc)
    for j in range(5):
        assert np.max((np.abs(got[j] - fd5[j]) / sc[j])[smooth]) <= BOUND_FD[j], NAMES[j]
        assert np.max(np.abs(got[j] - fd3[j]) / sc[j]) <= BOUND_FD3[j], NAMES[j]
        assert np.max(np.abs(got[j] - ex[j]) / sc[j]) <= BOUND_FD[j] + 1e-4, NAMES[j]


def test_greeks_signs_and_identities(gpu):
    book = books.make_book(100_000, books.SEED_BASE + 26)
    got, _ = gpu_greeks(gpu, book)
    call = book.otype == 0
    delta, vega, rho = got[1], got[2], got[3]
    assert np.all(delta[call] > -1e-6) and np.all(delta[call] < 1 + 1e-6)
    assert np.all(delta[~call] < 1e-6) and np.all(delta[~call] > -1 - 1e-6)
    assert np.all(vega > -1e-3)
    assert np.all(rho[call] > -1e-3) and np.all(rho[~call] < 1e-3)


@pytest.mark.parametrize("n", [1, 3, 5, 1027])
def test_greeks_ragged_and_misaligned(gpu, n):
    book = books.make_book(n, books.SEED_BASE + 27)
    base, _ = gpu_greeks(gpu, book)
    db = gpu.DeviceBook(book, pad=1)           # scalar path
    outs = gpu.greeks(db)
    mis = np.stack([o.download(np.float32, n) for o in outs]).astype(np.float64)
    assert np.array_equal(base, mis)


@pytest.mark.parametrize("n", [(1 << 22) - 1, 1 << 22, (1 << 22) + 3])
def test_width_by_size_gives_the_same_bits(gpu, n):
    """Books from 2^22 options on take four options per work-item, smaller ones
    two: on both sides of the line, whole and from an odd option on, the
    outputs are those of either width, to the bit."""
    db = gpu.DeviceBook(books.make_book(n, books.SEED_BASE + 5))
    outs = [gpu.DeviceBuffer(4 * n) for _ in range(5)]
    old = gpu.get_config(gpu.CFG_VECTOR_WIDTH)
    try:
        for first in (0, 3):
            got = []
            for width in (0, 2, 4):
                gpu.set_config(gpu.CFG_VECTOR_WIDTH, width)
                for o in outs:
                    gpu.call("bs_memset", o.ptr, 0xff, 4 * n, None)
                p = db.ptrs()
                gpu.call("bs_price_greeks_f32", *[a + 4 * first for a in p[:5]], p[5] + first,
                         *[o.ptr + 4 * first for o in outs], n - first, None)
                got.append(np.stack([o.download(np.uint32, n) for o in outs]))
            assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2]), first
            assert np.all(got[0][:, :first] == 0xffffffff)
            assert np.all(np.isfinite(got[0][:, first:].view(np.float32)))
    finally:
        gpu.set_config(gpu.CFG_VECTOR_WIDTH, old)
        for o in outs:
            o.free()
        db.free()


def test_price_output_on_degenerate_inputs(gpu):
    """On the degenerate book (T = 0, sigma = 0, zero and infinite S and K,
    NaN), the fused kernel's price output equals bs_price_f32's bit for bit,
    NaNs in the same places: the forward pass is the same code."""
    book = books.degenerate_book()
    db = gpu.DeviceBook(book)
    want = gpu.price(db).download(np.float32, book.n)
    got = [o.download(np.float32, book.n) for o in gpu.greeks(db)]
    assert np.array_equal(got[0].view(np.uint32), want.view(np.uint32))
    # the Greeks are finite for the rows whose inputs are ordinary (the rest meet
    # overflow or 0 * inf in float, as any float adjoint would)
    def within(x, lo, hi):
        return (x >= lo) & (x <= hi)
    ordinary = within(book.s, 1e-3, 1e6) & within(book.k, 1e-3, 1e6) & within(book.v, 1e-3, 10) \
        & within(book.t, 1e-3, 100) & within(np.abs(book.r), 0, 1)
    assert ordinary.sum() >= 4
    for g in got[1:]:
        assert np.all(np.isfinite(g[ordinary]))
    db.free()


def test_greeks_of_tiny_volatilities(gpu):
    """sigma sqrt(T) from FP32's smallest normal numbers up to 1e-20.  At the
    money with r = 0, vega is S n(0) sqrt(T) and theta -S n(0) sigma / (2 sqrt(T));
    off the money the option is the forward or nothing: vega 0, theta
    -r K e^{-rT} of a call that will be exercised and + that of such a put.
    CNDF's derivative at 0 is 6e-6 off n(0) and a dozen roundings add 1e-6."""
    rows = [(100.0, 100.0, 0.0, v, t) for v in (2e-38, 1e-37, 1e-36, 1e-30, 1e-20)
            for t in (0.5, 1.0, 4.0)]
    rows += [(s, 190.0 - s, 0.05, v, 1.0) for s in (100.0, 90.0) for v in (2e-38, 1e-30, 1e-20)]
    a = np.array(rows)
    at_money = np.tile(a[:, 0] == a[:, 1], 2)
    book = books.Book(*[np.concatenate([a[:, j]] * 2).astype(np.float32) for j in range(5)],
                      np.repeat([0, 1], len(rows)).astype(np.uint8))
    got, _ = gpu_greeks(gpu, book)
    s, k, r, v, t = (x.astype(np.float64) for x in book.arrays()[:5])
    put = book.otype != 0
    n0 = s / np.sqrt(2 * np.pi)
    vega = np.where(at_money, n0 * np.sqrt(t), 0.0)
    exercised = np.where(s > k, ~put, put)
    theta = np.where(at_money, -n0 * v / (2 * np.sqrt(t)),
                     np.where(exercised, np.where(put, 1.0, -1.0) * r * k * np.exp(-r * t), 0.0))
    assert np.all(np.abs(got[2] - vega) <= 2e-5 * vega)
    assert np.all(np.abs(got[4] - theta) <= 2e-5 * np.abs(theta))
