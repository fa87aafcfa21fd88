"""Portfolio reductions (bs_portfolio_f32) on the MI355X, through the C ABI.

* The sums equal the exact sums (math.fsum) of the map's own per-option
  outputs (bs_price_f32 / bs_price_greeks_f32) times the weights, up to the
  rounding of an FP64 reduction: each term w*p is exact in FP64, so only the
  additions round.
* Ragged and empty books, misaligned arrays (the one-option-per-work-item
  path), weights, and bit-reproducibility of repeated calls.
* Against the reference (the oracle's bit-exact prices), the price sum is
  within sum_i |w_i| * 1e-4 (the per-option parity bound); the observed
  difference is printed.
"""
import math

import numpy as np
import pytest

from p3arsec_amd import books

pytestmark = pytest.mark.gpu


def portfolio(capi, dbook, n, greeks, weights=None):
    out = capi.DeviceBuffer(40)
    pad = dbook.pad   # the weights get the book's misalignment too
    wbuf = None
    if weights is not None:
        wbuf = capi.DeviceBuffer.from_array(
            np.concatenate([np.zeros(pad, np.float32), weights.astype(np.float32)]))
    wptr = (wbuf.ptr + 4 * pad) if wbuf is not None else None
    capi.call("bs_portfolio_f32", *dbook.ptrs(), wptr, n, 1 if greeks else 0, out.ptr, None)
    capi.call("bs_stream_sync", None)
    sums = out.download(np.float64, 5 if greeks else 1)
    out.free()
    if wbuf is not None:
        wbuf.free()
    return sums


def map_outputs(capi, dbook, n, greeks):
    if greeks:
        return [o.download(np.float32, n) for o in capi.greeks(dbook)]
    return [capi.price(dbook).download(np.float32, n)]


def exact_sums(cols, w):
    res, scale = [], []
    for c in cols:
        terms = c.astype(np.float64) * (w.astype(np.float32).astype(np.float64) if w is not None else 1.0)
        res.append(math.fsum(terms.tolist()))
        scale.append(float(np.sum(np.abs(terms))))
    return np.array(res), np.array(scale)


@pytest.mark.parametrize("n", [0, 1, 2, 3, 255, 1023, 100_003, 1_000_000])
@pytest.mark.parametrize("greeks", [0, 1])
def test_sums_match_the_map(gpu, n, greeks):
    book = books.make_book(max(n, 1), books.SEED_BASE + 80 + n % 97).slice(0, n) if n else None
    if n == 0:
        db = gpu.DeviceBook(books.make_book(1, books.SEED_BASE + 80))
        sums = portfolio(gpu, db, 0, greeks)
        assert np.all(sums == 0.0)
        db.free()
        return
    rng = np.random.default_rng(n + 7 * greeks)
    w = rng.uniform(-2.0, 5.0, n).astype(np.float32)
    db = gpu.DeviceBook(book)
    cols = map_outputs(gpu, db, n, greeks)
    for weights in (None, w):
        got = portfolio(gpu, db, n, greeks, weights)
        ref, scale = exact_sums(cols, weights)
        assert np.all(np.abs(got - ref) <= 1e-13 * scale + 1e-300), (got, ref)
        again = portfolio(gpu, db, n, greeks, weights)
        assert np.array_equal(got.view(np.uint64), again.view(np.uint64))   # fixed order
    db.free()


def test_misaligned_arrays_take_the_scalar_path(gpu):
    n = 50_001
    book = books.make_book(n, books.SEED_BASE + 90)
    w = np.random.default_rng(3).uniform(0.5, 2.0, n).astype(np.float32)
    aligned = gpu.DeviceBook(book)
    shifted = gpu.DeviceBook(book, pad=1)
    cols = map_outputs(gpu, aligned, n, 1)
    for db in (aligned, shifted):
        got = portfolio(gpu, db, n, True, w)
        ref, scale = exact_sums(cols, w)
        assert np.all(np.abs(got - ref) <= 1e-13 * scale)
    aligned.free()
    shifted.free()


def test_price_sum_against_the_reference(gpu, oracle):
    n = 1_000_000
    book = books.make_book(n, books.SEED_BASE + 91)
    w = np.random.default_rng(4).uniform(0.0, 10.0, n).astype(np.float32)
    ref, _, _ = oracle.price_f32(book)
    db = gpu.DeviceBook(book)
    got = portfolio(gpu, db, n, False, w)[0]
    want = math.fsum((ref * w.astype(np.float64)).tolist())
    bound = float(np.sum(np.abs(w.astype(np.float64)))) * 1e-4
    print(f"\nportfolio 1M: |GPU sum - reference sum| = {abs(got - want):.3e} "
          f"(bound {bound:.3e}, relative {abs(got - want) / abs(want):.2e})")
    assert abs(got - want) <= bound
    db.free()


def test_argument_errors(gpu):
    L = gpu.load()
    db = gpu.DeviceBook(books.make_book(8, books.SEED_BASE + 92))
    assert L.bs_portfolio_f32(*db.ptrs(), None, 8, 0, None, None) == -1          # sums NULL
    out = gpu.DeviceBuffer(40)
    assert L.bs_portfolio_f32(*db.ptrs(), None, -1, 0, out.ptr, None) == -1      # n < 0
    page = gpu.DeviceBuffer(4096)                                                  # 5 sums need 40 B
    assert L.bs_portfolio_f32(*db.ptrs(), None, 8, 1, page.ptr + 4088, None) == -1
    db.free()
    out.free()
    page.free()


def _sums(capi, name, db, n, greeks, wptr, stream=None):
    out = capi.DeviceBuffer(40)
    capi.call(name, *db.ptrs(), wptr, n, greeks, out.ptr, stream)
    capi.call("bs_stream_sync", stream)
    got = out.download(np.uint64, 5 if greeks else 1)
    out.free()
    return got


@pytest.mark.parametrize("n", [511, 512, 513, 64 * 512 - 1, 64 * 512, 64 * 512 + 1, 1024 * 512 - 1,
                               1024 * 512, 2 * 1024 * 512 + 3, 8 * 1024 * 512 + 1,
                               8192 * 2048 - 1, 8192 * 2048 + 1, 1 << 25])
def test_one_launch_and_two_give_the_same_bits(gpu, n):
    """At the edges of blocks (512 options with one row), groups of 64 blocks,
    the rows per wave and the most blocks: the one-launch sums are the
    two-launch ones, and those of the same book off a vector boundary, bit for
    bit, and the exact sums within an FP64 reduction's rounding."""
    book = books.make_book(n, books.SEED_BASE + 93)
    w = np.random.default_rng(n).uniform(-1.0, 2.0, n).astype(np.float32)
    db, off = gpu.DeviceBook(book), gpu.DeviceBook(book, pad=1)
    wb = gpu.DeviceBuffer.from_array(w)
    wo = gpu.DeviceBuffer.from_array(np.concatenate([np.zeros(1, np.float32), w]))
    for greeks in (0, 1):
        want = _sums(gpu, "bs_portfolio_f32_noalloc", db, n, greeks, wb.ptr)
        got = _sums(gpu, "bs_portfolio_f32", db, n, greeks, wb.ptr)
        shifted = _sums(gpu, "bs_portfolio_f32", off, n, greeks, wo.ptr + 4)
        assert np.array_equal(got, want) and np.array_equal(shifted, want)
        if n < 3_000_000:
            ref, scale = exact_sums(map_outputs(gpu, db, n, greeks), w)
            assert np.all(np.abs(got.view(np.float64) - ref) <= 1e-13 * scale)
    for b in (db, off, wb, wo):
        b.free()


def test_many_calls_in_flight(gpu):
    """More calls than scratch slots at once, on four streams from four
    threads: every call's sums are its book's own."""
    import threading
    sizes = (700, 40_961, 300_001, 1_000_003)
    dbs = [gpu.DeviceBook(books.make_book(n, books.SEED_BASE + 94 + i)) for i, n in enumerate(sizes)]
    want = [[_sums(gpu, "bs_portfolio_f32_noalloc", d, n, g, None) for g in (0, 1)]
            for d, n in zip(dbs, sizes)]
    bad = []

    def work(k):
        st = gpu.Stream()
        outs = [gpu.DeviceBuffer(40) for _ in range(60)]
        for rep in range(5):
            for i, o in enumerate(outs):
                j = (i + k) % 4
                gpu.call("bs_portfolio_f32", *dbs[j].ptrs(), None, sizes[j], i & 1, o.ptr,
                         st.handle)
            st.sync()
            for i, o in enumerate(outs):
                j = (i + k) % 4
                if not np.array_equal(o.download(np.uint64, 5 if i & 1 else 1, st.handle),
                                      want[j][i & 1]):
                    bad.append((k, rep, i))
        for o in outs:
            o.free()
        st.destroy()

    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad[:5]
    for d in dbs:
        d.free()


def test_inside_a_callers_graph(gpu):
    """Captured, the call takes the form whose scratch is the graph's own;
    replays with eager calls between them give the eager sums."""
    import ctypes
    from test_gpu_capture import CAPTURE_THREAD_LOCAL, hip
    H, L, n = hip(), gpu.load(), 100_003
    db = gpu.DeviceBook(books.make_book(n, books.SEED_BASE + 98))
    want = _sums(gpu, "bs_portfolio_f32", db, n, 1, None)
    st, out = gpu.Stream(), gpu.DeviceBuffer(40)
    graph, gexec = ctypes.c_void_p(), ctypes.c_void_p()
    assert H.hipStreamBeginCapture(st.handle, CAPTURE_THREAD_LOCAL) == 0
    rc = L.bs_portfolio_f32(*db.ptrs(), None, n, 1, out.ptr, st.handle)
    assert H.hipStreamEndCapture(st.handle, ctypes.byref(graph)) == 0 and rc == 0
    assert H.hipGraphInstantiate(ctypes.byref(gexec), graph, None, None, 0) == 0
    for rep in range(4):
        assert H.hipGraphLaunch(gexec, st.handle) == 0
        gpu.call("bs_stream_sync", st.handle)
        assert np.array_equal(out.download(np.uint64, 5), want), rep
        assert np.array_equal(_sums(gpu, "bs_portfolio_f32", db, n, 1, None), want)
    H.hipGraphExecDestroy(gexec)
    H.hipGraphDestroy(graph)
    st.destroy()
    out.free()
    db.free()


@pytest.mark.parametrize("n", [1, 4097, 524_287, 1_048_577, 1_600_001, 2_500_003, 10_000_000])
@pytest.mark.parametrize("name", ["bs_portfolio_f32", "bs_portfolio_f32_noalloc"])
def test_price_sum_with_and_without_greeks(gpu, name, n):
    """sums[0] is the same bits whether Greeks are asked for or not, at every
    number of rows a wave takes, with weights and without."""
    rng = np.random.default_rng(n)
    db = gpu.DeviceBook(books.make_book(n, books.SEED_BASE + 84))
    w = gpu.DeviceBuffer.from_array(rng.uniform(-3.0, 10.0, n).astype(np.float32))
    for wptr in (None, w.ptr):
        one, five = (_sums(gpu, name, db, n, greeks, wptr) for greeks in (0, 1))
        assert one[0] == five[0]
    w.free()
    db.free()
