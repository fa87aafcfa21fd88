"""Workloads of the library, one entry each, for timing it and checking its outputs.

A case names an entry point of the C ABI (include/bs_mi355.h), reached through
the Python binding as a user's program reaches it, and the sizes of one call.
Books have the distributions of p3arsec_amd/books.py; swaptions are the
reference driver's portfolio or desks with later starts.  Inputs are device
tensors made from a seed, so no call waits for a host upload it would not have
in a program that keeps its books on the GPU.  exact() restates each path in
64-bit PyTorch.
"""
import ctypes
import math

import numpy as np
import torch

from p3arsec_amd import books, capi, swaptions

MAX_BOOK = 10_000_000      # the headline book
PASSES = 100               # NUM_RUNS of the reference
SERVE_BOOKS = 32


def listed():
    return [
        # One pricing call on the reference's CPU-sized book: a quote on a
        # small desk's positions, where the launch and the call are the cost.
        {"name": "price-4096", "kind": "price", "n": 4096, "types": "u8", "offset": 0},
        # The reference's NUM_RUNS loop over the same book in one call.
        {"name": "passes-4096", "kind": "passes", "n": 4096, "types": "i32", "passes": PASSES},
        # The second half of a book that is split in two: the arrays start at
        # an odd option, and so does the slice of the output.
        {"name": "price-slice-5m", "kind": "price", "n": 4_999_997, "types": "u8", "offset": 3},
        # The headline: one pass over 10M options, FP32 and FP64.
        {"name": "price-10m", "kind": "price", "n": MAX_BOOK, "types": "u8", "offset": 0},
        {"name": "price-f64-10m", "kind": "price_f64", "n": MAX_BOOK},
        # Risk of the whole book: price and adjoint.
        {"name": "greeks-10m", "kind": "greeks", "n": MAX_BOOK},
        # The value of one desk's book, and the weighted risk of all of it.
        {"name": "portfolio-64k", "kind": "portfolio", "n": 65_537, "greeks": False,
         "weights": False},
        {"name": "portfolio-greeks-10m", "kind": "portfolio", "n": MAX_BOOK, "greeks": True,
         "weights": True},
        # Loading the reference's records: AoS to SoA once per book.
        {"name": "repack-10m", "kind": "repack", "n": 9_999_991},
        # PARSEC's native swaptions run, the largest call.
        {"name": "swaptions-native", "kind": "swaptions", "count": 128, "trials": 1_000_000,
         "steps": 0, "factors": 3, "start": 0},
        # A swaptions desk with later starts on a finer curve.
        {"name": "swaptions-starts", "kind": "swaptions", "count": 32, "trials": 50_000,
         "steps": 21, "factors": 4, "start": 10},
        # One round of requests against resident books, replies on the host.
        {"name": "serve-32", "kind": "serve", "requests": SERVE_BOOKS, "most": 65_536},
    ]


def _log_uniform(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["price", "price", "price_f64", "greeks", "portfolio", "portfolio",
                       "passes", "repack", "swaptions", "swaptions", "serve"])
    if kind == "price":
        return {"kind": kind, "n": _log_uniform(rng, 1000, MAX_BOOK),
                "types": rng.choice(["u8", "u8", "i32"]), "offset": rng.choice([0, 0, 1, 2, 3])}
    if kind in ("price_f64", "greeks", "repack"):
        return {"kind": kind, "n": _log_uniform(rng, 1000, MAX_BOOK)}
    if kind == "portfolio":
        return {"kind": kind, "n": _log_uniform(rng, 1000, MAX_BOOK),
                "greeks": rng.random() < 0.5, "weights": rng.random() < 0.5}
    if kind == "passes":
        return {"kind": kind, "n": _log_uniform(rng, 256, 200_000),
                "types": rng.choice(["u8", "i32"]), "passes": rng.randint(2, PASSES)}
    if kind == "serve":
        return {"kind": kind, "requests": rng.randint(4, SERVE_BOOKS),
                "most": _log_uniform(rng, 4096, 262_144)}
    if rng.random() < 0.5:     # the driver's portfolio: PARSEC's smallest run to its native one
        return {"kind": kind, "count": rng.randint(1, 128),
                "trials": _log_uniform(rng, 1000, 1_000_000), "steps": 0, "factors": 3, "start": 0}
    factors = rng.randint(1, 6)
    steps = rng.randint(11, 32)
    return {"kind": kind, "count": rng.randint(1, 32), "trials": _log_uniform(rng, 1000, 50_000),
            "steps": steps, "factors": factors,
            "start": rng.randint(1, min(steps // 2, 64 // factors))}


# ---- inputs -----------------------------------------------------------------------
def _book(n, seed, dtype=torch.float32):
    """s, k, r, v, t, put with the distributions of books.make_book, on the GPU."""
    g = torch.Generator(device="cuda").manual_seed(seed)

    def uniform(lo, hi):
        return torch.rand(n, generator=g, device="cuda", dtype=dtype) * (hi - lo) + lo

    s = uniform(10.0, 200.0)
    return (s, s * uniform(0.5, 1.5), uniform(0.01, 0.10), uniform(0.05, 0.65),
            uniform(0.05, 2.0), torch.rand(n, generator=g, device="cuda") < 0.5)


def _type_array(put, types):
    return put.to(torch.uint8 if types == "u8" else torch.int32)


def _records(n, seed):
    """n of the reference's 36-byte OptionData records (blackscholes.c:89-100)."""
    s, k, r, v, t, put = _book(n, seed)
    z = torch.zeros_like(s)
    rec = torch.stack([s, k, r, z, v, t, z, z, z], 1).view(torch.int32)
    rec[:, 6] = torch.where(put, ord("P"), ord("C")).to(torch.int32)
    return rec.contiguous()


def _desk(case, seed):
    """(swaptions, base seed) of a swaptions case."""
    rng = np.random.default_rng(seed)
    if case["steps"] == 0:
        return swaptions.parsec_portfolio(case["count"], int(rng.integers(1, 1 << 30)))
    n, factors, sws = case["steps"], case["factors"], []
    sigma = rng.uniform(0.001, 0.01, (factors, n - 1))
    yld = 0.05 + 0.004 * np.arange(n)
    for i in range(case["count"]):
        years = float(rng.uniform(5.0, 20.0))
        dt = years / n
        start = 1 + i % case["start"]
        tenor = int(rng.integers(2, n - start))
        sws.append({"strike": float(rng.uniform(0.05, 0.2)), "compounding": 0.0,
                    "maturity": start * dt, "tenor": tenor * dt, "interval": dt, "years": years,
                    "yield": yld, "factors": sigma})
    return sws, int(rng.integers(1, 1 << 30))


def _request_sizes(case):
    """Book sizes of a round of requests: log-uniform over [1, most], the
    fractions of the golden ratio in place of random ones."""
    golden = (math.sqrt(5.0) - 1.0) / 2.0
    return [max(1, round(case["most"] ** ((1.0 + i * golden) % 1.0 if i else 1.0)))
            for i in range(case["requests"])]


def _request_kinds(case):
    return [capi.REQ_GREEKS if i % 3 == 1 else capi.REQ_PRICE for i in range(case["requests"])]


class _Server:
    """A serving context with resident books, as a pricing service keeps one."""

    def __init__(self, case, seed):
        sizes = _request_sizes(case)
        self.books = [books.make_book(n, seed * 1000 + i) for i, n in enumerate(sizes)]
        self.kinds = _request_kinds(case)
        count, i64 = len(sizes), ctypes.c_int64
        opts = capi.ServeOpts()
        self.ctx = ctypes.c_void_p()
        capi.call("bs_ctx_create", 0, 256 << 20, ctypes.byref(opts), ctypes.byref(self.ctx))
        self.ids, self.c_kinds = (i64 * count)(), (ctypes.c_int * count)(*self.kinds)
        self.tickets = (i64 * count)()
        for i, b in enumerate(self.books):
            book = i64(0)
            capi.call("bs_book_register", self.ctx, *[a.ctypes.data for a in b.arrays()], b.n,
                      ctypes.byref(book))
            self.ids[i] = book.value
        total = sum(b.n for b in self.books)
        risky = sum(b.n for b, k in zip(self.books, self.kinds) if k == capi.REQ_GREEKS)
        self.price = np.empty(total, np.float32)
        self.risk = np.empty((4, risky), np.float32)
        self.where, at, at_risk = [], 0, 0      # the reply arrays of each request
        for b, k in zip(self.books, self.kinds):
            greeks = k == capi.REQ_GREEKS
            to = [self.price[at:].ctypes.data]
            to += [self.risk[q, at_risk:].ctypes.data if greeks else None for q in range(4)]
            self.where.append(to)
            at, at_risk = at + b.n, at_risk + (b.n if greeks else 0)

    def round(self):
        count = len(self.books)
        capi.call("bs_submit_many", self.ctx, self.ids, self.c_kinds, None, count, self.tickets)
        for i in range(count):
            capi.call("bs_wait", self.ctx, self.tickets[i], -1)
            capi.call("bs_result_copy", self.ctx, self.tickets[i], *self.where[i])
        capi.call("bs_result_release_many", self.ctx, self.tickets, count)
        return self.price, self.risk

    def __del__(self):
        if getattr(self, "ctx", None):
            capi.load().bs_ctx_destroy(self.ctx)
            self.ctx = None


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case, "stream": torch.cuda.current_stream().cuda_stream}
    if kind == "serve":
        state["server"] = _Server(case, seed)
        return state
    if kind == "swaptions":
        sws, base = _desk(case, seed)
        state.update(desk=swaptions.Prepared(sws), seed=base)
        return state
    n = case["n"]
    if kind == "repack":
        state["records"] = _records(n, seed)
        state["out"] = [torch.empty(n, device="cuda") for _ in range(5)]
        state["out"].append(torch.empty(n, device="cuda", dtype=torch.uint8))
        return state
    off = case.get("offset", 0)
    dtype = torch.float64 if kind == "price_f64" else torch.float32
    arrays = _book(n + off, seed, dtype)
    state["book"] = [a[off:] for a in arrays[:5]]
    state["types"] = _type_array(arrays[5], case.get("types", "u8"))[off:]
    if kind == "portfolio":
        if case["weights"]:
            g = torch.Generator(device="cuda").manual_seed(seed + 1)
            state["weights"] = torch.rand(n, generator=g, device="cuda") * 9.0 + 1.0
        state["out"] = [torch.empty(5 if case["greeks"] else 1, device="cuda",
                                    dtype=torch.float64)]
    else:
        state["out"] = [torch.empty(n + off, device="cuda", dtype=dtype)[off:]
                        for _ in range(5 if kind == "greeks" else 1)]
    return state


# ---- one pass ---------------------------------------------------------------------
def run(state):
    case, stream = state["case"], state["stream"]
    kind = case["kind"]
    if kind == "serve":
        return state["server"].round()
    if kind == "swaptions":
        return swaptions.price(state["desk"], case["trials"], state["seed"], stream=stream)
    out, n = state["out"], case["n"]
    to = [o.data_ptr() for o in out]
    if kind == "repack":
        capi.call("bs_repack_aos_f32", state["records"].data_ptr(), n, *to, stream)
        return out
    book = [a.data_ptr() for a in state["book"]]
    types = state["types"].data_ptr()
    if kind == "price":
        entry = "bs_price_f32" if case["types"] == "u8" else "bs_price_i32type_f32"
        capi.call(entry, *book, types, *to, n, stream)
    elif kind == "price_f64":
        capi.call("bs_price_f64", *book, types, *to, n, stream)
    elif kind == "greeks":
        capi.call("bs_price_greeks_f32", *book, types, *to, n, stream)
    elif kind == "passes":
        capi.call("bs_price_passes_f32", *book, types, state["types"].element_size(), *to, n,
                  case["passes"], stream)
    else:
        weights = state["weights"].data_ptr() if case["weights"] else None
        capi.call("bs_portfolio_f32", *book, types, weights, n, int(case["greeks"]), *to, stream)
    return out


# ---- what a pass cannot do without -------------------------------------------------
# Flops per option of the price formula and of price with its adjoint.
PRICE_FLOPS, GREEKS_FLOPS = 70, 110


def work(case):
    kind = case["kind"]
    if kind == "serve":
        cost = {capi.REQ_PRICE: (25, PRICE_FLOPS), capi.REQ_GREEKS: (41, GREEKS_FLOPS)}
        each = [(n, *cost[k]) for n, k in zip(_request_sizes(case), _request_kinds(case))]
        return {"bytes": sum(n * b for n, b, _ in each), "flops": sum(n * f for n, _, f in each)}
    if kind == "swaptions":
        paths, factors = case["count"] * case["trials"], case["factors"]
        steps = case["steps"] or swaptions.N_STEPS
        start = (1 + case["start"]) / 2 if case["start"] else 1.5
        # per draw the generator and the inverse normal, per live point of the
        # curve and step the drift and the shocks, per rate an exponential
        flops = start * factors * 25 + start * steps / 2 * (2 * factors + 2) + steps / 2 * 20
        return {"bytes": case["count"] * 16, "flops": paths * flops}
    n = case["n"]
    if kind == "repack":
        return {"bytes": n * 57, "flops": 0}
    if kind == "price_f64":
        return {"bytes": n * 49, "flops": n * PRICE_FLOPS}
    if kind == "greeks":
        return {"bytes": n * 41, "flops": n * GREEKS_FLOPS}
    if kind == "portfolio":
        return {"bytes": n * (25 if case["weights"] else 21),
                "flops": n * (GREEKS_FLOPS if case["greeks"] else PRICE_FLOPS)}
    passes = case.get("passes", 1)
    return {"bytes": n * (25 if case["types"] == "u8" else 28), "flops": n * PRICE_FLOPS * passes}


# ---- the same in 64 bits -------------------------------------------------------------
def _cndf(x):
    """Abramowitz & Stegun 26.2.17, as the reference approximates the normal."""
    ax = x.abs()
    k = 1.0 / (1.0 + 0.2316419 * ax)
    poly = k * (0.319381530 + k * (-0.356563782 + k * (1.781477937 + k * (
        -1.821255978 + k * 1.330274429))))
    y = 1.0 - 0.39894228040143270286 * torch.exp(-0.5 * ax * ax) * poly
    return torch.where(x < 0, 1.0 - y, y)


def _price64(s, k, r, v, t, put):
    den = v * torch.sqrt(t)
    d1 = ((r + 0.5 * v * v) * t + torch.log(s / k)) / den
    n1, n2 = _cndf(d1), _cndf(d1 - den)
    fv = k * torch.exp(-r * t)
    return torch.where(put, fv * (1.0 - n2) - s * (1.0 - n1), s * n1 - fv * n2)


def _greeks64(arrays, put):
    """price, delta, vega, rho and theta of the same formula."""
    out = []
    for at in range(0, len(put), 1 << 21):
        s, k, r, v, t = (a[at:at + (1 << 21)].double().requires_grad_() for a in arrays)
        p = _price64(s, k, r, v, t, put[at:at + (1 << 21)])
        p.sum().backward()
        out.append((p.detach(), s.grad, v.grad, r.grad, -t.grad))
    return [torch.cat(c) for c in zip(*out)]


# Moro's inverse normal (Moro 1995; Glasserman 2003, fig. 2.13).
_MORO_A = (2.50662823884, -18.61500062529, 41.39119773534, -25.44106049637)
_MORO_B = (-8.47351093090, 23.08336743743, -21.06224101826, 3.13082909833)
_MORO_C = (0.3374754822726147, 0.9761690190917186, 0.1607979714918209, 0.0276438810333863,
           0.0038405729373609, 0.0003951896511919, 0.0000321767881768, 0.0000002888167364,
           0.0000003960315187)


def _horner(x, c):
    y = torch.full_like(x, c[-1])
    for a in reversed(c[:-1]):
        y = y * x + a
    return y


def _normal(counter):
    """The normal draw of a counter: PARSEC's RanUnif and CumNormalInv."""
    m31 = (1 << 31) - 1
    u = ((counter * 1513517) % m31 * 16807 % m31).double() * 4.656612875e-10
    x = u - 0.5
    r = x * x
    central = x * _horner(r, _MORO_A) / (_horner(r, _MORO_B) * r + 1.0)
    t = torch.log(-torch.log(torch.where(x > 0, 1.0 - u, u)))
    tail = _horner(t, _MORO_C)
    return torch.where(x.abs() < 0.42, central, torch.where(x < 0, -tail, tail))


def _swaption64(sw, seed, trials):
    """(price, standard error): HJM paths by time step, the whole curve."""
    yld, sigma = np.asarray(sw["yield"]), np.asarray(sw["factors"])
    n, factors = len(yld), sigma.shape[0]
    dt = sw["years"] / n
    m, points = int(sw["maturity"] / dt + 0.5), int(sw["tenor"] / dt + 0.5)
    freq = int(sw["interval"] / dt + 0.5)
    curve = int(n - sw["maturity"] / dt + 0.5)
    j = np.arange(n)
    forward = (j + 1) * yld - j * np.concatenate([[0.0], yld[:-1]])
    cum = np.concatenate([np.zeros((factors, 1)), 0.5 * dt * np.cumsum(sigma, 1) ** 2], 1)
    drift = np.diff(cum, axis=1).sum(0) * dt
    cash = np.zeros(curve)
    grow = math.exp(sw["strike"] * sw["interval"])      # compounding 0: a continuous strike
    for at in range(freq, points + 1, freq):
        cash[at] = grow - 1.0 if at != points else grow
    block = swaptions.BLOCK_SIZE
    paths = -(-trials // block) * block
    sums = torch.zeros(2, dtype=torch.float64, device="cuda")
    for first in range(0, paths, 1 << 20):
        p = torch.arange(first, min(paths, first + (1 << 20)), device="cuda")
        f = torch.tensor(forward, device="cuda").expand(len(p), n)
        disc = torch.ones(len(p), dtype=torch.float64, device="cuda")
        for s in range(m):
            disc = disc * torch.exp(-f[:, 0] * dt)
            z = _normal((seed + p * ((n - 1) * factors) + s * factors)[:, None]
                        + torch.arange(factors, device="cuda"))
            live = n - 1 - s
            shock = sum(z[:, i:i + 1] * torch.tensor(sigma[i, :live], device="cuda")
                        for i in range(factors))
            f = f[:, 1:] + torch.tensor(drift[:live], device="cuda") + math.sqrt(dt) * shock
        leg = torch.zeros_like(disc)
        bond = torch.ones_like(disc)
        for at in range(points + 1):
            leg = leg + cash[at] * bond
            if at < f.shape[1]:
                bond = bond * torch.exp(-f[:, at] * dt)
        pay = (leg - 1.0).clamp(min=0.0) * disc
        sums += torch.stack([pay.sum(), (pay * pay).sum()])
    total, squares = sums.tolist()
    return (total / trials,
            math.sqrt((squares - total * total / trials) / (trials - 1.0)) / math.sqrt(trials))


def exact(case, seed):
    kind = case["kind"]
    if kind == "serve":
        server = _Server(case, seed)
        price, risk = [], []
        for b, k in zip(server.books, server.kinds):
            arrays = [torch.from_numpy(a).cuda() for a in b.arrays()]
            cols = _greeks64(arrays[:5], arrays[5] != 0)
            price.append(cols[0])
            if k == capi.REQ_GREEKS:
                risk.append(torch.stack(cols[1:]))
        return torch.cat(price), torch.cat(risk, 1)
    if kind == "swaptions":
        sws, base = _desk(case, seed)
        got = [_swaption64(sw, base + i, case["trials"]) for i, sw in enumerate(sws)]
        return np.array([g[0] for g in got]), np.array([g[1] for g in got])
    if kind == "repack":
        rec = _records(case["n"], seed)
        fields = rec.view(torch.float32)
        return [fields[:, j].double() for j in (0, 1, 2, 4, 5)] + [None]
    state = prepare(case, seed)
    arrays, put = state["book"], state["types"] != 0
    if kind == "greeks":
        return _greeks64(arrays, put)
    if kind == "portfolio":
        cols = (_greeks64(arrays, put) if case["greeks"] else
                [_price64(*(a.double() for a in arrays), put)])
        w = state["weights"].double() if case["weights"] else 1.0
        return [torch.stack([(c * w).sum() for c in cols])]
    return [_price64(*(a.double() for a in arrays), put)]
