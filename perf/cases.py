"""Timing cases: the pricing work a user of this library has it do, through its public entry points.

A case names an entry point (`op`), a distribution of options (`dist`), their number (`n`) and the options of the call:

  plan       capi.Plan.execute over device arrays: a service that keeps its batch on the GPU
  price      capi.price on host arrays, the drop-in for seq::computeOptions
  price_f32  capi.price_f32, the same for a caller built with real = float (the reference's default)
  batch      capi.Batch.price: a batch uploaded once and priced again and again, prices back on the host
  surrogate  Surrogate.price: the ensemble with the FP64 tree as fallback
  train      Surrogate.train: one epoch of forward, backward and Adam over every member

The distributions are those of the repository's workloads and of the reference's benchmark sets.
"""
import functools
import math

import numpy as np
import torch

import __graft_entry__

pkg = __graft_entry__.load_package()
capi, surrogate = pkg.capi, pkg.surrogate

REAL_FIELDS = ("strike", "maturity", "length", "a", "sigma")
SPREAD_THRESHOLD = 8.0e-5  # sends 1% to 3% of the in-box options of an ensemble as prepared here to the tree


def listed():
    return [
        # Hull's book example, five options handed over as host arrays: the smallest call, all latency
        {"name": "price_book_5", "op": "price", "dist": "book", "n": 5},
        # a strike ladder on one bond, resident on the GPU: small enough that launches count
        {"name": "plan_ladder_1k", "op": "plan", "dist": "ladder", "n": 1000, "precision": "fp64"},
        # the headline batch: 90% small trees, 10% large ones
        {"name": "plan_skewed_60k", "op": "plan", "dist": "skewed", "n": 60000, "precision": "fp64"},
        # the same batch for a user who asked for mixed precision
        {"name": "plan_skewed_60k_mixed", "op": "plan", "dist": "skewed", "n": 60000, "precision": "mixed"},
        # the reference's random set: widths 7 to 511, heights to 1,200 steps
        {"name": "plan_rand_65k", "op": "plan", "dist": "rand", "n": 65536, "precision": "fp64"},
        # many tiny trees (3 to 21 nodes wide), an odd count
        {"name": "plan_tiny_250k", "op": "plan", "dist": "tiny", "n": 250007, "precision": "fp64"},
        # the largest batch: what the surrogate is measured against
        {"name": "plan_box_mix_1m", "op": "plan", "dist": "box_mix", "n": 1000000, "precision": "fp64"},
        # the reference's skewed set from a default (float) build, host arrays in and out
        {"name": "price_f32_ref_skewed_65k", "op": "price_f32", "dist": "ref_skewed", "n": 65536},
        # an uploaded batch priced repeatedly, an odd count
        {"name": "batch_skewed_20k", "op": "batch", "dist": "skewed", "n": 20011, "form": "wave"},
        # the same through the one-lane-per-option form, which the cuda-option runners select
        {"name": "batch_lane_uniform_16k", "op": "batch", "dist": "uniform", "n": 16384, "form": "lane"},
        # the ensemble in front of the tree on the 95% / 5% mix
        {"name": "surrogate_box_mix_500k", "op": "surrogate", "dist": "box_mix", "n": 500000},
        # one epoch of training at the default batch
        {"name": "train_131k", "op": "train", "dist": "box", "n": 131072, "batch": 8192},
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    # most options per distribution that stay below the largest listed case's cost
    most = {"ladder": 20000, "skewed": 500000, "rand": 200000, "tiny": 1000000, "box_mix": 800000, "uniform": 500000,
            "ref_skewed": 500000}
    op = rng.choice(["plan", "plan", "plan", "price", "price_f32", "batch", "surrogate", "train"])
    if op == "plan":
        dist = rng.choice(sorted(most))
        return {"op": op, "dist": dist, "n": size(20, most[dist]), "precision": rng.choice(["fp64", "fp64", "mixed"])}
    if op in ("price", "price_f32"):
        dist = rng.choice(["skewed", "ref_skewed", "ladder", "uniform"])
        return {"op": op, "dist": dist, "n": size(1, 100000 if dist != "ladder" else 20000)}
    if op == "batch":
        form = rng.choice(["wave", "wave", "lane"])
        dist = rng.choice(["uniform", "ladder"] if form == "lane" else ["skewed", "rand", "ref_skewed"])
        return {"op": op, "dist": dist, "n": size(10, 30000 if form == "lane" else 100000), "form": form}
    if op == "surrogate":
        return {"op": op, "dist": "box_mix", "n": size(1000, 500000)}
    batch = 128 * rng.choice([8, 16, 24, 32, 48, 64])
    return {"op": op, "dist": "box", "n": size(batch, 131072), "batch": batch}


# ------------------------------------------------------------------- inputs
def _rate_for_width(width, steps=12):
    """The smallest reversion rate with five decimals whose tree is `width` nodes wide."""
    lo = -np.log1p(-0.184 / ((width - 1) // 2)) * steps
    return np.ceil(lo * 1e5 + 0.5) / 1e5


def _inputs(dist, n, seed):
    """Options (field -> array) and the yield curve (rates, days)."""
    r = np.random.default_rng(seed)
    o = {"strike": r.uniform(60, 100, n), "sigma": r.uniform(0.005, 0.02, n), "type": r.integers(0, 2, n)}
    o["term_steps"] = np.full(n, 12)
    if dist == "book":  # a 3-year put on a 9-year bond
        o.update(strike=63 + r.uniform(-3, 3, n), maturity=np.full(n, 9.0), length=np.full(n, 3.0), a=np.full(n, 0.1),
                 sigma=np.full(n, 0.01), type=np.ones(n), term_steps=1 + np.arange(n) % 5)
    elif dist == "ladder":  # puts on one bond at many strikes
        o.update(maturity=np.full(n, 10.0), length=np.full(n, 5.0), a=np.full(n, 0.1), sigma=np.full(n, 0.01),
                 type=np.ones(n))
    elif dist == "uniform":  # one tree shape, quotes around it
        o.update(maturity=np.full(n, 9.0), length=np.full(n, 3.0), a=np.full(n, 0.1), type=np.ones(n))
    elif dist == "skewed":
        large = r.permutation(n) < round(0.1 * n)
        mat = np.where(large, r.uniform(10, 30, n), r.uniform(1, 5, n))
        o.update(maturity=mat, length=r.uniform(0.2, 0.8, n) * mat, term_steps=np.where(large, 36, 12),
                 a=np.where(large, r.uniform(0.01, 0.05, n), r.uniform(0.1, 0.2, n)))
    elif dist == "rand":
        o.update(maturity=r.integers(1, 101, n), length=np.full(n, 3.0), a=_rate_for_width(2 * r.integers(3, 256, n) + 1))
    elif dist == "ref_skewed":
        large = r.permutation(n) < np.ceil(0.01 * n)
        width = np.where(large, 2 * r.integers(205, 256, n) + 1, 2 * r.integers(3, 54, n) + 1)
        o.update(maturity=np.where(large, r.integers(70, 101, n), r.integers(1, 31, n)), length=np.full(n, 3.0),
                 a=_rate_for_width(width), type=np.ones(n), sigma=np.full(n, 0.01))
    elif dist == "tiny":
        width = 2 * r.integers(1, 11, n) + 1
        mat = r.uniform(1, 30, n)
        o.update(maturity=mat, length=r.uniform(0.2, 0.8, n) * mat,
                 a=np.where(width == 3, 3.0, _rate_for_width(np.maximum(width, 5))))
    elif dist in ("box", "box_mix"):
        length, a = r.uniform(1, 30, n), r.uniform(0.01, 0.2, n)
        mat = length + r.uniform(1, 10, n)
        if dist == "box_mix":  # 5% outside the training box: fast reversion, or a long option
            u = r.uniform(0, 1, n)
            a = np.where(u < 0.025, a + 0.2, a)
            late = u > 0.975
            mat, length = np.where(late, mat + 30, mat), np.where(late, length + 30, length)
            over = late & (length > 40)
            mat, length = np.where(over, mat - 20, mat), np.where(over, length - 20, length)
        o.update(maturity=mat, length=length, term_steps=np.where(r.integers(0, 2, n) == 0, 12, 36), a=a)
    else:
        raise ValueError(dist)
    o["term_unit"] = np.full(n, 365)
    kinds = {"term_unit": np.uint16, "term_steps": np.uint16, "type": np.int8}
    o = {f: np.ascontiguousarray(v, dtype=kinds.get(f, np.float64)) for f, v in o.items()}
    k = np.arange(1, 121)
    return o, (0.01 + 0.03 * (k - 1) / 119.0, np.rint(365.0 * k / 12.0).astype(np.int32))


def _weights(seed, members=4):
    """Ensemble parameters: hidden layers that keep their signal's size, output layers whose members differ by about what
    those of a trained ensemble do (1e-4 in price)."""
    r = np.random.default_rng(seed + 101)
    P = np.zeros((members, surrogate.NPARAMS), np.float32)
    for m in range(members):
        for k, off in surrogate.OFFSETS.items():
            count, fan_in = int(np.prod(surrogate.SHAPES[k])), 8 if k == "W1" else 256
            gain = 0.1 if k[0] == "b" else 0.01 if k == "W5" else 2.5
            P[m, off:off + count] = gain * r.uniform(-1, 1, count) / math.sqrt(fan_in)
        P[m, surrogate.OFFSETS["b5"]] = 0.0
    return P


class _Device:
    """A torch tensor as the device buffer the bindings take (an address in .value)."""

    def __init__(self, host):
        self.t = torch.from_numpy(host).cuda()
        self.value = self.t.data_ptr()


@functools.lru_cache(maxsize=None)
def _stream():
    return torch.cuda.Stream()


def _device(o, curve):
    dev = {f: _Device(v) for f, v in o.items()}
    dev.update(rates=_Device(curve[0]), days=_Device(curve[1]), out=_Device(np.zeros(len(o["strike"]))),
               n=len(o["strike"]), ny=len(curve[0]))
    return dev


def prepare(case, seed):
    n, op = case["n"], case["op"]
    o, curve = _inputs(case["dist"], n, seed)
    s = {"op": op}
    if op in ("price", "price_f32", "batch"):
        s["opts"], s["yield"] = pkg.Options(**o), pkg.Yield(*curve)
        s["cfg"] = capi.config(form=capi.FORM_LANE if case.get("form") == "lane" else capi.FORM_AUTO)
        if op == "batch":
            s["batch"] = capi.Batch(s["opts"], s["yield"])
        return s
    s["dev"] = dev = _device(o, curve)
    if op == "plan":
        mixed = case["precision"] == "mixed"
        s["plan"] = capi.Plan(n, dev["ny"], capi.config(precision=capi.PREC_MIXED if mixed else capi.PREC_FP64))
    elif op == "surrogate":
        s["surr"] = surrogate.Surrogate(0, n, dev["ny"], surrogate.config(spread_threshold=SPREAD_THRESHOLD))
        s["surr"].set_params(_weights(seed))
        s["plan"] = surrogate.fallback_plan(n, dev["ny"])
    else:
        # the library's own initial weights and data order; labels: the closed form (what the network's residual is
        # taken from) and a lattice-sized difference
        r = np.random.default_rng(seed + 7)
        labels = _closed_form(o, curve)[0].cpu().numpy() + 0.01 * np.sin(o["strike"] + 20 * o["a"]) * r.uniform(0.5, 1, n)
        s["surr"] = surrogate.Surrogate(n, 1, dev["ny"], surrogate.config(seed=seed, batch=case["batch"], warmup_frac=0.0))
        s["surr"].set_training_data(dev, _Device(labels))
    torch.cuda.synchronize()
    return s


def run(s):
    op = s["op"]
    if op == "plan":
        s["plan"].execute(s["dev"], stream=_stream().cuda_stream)
        return s["dev"]["out"].t
    if op == "price":
        return capi.price(s["opts"], s["yield"], s["cfg"])
    if op == "price_f32":
        return capi.price_f32(s["opts"], s["yield"], s["cfg"])
    if op == "batch":
        return s["batch"].price(s["cfg"])
    if op == "surrogate":
        s["surr"].price(s["plan"], s["dev"])
        return s["dev"]["out"].t
    loss = s["surr"].train(1, 1 << 20)["loss"]
    return {"loss": loss, "params": s["surr"].get_params()}


# --------------------------------------------------------------------- work
def _shape(o):
    """Tree constants of every option: n, exercise step (-1: none), jmax, M, dr, dt."""
    tuy = np.ceil(365.0 / o["term_unit"])
    n = (o["term_steps"] * tuy * o["maturity"]).astype(np.int64)
    dt = tuy / o["term_steps"]
    M = np.exp(-o["a"] * dt) - 1
    dr = np.sqrt(3 * o["sigma"] ** 2 * (1 - np.exp(-2 * o["a"] * dt)) / (2 * o["a"]))
    q = o["length"] / dt
    e = np.where((q > -1) & (q < n), q.astype(np.int64), -1)
    return {"n": n, "e": e, "jmax": (-0.184 / M).astype(np.int64) + 1, "M": M, "dr": dr, "dt": dt}


def _shape_f32(o):
    """The same as a real = float caller derives them (floats; exp, sqrt and ceil in double)."""
    f = np.float32
    mat, length, a, sg = (o[k].astype(f) for k in ("maturity", "length", "a", "sigma"))
    tuy = np.ceil((f(365) / o["term_unit"].astype(f)).astype(np.float64)).astype(np.int64)
    n = ((o["term_steps"].astype(np.int64) * tuy).astype(f) * mat).astype(np.int64)
    dt = tuy.astype(f) / o["term_steps"].astype(f)
    V = (sg * sg).astype(np.float64) * (1 - np.exp((f(-2) * a * dt).astype(np.float64))) / (f(2) * a).astype(np.float64)
    dr = np.sqrt(3 * V).astype(f)
    M = (np.exp((-a * dt).astype(np.float64)) - 1).astype(f)
    q = length / dt
    e = np.where((q > -1) & (q < n), q.astype(np.int64), -1)
    d = {"n": n, "e": e, "jmax": (f(-0.184) / M).astype(np.int64) + 1}
    d.update({k: v.astype(np.float64) for k, v in (("M", M), ("dr", dr), ("dt", dt))})
    return d


def _tree_flops(o):
    """Each node of the tree below the exercise date once, and each bond node above it that the exercise nodes reach,
    at two multiply-adds."""
    c = _shape(o)
    n, e, J = c["n"], c["e"], c["jmax"]

    def upto(m):
        m = np.maximum(m, 0)
        return np.where(m <= J, m * (m + 1) // 2, J * (J + 1) // 2 + (m - J) * J)

    ep = np.minimum(e, J)
    nodes = 2 * upto(e) + e + 2 * (upto(ep + n - 1 - e) - upto(ep - 1)) + n - e
    return 4.0 * float(np.where(e < 0, 0, nodes).sum())


def work(case):
    n, op = case["n"], case["op"]
    o, curve = _inputs(case["dist"], min(n, 50000), 1)
    tree, per = _tree_flops(o) / min(n, 50000), 8 * 5 + 5 + 8
    if op == "price_f32":
        per = 4 * 5 + 5 + 4
    if op == "surrogate":  # four members on 95% of the batch, the tree on the rest
        return {"bytes": n * per + 12 * len(curve[0]), "flops": n * (0.95 * 4 * 2 * 199168 + 0.07 * tree)}
    if op == "train":
        steps = n // case["batch"]
        # a gathered row and its label; weights and both moments in and out
        return {"bytes": 4 * steps * (case["batch"] * 40 + 6 * 4 * 199937), "flops": 4.0 * steps * case["batch"] * 6 * 199168}
    return {"bytes": n * per + 12 * len(curve[0]), "flops": n * tree}


# -------------------------------------------------------------------- exact
def _zero_rates(t, curve):
    """The curve at t years: linear in whole days, flat beyond its ends."""
    days = torch.floor(t * 365.0 + 0.5)
    x, p = (torch.as_tensor(v, dtype=torch.float64, device=t.device) for v in (curve[1], curve[0]))
    hi = torch.clamp(torch.searchsorted(x, days), 1, len(x) - 1)
    lo = hi - 1
    w = torch.clamp((days - x[lo]) / (x[hi] - x[lo]), 0.0, 1.0)
    return p[lo] + w * (p[hi] - p[lo])


def _tree(o, c, curve):
    """The trinomial tree as it is written down: Arrow-Debreu prices up with a shift fitted to the curve at each step, bond
    values back down with those shifts, the payoff at the exercise step."""
    g = "cuda" if torch.cuda.is_available() else "cpu"
    price = torch.empty(len(c["n"]), dtype=torch.float64, device=g)
    order = np.lexsort((c["jmax"], c["n"] // 32))
    at = 0
    while at < len(order):
        end = at + 1
        top = int(c["jmax"][order[at]])
        while end < len(order) and end - at < 16384:
            J = max(top, int(c["jmax"][order[end]]))
            # a group shares about a height; a much wider tree starts its own
            if (2 * J + 1) * (end - at + 1) > 12_000_000 or c["n"][order[end]] > c["n"][order[at]] * 1.1 + 32:
                break
            if end - at > 512 and J > 1.5 * top + 8:
                break
            top = J
            end += 1
        idx = order[at:end]
        price[torch.as_tensor(idx, device=g)] = _tree_group({k: v[idx] for k, v in o.items()},
                                                             {k: v[idx] for k, v in c.items()}, curve, g)
        at = end
    return price


def _tree_group(o, c, curve, g):
    f = {k: torch.as_tensor(v.astype(np.float64), device=g)[:, None] for k, v in c.items()}
    n, e, J, M, dr, dt = (f[k] for k in ("n", "e", "jmax", "M", "dr", "dt"))
    Jm, N = int(c["jmax"].max()), int(c["n"].max())
    j = torch.arange(-Jm, Jm + 1, dtype=torch.float64, device=g)[None, :]
    m, W = len(c["n"]), 2 * Jm + 1
    x = j * M
    inside = (j.abs() < J).double()
    up, mid, dn = ((1 / 6 + (x * x + x) / 2) * inside, (2 / 3 - x * x) * inside, (1 / 6 + (x * x - x) / 2) * inside)
    # the edges branch inwards: j = J to J, J-1, J-2 and j = -J to -J, -J+1, -J+2
    hi, lo = (j == J).double(), (j == -J).double()
    mid = mid + hi * (7 / 6 + (x * x + 3 * x) / 2) + lo * (7 / 6 + (x * x - 3 * x) / 2)
    dn = dn + hi * (-1 / 3 - x * x - 2 * x)
    up = up + lo * (-1 / 3 - x * x + 2 * x)
    dn2, up2 = hi * (1 / 6 + (x * x + x) / 2), lo * (1 / 6 + (x * x - x) / 2)
    up2 = up2[:, :-2] if W > 2 else up2
    E = torch.exp(-j * dr * dt)
    steps = torch.arange(1, N + 2, dtype=torch.float64, device=g)[None, :] * dt
    logP = -_zero_rates(steps, curve) * steps  # of step 1, 2, ...
    Q = torch.zeros(m, W, dtype=torch.float64, device=g)
    Q[:, Jm] = 1.0
    shift = torch.empty(m, N + 1, dtype=torch.float64, device=g)  # alpha dt
    for i in range(N):
        qe = Q * E
        shift[:, i] = torch.log(qe.sum(1)) - logP[:, i]
        qe *= torch.exp(-shift[:, i])[:, None]
        Q = mid * qe
        Q[:, 1:] += (up * qe)[:, :-1]
        Q[:, :-1] += (dn * qe)[:, 1:]
        Q[:, 2:] += up2 * qe[:, :-2]
        Q[:, :-2] += (dn2 * qe)[:, 2:]
    X = torch.as_tensor(o["strike"].astype(np.float64), device=g)[:, None]
    put = torch.as_tensor(o["type"] == 1, device=g)[:, None]
    B = torch.full((m, W), 100.0, dtype=torch.float64, device=g)
    for i in range(N - 1, -1, -1):
        V = mid * B
        V[:, :-1] += up[:, :-1] * B[:, 1:]
        V[:, 1:] += dn[:, 1:] * B[:, :-1]
        V[:, :-2] += up2 * B[:, 2:]
        V[:, 2:] += dn2[:, 2:] * B[:, :-2]
        V *= E * torch.exp(-shift[:, i])[:, None]
        B = torch.where(n > i, V, B)
        due = e == i
        B = torch.where(due, torch.clamp(torch.where(put, X - B, B - X), min=0.0), B)
    return B[:, Jm]


def _closed_form(o, curve):
    """The bond option in closed form on the tree's dates, and the network's eight inputs."""
    g = "cuda" if torch.cuda.is_available() else "cpu"
    c = _shape(o)
    t = {k: torch.as_tensor(v.astype(np.float64), device=g) for k, v in {**o, **c}.items()}
    X, a, sg, dt = t["strike"], t["a"], t["sigma"], t["dt"]
    T, S = t["e"] * dt, t["n"] * dt
    PT, PS = torch.exp(-_zero_rates(T, curve) * T), torch.exp(-_zero_rates(S, curve) * S)
    B = (1 - torch.exp(-a * (S - T))) / a
    var = (1 - torch.exp(-2 * a * T)) / (2 * a)
    sp = sg * B * torch.sqrt(var)
    h = torch.log(100 * PS / (X * PT)) / sp + sp / 2

    def cdf(v):
        return 0.5 * torch.erfc(-v / math.sqrt(2.0))

    base = torch.where(t["type"] == 1, X * PT * cdf(sp - h) - 100 * PS * cdf(-h), 100 * PS * cdf(h) - X * PT * cdf(h - sp))
    q = torch.exp(-a * dt)
    Bd = dt * (1 - q ** (t["n"] - t["e"])) / (1 - q)
    c0 = torch.log(100 * PS / PT) - B * sg**2 * (1 - torch.exp(-a * T)) ** 2 / (2 * a * a) - B**2 * sg**2 * var / 2
    ph = 2 * math.pi * (c0 - torch.log(X)) / (Bd * t["dr"])
    feats = torch.stack([(X - 80) / 20, (T - 15.5) / 14.5, (S - T - 5.5) / 4.5, (t["term_steps"] - 24) / 12,
                         (a - 0.105) / 0.095, (sg - 0.0125) / 0.0075, torch.sin(ph), torch.cos(ph)], 1)
    return base, feats


def _ensemble(o, curve, P):
    base, x = _closed_form(o, curve)
    ys = []
    for p in P.astype(np.float64):
        w = {k: torch.as_tensor(p[off:off + int(np.prod(surrogate.SHAPES[k]))].reshape(surrogate.SHAPES[k]), device=x.device)
             for k, off in surrogate.OFFSETS.items()}
        h = x
        for k in "1234":
            h = torch.nn.functional.silu(h @ w["W" + k].T + w["b" + k])
        ys.append((h @ w["W5"].T + w["b5"])[:, 0])
    y = torch.stack(ys)
    return base + 0.01 * y.mean(0), 0.01 * (y.max(0).values - y.min(0).values)


def exact(case, seed):
    n, op = case["n"], case["op"]
    if op == "train":
        return None  # the order of its samples is the library's own random stream
    o, curve = _inputs(case["dist"], n, seed)
    if op == "price_f32":
        c = _shape_f32(o)
        o = {f: v.astype(np.float32) if f in REAL_FIELDS else v for f, v in o.items()}
        curve = (curve[0].astype(np.float32).astype(np.float64), curve[1])
    else:
        c = _shape(o)
    # node updates of one pass in all; beyond this it takes too long
    if op != "surrogate" and float((c["n"] * c["jmax"]).sum()) > 1.2e10:
        return None
    if op != "surrogate":
        return _tree(o, c, curve)
    mean, spread = _ensemble(o, curve, _weights(seed))
    boxed = torch.as_tensor((o["a"] <= 0.2) & (o["length"] <= 30), device=mean.device)
    rest = torch.nonzero(~boxed | (spread > SPREAD_THRESHOLD))[:, 0]
    at = rest.cpu().numpy()
    mean[rest] = _tree({k: v[at] for k, v in o.items()}, {k: v[at] for k, v in c.items()}, curve)
    return mean
