"""One-shot calls take their plan and buffers from a pool of idle workspaces: each
call's prices are those of a batch uploaded and priced by itself, bit for bit, from
several threads at once, as sizes and settings change, and after hwt_trim."""
import math
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = (1, 5, 1023, 1024, 1025, 7000)


def book(pkg, n, seed):
    r = np.random.default_rng(seed)
    length = r.choice([1.0, 2.0, 3.0], n)
    return pkg.Options(strike=r.uniform(30, 90, n), maturity=length + r.choice([1.0, 4.0], n), length=length,
                       term_unit=np.full(n, 365, np.uint16), term_steps=r.integers(5, 40, n).astype(np.uint16),
                       a=r.uniform(0.02, 0.2, n), sigma=r.uniform(0.005, 0.02, n),
                       type=r.integers(0, 2, n).astype(np.int8))


def curve(pkg, golden_yield, points):
    days = np.linspace(1, 12000, points).astype(np.int32)
    return pkg.formats.Yield(np.interp(days, golden_yield.days, golden_yield.rates), days)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_threads_sizes_and_trim(pkg, golden_yield, precision):
    capi = pkg.capi
    prec = {"fp64": capi.PREC_FP64, "mixed": capi.PREC_MIXED}[precision]
    cfg, other = capi.config(precision=prec), capi.config(precision=prec, flags=capi.FLAG_NO_FLAT)
    jobs = []
    for k, n in enumerate(SIZES):
        o, y = book(pkg, n, k), curve(pkg, golden_yield, 3 + 300 * (k % 2))
        b = capi.Batch(o, y)
        jobs.append((o, y, b.price(cfg), b.price(other)))
        b.close()
    bad = []

    def worker(first):
        for i in range(2 * len(jobs)):
            o, y, want, flat = jobs[(first + i) % len(jobs)]
            if not np.array_equal(capi.price(o, y, cfg), want) or not np.array_equal(capi.price(o, y, other), flat):
                bad.append(o.N)
            if i == 3:
                capi.trim()

    ts = [threading.Thread(target=worker, args=(k,)) for k in range(6)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert bad == []
    got, st = capi.price(*jobs[2][:2], cfg, stats=True)
    assert np.array_equal(got, jobs[2][2]) and st["tasks"] > 0 and st["kernel_ms"] > 0


def test_an_invalid_option_leaves_the_others(pkg, golden_yield):
    capi = pkg.capi
    o = book(pkg, 9, 1)
    want = capi.price(o, golden_yield)
    o.a[4] = -1.0
    rc, got = capi.price_status(o, golden_yield)
    keep = np.arange(9) != 4
    assert rc == capi.HWT_EINVAL and np.isnan(got[4]) and np.array_equal(got[keep], want[keep])
    o.a[4] = 0.1
    rc, got = capi.price_status(o, golden_yield)
    assert rc == capi.HWT_OK and np.array_equal(got[keep], want[keep])


def test_float_constants_as_the_c_library_has_them(pkg, golden_yield):
    """hwt_price_f32 derives its constants on the device; priced from constants
    derived here (math.exp and math.sqrt are the C library's) every price is the
    same.  Reversions from 1e-3 to 2 (trees to 1,343 nodes) and steps of a day to a
    year, volatility 0 and 300%, an expiry beyond the tree."""
    capi, f = pkg.capi, np.float32
    n = 3000
    r = np.random.default_rng(5)
    steps = r.choice([1, 2, 12, 52, 365], n).astype(np.uint16)
    a = np.maximum(np.exp(r.uniform(np.log(1e-3), np.log(2.0), n)), 3.0e-4 * steps)
    mat = np.where(steps > 52, r.uniform(0.1, 2, n), r.uniform(1, 20, n))
    o = pkg.Options(strike=r.uniform(30, 90, n), maturity=mat, length=mat * r.uniform(0.01, 1.1, n),
                    term_unit=np.full(n, 365, np.uint16), term_steps=steps, a=a,
                    sigma=r.choice([0.0, 0.003, 0.02, 3.0], n, p=[.05, .5, .4, .05]),
                    type=r.integers(0, 2, n).astype(np.int8))
    ks = (capi.ConstantsF32C * n)()
    for i in range(n):
        af, sg, nf = f(o.a[i]), f(o.sigma[i]), f(int(steps[i])) * f(o.maturity[i])
        dt = f(1) / f(steps[i])
        v = float(sg * sg) * (1.0 - math.exp(float(f(-2) * af * dt))) / float(f(2) * af)
        m = f(math.exp(float(-af * dt)) - 1.0)
        jmax = int(f(-0.184) / m) + 1
        ks[i] = capi.ConstantsF32C(f(o.length[i]), dt, f(math.sqrt(3.0 * v)), f(o.strike[i]), m, jmax, int(nf),
                                   2 * jmax + 1, 365, int(o.type[i]))
    assert max(k.width for k in ks) > 1000
    assert np.array_equal(capi.price_f32(o, golden_yield), capi.price_constants_f32(ks, golden_yield), equal_nan=True)
