"""FP64 wide trees price over windows that follow the tree's weight (Reach,
csrc/hwt_wave.h): every price against the oracle's whole tree, in relative
terms, also where the price is itself a far tail.  The bar is the parity bar
without its absolute floor: the oracle rounds each of its up to 2n steps over
positive terms, so a price of any size carries about 2 n 2^-53 < 1e-12."""
import numpy as np
import pytest

from conftest import parity_tol

pytestmark = pytest.mark.gpu


def _batch(pkg, kind, n=96):
    r = np.random.default_rng(17)
    steps = np.full(n, 36, np.uint16)
    a, sigma = r.uniform(0.0098, 0.1, n), r.uniform(0.002, 0.02, n)
    mat = r.uniform(2, 30, n)
    length = r.uniform(0.02, 0.97, n) * mat
    strike = r.uniform(60, 100, n)
    typ = r.integers(0, 2, n).astype(np.int8)
    if kind == "far_strikes":  # prices down to 1e-200, and deep in the money
        strike = np.exp(r.uniform(np.log(5), np.log(400), n))
    elif kind == "volatile":  # the discounted path drifts many nodes down
        sigma = r.uniform(0.03, 0.3, n)
    elif kind == "edges":  # widths around the classes and window sizes
        steps = np.full(n, 12, np.uint16)
        jmax = np.tile([64, 65, 95, 96, 97, 127, 128, 160, 255, 320, 447, 671], n // 12)
        a = -np.log1p(-0.184 / (jmax - 0.5)) * 12
        mat = r.uniform(1, 100, n)
        length = np.where(r.uniform(size=n) < 0.2, 0.01, r.uniform(0, 1, n) * mat)
    elif kind == "degenerate":  # no volatility; strikes without a logarithm; exercise at once
        sigma[::3] = 0.0
        strike[1::3] = np.resize([0.0, -5.0, 1e-300, 1e300], strike[1::3].size)
        length[2::3] = 0.0
    return pkg.Options(strike=strike, maturity=mat, length=length, term_unit=np.full(n, 365, np.uint16),
                       term_steps=steps, a=a, sigma=sigma, type=typ)


@pytest.mark.parametrize("kind", ["usual", "far_strikes", "volatile", "edges", "degenerate"])
def test_windows_price_the_whole_tree(pkg, oracle, kind):
    y = pkg.datasets.synthetic_yield()
    opts = _batch(pkg, kind)
    ref = oracle.price(opts, y)
    got, st = pkg.capi.price(opts, y, stats=True)
    fin = np.isfinite(ref) & (np.abs(ref) < 1e290)
    assert fin.sum() > opts.N // 2 and st["wide_tasks"] > opts.N // 2
    tail = fin & (ref > 1e-250)  # below, the oracle's own terms underflow
    rel = np.abs(got[tail] - ref[tail]) / np.abs(ref[tail])
    print(f"\n{kind}: {tail.sum()} prices from {ref[tail].min():.1e}, max relative error {rel.max():.2e}")
    assert rel.max() <= 1e-10, np.nonzero(rel > 1e-10)[0][:5]
    assert np.all(np.abs(got[fin] - ref[fin]) <= parity_tol(ref[fin]))


@pytest.mark.parametrize("n", [400, 17000], ids=["spread", "packed"])
def test_groups_price_every_width(pkg, oracle, n):
    """Every odd width from 3 to 181 (the lane groups of L = 1 to 16, their
    K = 2 to 11, the first windows beyond), heights from one step to 300 in one
    batch, exercise from step 0 to the last: against the oracle as above.  n
    decides how many lanes a tree gets (TRI_SPREAD)."""
    r = np.random.default_rng(23)
    width = np.resize(np.arange(3, 182, 2), n)
    a = np.where(width == 3, 3.0, -np.log1p(-0.184 / (width // 2 - 0.5)) * 12)
    h = r.integers(1, 301, n)
    h[: width.size // 4] = r.integers(1, 6, width.size // 4)
    e = np.where(r.uniform(size=n) < 0.1, 0, (r.uniform(size=n) * h).astype(int))
    opts = pkg.Options(strike=r.uniform(60, 100, n), maturity=(h + 0.5) / 12, length=(e + 0.5) / 12,
                       term_unit=np.full(n, 365, np.uint16), term_steps=np.full(n, 12, np.uint16), a=a,
                       sigma=r.uniform(0.001, 0.05, n), type=r.integers(0, 2, n).astype(np.int8))
    y = pkg.datasets.synthetic_yield()
    got = pkg.capi.price(opts, y)
    sub = np.arange(0, n, max(1, n // 1500))
    assert {oracle.constants(opts, int(i)).width for i in np.arange(min(n, 90))} == set(range(3, 182, 2))
    ref = oracle.price(opts.take(sub), y)
    tail = ref > 1e-250
    rel = np.abs(got[sub][tail] - ref[tail]) / ref[tail]
    assert rel.max() <= 1e-10, (width[sub][tail][rel.argmax()], rel.max())
    assert np.all(np.abs(got[sub] - ref) <= parity_tol(ref))


@pytest.mark.parametrize("block", [0, 512])
def test_lane_form_sweeps(pkg, oracle, block):
    """Form 1 steps its columns several steps to a sweep: every count of steps
    from 0 to 40 in both passes, columns narrower and wider than a chunk, both
    workgroup sizes' kernels, and trees that leave the tridiagonal form."""
    h, e = np.meshgrid(np.arange(1, 42), np.arange(0, 41))
    h, e = h[e < h], e[e < h]
    n = h.size
    r = np.random.default_rng(29)
    width = np.resize([3, 5, 7, 9, 15, 17, 19, 25, 47, 61, 127], n)
    a = np.where(width == 3, 3.0, -np.log1p(-0.184 / (width // 2 - 0.5)) * 12)
    sigma = np.where(np.arange(n) % 9 == 0, 4.0, r.uniform(0.001, 0.05, n))
    opts = pkg.Options(strike=r.uniform(60, 100, n), maturity=(h + 0.5) / 12, length=(e + 0.5) / 12,
                       term_unit=np.full(n, 365, np.uint16), term_steps=np.full(n, 12, np.uint16), a=a, sigma=sigma,
                       type=r.integers(0, 2, n).astype(np.int8))
    y = pkg.datasets.synthetic_yield()
    got = pkg.capi.price(opts, y, pkg.capi.config(form=pkg.capi.FORM_LANE, block_size=block))
    ref = oracle.price(opts, y)
    assert np.all(np.abs(got - ref) <= parity_tol(ref)), np.nonzero(~(np.abs(got - ref) <= parity_tol(ref)))[0][:5]
