"""Wide trees of a few steps whose rates lie far apart: the nodes a price depends on are
close to the root, the discounts of the windows' other nodes leave FP64's range."""
import numpy as np
import pytest

from conftest import parity_tol

pytestmark = pytest.mark.gpu


def _options(pkg, seed, n, h, heights):
    """Yearly steps; h is the rate spacing times the step, drawn between the given bounds."""
    r = np.random.default_rng(seed)
    jmax = r.integers(33, 346, n)
    a = -np.log1p(-0.184 / (jmax - 0.5))
    height = r.integers(heights[0], heights[1] + 1, n)
    e = (r.uniform(size=n) * height).astype(int)
    sigma = np.exp(r.uniform(*np.log(h), n)) / np.sqrt(3 * -np.expm1(-2 * a) / (2 * a))
    return pkg.Options(strike=np.exp(r.uniform(0, np.log(400), n)), maturity=height + 0.5, length=e + 0.5,
                       term_unit=np.full(n, 365, np.uint16), term_steps=np.ones(n, np.uint16), a=a, sigma=sigma,
                       type=r.integers(0, 2, n).astype(np.int8))


def _check(pkg, oracle, opts):
    y = pkg.datasets.synthetic_yield()
    ref = oracle.price(opts, y)
    fin = np.isfinite(ref)
    assert fin.mean() > 0.9
    for n in (opts.N, 600):  # through the general pipeline, and the kernel for small batches
        got = pkg.capi.price(opts.take(np.arange(n)), y)
        bad = np.nonzero(fin[:n] & ~(np.abs(got - ref[:n]) <= parity_tol(ref[:n])))[0]
        assert bad.size == 0, (bad.size, bad[:4], got[bad[:4]], ref[bad[:4]])


def test_windows_within_the_scales_range(pkg, oracle):
    _check(pkg, oracle, _options(pkg, 67, 2500, (0.02, 0.5), (1, 3)))


def test_discounts_out_of_range_beside_the_root(pkg, oracle):
    """One step, rate spacing times step up to 5,000: the root's own discount is 1, its
    neighbours' may overflow and underflow."""
    _check(pkg, oracle, _options(pkg, 71, 2500, (20.0, 5000.0), (1, 1)))


@pytest.mark.parametrize("n", [2500, 600])
def test_states_beyond_the_range(pkg, oracle, n):
    """Volatilities at which a tree's undiscounted states, or their products, exceed 1e308
    (n h jmax up to 900): out of the tridiagonal form's range, priced by the general
    kernel.  The bar as for tall trees: the steps' own rounding on top of the parity bar."""
    r = np.random.default_rng(73)
    jmax = r.integers(1, 86, n)
    a = np.where(jmax == 1, 0.9, -np.log1p(-0.184 / (jmax - 0.5)))
    height = r.integers(300, 3000, n)
    h = r.uniform(310, 900, n) / (height * jmax)
    opts = pkg.Options(strike=np.exp(r.uniform(0, np.log(400), n)), maturity=height + 0.5,
                       length=(r.uniform(size=n) * height).astype(int) + 0.5, term_unit=np.full(n, 365, np.uint16),
                       term_steps=np.ones(n, np.uint16), a=a, sigma=h / np.sqrt(3 * -np.expm1(-2 * a) / (2 * a)),
                       type=r.integers(0, 2, n).astype(np.int8))
    days = np.array([365, 365000], np.int32)
    y = pkg.formats.Yield(np.array([0.001, 0.0012]), days)  # bonds of thousands of years worth something
    ref = oracle.price(opts, y)
    fin = np.isfinite(ref)
    assert fin.mean() > 0.9
    got = pkg.capi.price(opts, y)
    tol = parity_tol(ref) + 100 * 8 * height * 2.0**-53
    bad = np.nonzero(fin & ~(np.abs(got - ref) <= tol))[0]
    assert bad.size == 0, (bad.size, bad[:4], got[bad[:4]], ref[bad[:4]])


@pytest.mark.parametrize("n", [300, 3000, 17000])
def test_bonds_of_any_finite_price(pkg, oracle, n):
    """Thousands of years at -4%: bonds worth up to 1e300, puts on them nothing."""
    r = np.random.default_rng(79)
    jmax = np.resize(np.r_[np.arange(2, 60), 88, 90, 150], n)
    height = r.integers(13000, 17001, n)
    opts = pkg.Options(strike=r.uniform(60, 100, n), maturity=height + 0.5, length=r.integers(0, 200, n) + 0.5,
                       term_unit=np.full(n, 365, np.uint16), term_steps=np.ones(n, np.uint16),
                       a=-np.log1p(-0.184 / (jmax - 0.5)), sigma=r.uniform(1e-5, 1e-4, n),
                       type=r.integers(0, 2, n).astype(np.int8))
    y = pkg.formats.Yield(np.array([-0.04, -0.04]), np.array([1, 2], np.int32))
    some = np.arange(0, n, n // 30)
    ref, got = oracle.price(opts.take(some), y), pkg.capi.price(opts, y)
    assert np.isfinite(ref).all() and ref.max() > 1e270 and (ref[opts.type[some] == 1] == 0).all()
    # relative: the oracle rounds each of its 2 x 17,000 steps
    assert np.all(np.abs(got[some] - ref) <= 1e-10 * ref), (got[some][:5], ref[:5])
    assert np.isfinite(got).all() and (got[opts.type == 1] == 0).all()


def test_states_beyond_any_start_are_no_number(pkg, oracle):
    """n h jmax from 1,300 to 4,000: where a state leaves the range the price is right or
    NaN, never a wrong number."""
    n = 2500
    r = np.random.default_rng(83)
    jmax = r.integers(1, 400, n)
    a = np.where(jmax == 1, 0.9, -np.log1p(-0.184 / (np.maximum(jmax, 2) - 0.5)))
    height = r.integers(600, 3000, n)
    h = r.uniform(1300, 4000, n) / (height * jmax)
    opts = pkg.Options(strike=np.exp(r.uniform(0, np.log(100), n)), maturity=height + 0.5,
                       length=(r.uniform(size=n) * height).astype(int) + 0.5, term_unit=np.full(n, 365, np.uint16),
                       term_steps=np.ones(n, np.uint16), a=a, sigma=h / np.sqrt(3 * -np.expm1(-2 * a) / (2 * a)),
                       type=r.integers(0, 2, n).astype(np.int8))
    y = pkg.formats.Yield(np.array([0.001, 0.0012]), np.array([365, 365000], np.int32))
    ref, got = oracle.price(opts, y), pkg.capi.price(opts, y)
    fin = np.isfinite(ref) & ~np.isnan(got)
    tol = parity_tol(ref) + 100 * 8 * height * 2.0**-53
    print(f"\n{np.isnan(got).sum()} NaN, {fin.sum()} to compare")
    bad = np.nonzero(fin & ~(np.abs(got - ref) <= tol))[0]
    assert bad.size == 0, (bad.size, bad[:4], got[bad[:4]], ref[bad[:4]])


@pytest.mark.parametrize("n", [300, 3000, 17000])
def test_puts_on_bonds_beyond_the_range(pkg, n):
    """18,000 to 30,000 years at -4%: the bond is worth more than 1e308, a put on it
    nothing, in groups and windows with and without padding nodes.  (The oracle steps
    through infinite bond values and has no number here.)"""
    r = np.random.default_rng(97)
    jmax = np.resize(np.r_[np.arange(1, 60), 88, 90, 150], n)
    opts = pkg.Options(strike=r.uniform(60, 100, n), maturity=r.integers(18000, 30001, n) + 0.5,
                       length=r.integers(0, 200, n) + 0.5, term_unit=np.full(n, 365, np.uint16),
                       term_steps=np.ones(n, np.uint16), sigma=r.uniform(1e-5, 1e-4, n), type=np.ones(n, np.int8),
                       a=np.where(jmax == 1, 0.9, -np.log1p(-0.184 / (np.maximum(jmax, 2) - 0.5))))
    got = pkg.capi.price(opts, pkg.formats.Yield(np.array([-0.04, -0.04]), np.array([1, 2], np.int32)))
    assert (got == 0).all(), (np.isnan(got).sum(), got[got != 0][:5])
