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
