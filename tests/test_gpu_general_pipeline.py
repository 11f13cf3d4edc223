"""What a batch of up to 2,048 options prices in one kernel of its own, through the general
pipeline's k_price_tri as well: every width of the lane groups in the split of batches up
to 16,384 options (four trees of 16 lanes to a wave, whose starts and swaps fall at
different steps), and the windows' kinds from its queue."""
import numpy as np
import pytest

from conftest import parity_tol
from test_gpu_windows import _batch, test_groups_price_every_width as every_width

pytestmark = pytest.mark.gpu


def test_spread_groups_price_every_width(pkg, oracle):
    every_width(pkg, oracle, 6000)


@pytest.mark.parametrize("kind", ["usual", "far_strikes", "volatile", "edges", "degenerate"])
def test_windows_from_the_queue(pkg, oracle, kind):
    y = pkg.datasets.synthetic_yield()
    opts = _batch(pkg, kind)
    n = opts.N
    small = pkg.datasets.skewed(seed=89, n=2400, large_frac=0.0)
    got = pkg.capi.price(pkg.Options.concat([small.take(np.arange(1200)), opts, small.take(np.arange(1200, 2400))]), y)
    ref, got = oracle.price(opts, y), got[1200:1200 + n]
    fin = np.isfinite(ref) & (np.abs(ref) < 1e290)
    tail = fin & (ref > 1e-250)  # below, the oracle's own terms underflow
    assert fin.sum() > n // 2
    assert (np.abs(got[tail] - ref[tail]) / np.abs(ref[tail])).max() <= 1e-10
    assert np.all(np.abs(got[fin] - ref[fin]) <= parity_tol(ref[fin]))
