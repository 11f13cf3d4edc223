"""Form 1's workgroup size is a matter of scheduling: the same prices to the bit, and the
larger sizes take no longer than twice what 256 does (workgroups of 1,024 left the kernel
too few registers: eleven times as long on this batch)."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_workgroup_sizes_price_alike(pkg):
    capi, n = pkg.capi, 2000
    r = np.random.default_rng(61)
    opts = pkg.Options(strike=r.uniform(60, 100, n), maturity=np.full(n, 9.0), length=np.full(n, 3.0),
                       term_unit=np.full(n, 365, np.uint16), term_steps=np.full(n, 12, np.uint16), a=np.full(n, 0.1),
                       sigma=r.uniform(0.005, 0.02, n), type=r.integers(0, 2, n).astype(np.int8))
    batch = capi.Batch(opts, pkg.datasets.synthetic_yield())
    prices, times = {}, {}
    for size in (64, 256, 320, 512, 1024):
        cfg = capi.config(form=capi.FORM_LANE, block_size=size)
        runs = []
        for _ in range(9):
            t = time.perf_counter()
            prices[size] = batch.price(cfg)
            runs.append(time.perf_counter() - t)
        times[size] = sorted(runs)[4]
    print({k: f"{v * 1e6:.0f} us" for k, v in times.items()})
    for size in prices:
        assert np.array_equal(prices[size], prices[256])
        assert times[size] < 2 * times[256]
