"""FP64 batches of up to 2,048 options and 512 curve points run in one kernel, larger
ones through the general pipeline; both sides of each line against the oracle, with
every kind of option (invalid, too wide, no steps, no exercise, one tree of each way it
can be priced), and their counts as one plan goes from one side to the other."""
import numpy as np
import pytest

from conftest import parity_tol

pytestmark = pytest.mark.gpu


def _batch(pkg, n):
    r = np.random.default_rng(n)
    jmax = r.choice([1, 3, 15, 16, 23, 24, 31, 32, 64, 100, 300, 640], n)
    steps = np.full(n, 12, np.uint16)
    a = -np.log1p(-0.184 / (jmax - 0.5)) * 12
    mat = r.uniform(0.5, 12, n)
    length = r.uniform(0, 1.1, n) * mat
    sigma = r.uniform(0.001, 0.02, n)
    if n >= 16:
        a[3], a[5] = -1.0, 1e-5  # invalid; wider than any form supports
        mat[7] = 0.01            # no steps
        length[9] = 0.0
        # beyond the tridiagonal form's range: long trees of a huge volatility
        a[11::16], steps[11::16], mat[11::16], sigma[11::16] = 0.06, 40, 40.0, 0.35
    return pkg.Options(strike=r.uniform(60, 100, n), maturity=mat, length=length, term_unit=np.full(n, 365, np.uint16),
                       term_steps=steps, a=a, sigma=sigma, type=r.integers(0, 2, n).astype(np.int8))


def _check(pkg, oracle, opts, y, rc, got):
    bad = np.zeros(opts.N, bool)
    if opts.N >= 16:
        bad[[3, 5]] = True
    assert np.isnan(got[bad]).all() and rc == (pkg.capi.HWT_EINVAL if bad.any() else pkg.capi.HWT_OK)
    ref = oracle.price(opts.take(np.nonzero(~bad)[0]), y)
    assert np.all(np.abs(got[~bad] - ref) <= parity_tol(ref))


@pytest.mark.parametrize("n", [1, 63, 2048, 2049])
@pytest.mark.parametrize("points", [1, 512, 513])
def test_both_sides_of_the_line(pkg, oracle, n, points):
    days = np.unique(np.linspace(1, 11000, points).astype(np.int32))
    y = pkg.formats.Yield(0.03 + 0.01 * np.sin(days / 900.0), days)
    opts = _batch(pkg, n)
    _check(pkg, oracle, opts, y, *pkg.capi.price_status(opts, y))


def test_counts_follow_the_last_execution(pkg):
    capi, y = pkg.capi, pkg.datasets.synthetic_yield()
    ok = _batch(pkg, 1).take(np.zeros(3000, int))
    ok.a[:], ok.term_steps[:] = np.linspace(0.02, 0.3, 3000), 36
    dev = capi.to_device(ok, y)
    p = capi.Plan(3000, y.N)
    small = []
    for n in (3000, 100, 3000, 0, 100, 100):
        p.execute(dev, n=n)
        st = p.sync()
        assert st["tasks"] == n and (n == 0) == (st["node_updates"] == 0)
        small += [st] if n == 100 else []
        p.execute(dev, n=n)  # and on a replay
        assert p.sync()["node_updates"] == st["node_updates"]
    for k in ("node_updates", "wide_node_updates", "seq_node_updates", "wide_tasks", "wide_step_ops"):
        assert len({st[k] for st in small}) == 1
    p.close()
