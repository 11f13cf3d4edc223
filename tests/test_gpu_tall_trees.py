"""FP64 trees of many steps, exercised anywhere in them: a state grows about sixfold a
step in the tridiagonal form and is scaled back on the way (csrc/hwt_scale.h), in step
with its growth however the passes are cut into pieces.

Bar: the parity bar, plus what the steps' own rounding may add up to: of each of an
option's n steps the oracle's and the pricer's few roundings, 8 x 2^-53 of the
notional of 100."""
import numpy as np
import pytest

from conftest import parity_tol

pytestmark = pytest.mark.gpu


def _options(pkg, seed, n, widths, steps, years):
    r = np.random.default_rng(seed)
    steps = np.resize(np.asarray(steps), n)
    a = -np.log1p(-0.184 / (r.choice(np.asarray(widths) // 2, n) - 0.5)) * steps
    mat = r.uniform(*years, n)
    return pkg.Options(strike=r.uniform(20, 100, n), maturity=mat, length=r.uniform(0, 1, n) * mat,
                       term_unit=np.full(n, 365, np.uint16), term_steps=steps.astype(np.uint16), a=a,
                       sigma=r.uniform(0.005, 0.02, n), type=r.integers(0, 2, n).astype(np.int8))


def _tol(opts, ref):
    height = opts.term_steps * opts.maturity
    return parity_tol(ref) + 100 * 8 * height * 2.0**-53


def _check(oracle, opts, y, got, sub=slice(None)):
    assert np.isfinite(got).all()
    o = opts.take(np.arange(opts.N)[sub])
    ref = oracle.price(o, y)
    err = np.abs(got[sub] - ref)
    bad = np.nonzero(~(err <= _tol(o, ref)))[0]
    assert bad.size == 0, f"{bad.size} of {o.N}: got {got[sub][bad[:4]]}, want {ref[bad[:4]]}"


GROUPS = np.arange(7, 176, 2)


@pytest.mark.parametrize("steps, years", [(36, (20, 60)), (52, (20, 60)), (52, (28, 30))])
def test_tall_groups(pkg, oracle, steps, years):
    """More than 16,384 options (trees packed into as few lanes as hold them), then the
    same in two calls (16 lanes each up to 64 nodes, a wave above): both against the
    oracle on a sample, and against each other on every option."""
    y = pkg.datasets.synthetic_yield()
    opts = _options(pkg, 31, 20000, GROUPS, steps, years)
    packed = pkg.capi.price(opts, y)
    spread = np.concatenate([pkg.capi.price(opts.take(np.arange(k, k + 10000)), y) for k in (0, 10000)])
    _check(oracle, opts, y, packed, slice(0, None, 16))
    _check(oracle, opts, y, spread, slice(7, None, 16))
    assert np.all(np.abs(packed - spread) <= _tol(opts, packed))


def _filler(pkg, n):
    return _options(pkg, 37, n, [25], [12], (1, 2))


@pytest.mark.parametrize("kernel", ["small", "tri"])
@pytest.mark.parametrize("steps", [252, 365])
def test_tall_windows(pkg, oracle, kernel, steps):
    """Daily steps over up to 60 years, in windows: as a batch of 128 (k_price_small) and
    as part of one of more than 2,048 (k_price_tri's window queue)."""
    y = pkg.datasets.synthetic_yield()
    opts = _options(pkg, 41, 128, np.arange(177, 1344, 2), steps, (5, 60))
    if kernel == "small":
        _check(oracle, opts, y, pkg.capi.price(opts, y))
    else:
        got = pkg.capi.price(pkg.Options.concat([_filler(pkg, 1100), opts, _filler(pkg, 1100)]), y)
        _check(oracle, opts, y, got[1100:1228])


@pytest.mark.parametrize("kernel", ["small", "tri"])
def test_hundreds_of_thousands_of_steps(pkg, oracle, kernel):
    """The scaling follows log2 6 bits a step: at 165 for every 64 the 0.44 left over
    would reach 2^1024 at 150,000 steps."""
    y = pkg.datasets.synthetic_yield()
    opts = _options(pkg, 43, 24, [3, 7, 25, 61, 91, 175, 401], 7300, (22, 45))
    if kernel == "small":
        _check(oracle, opts, y, pkg.capi.price(opts, y))
    else:
        got = pkg.capi.price(pkg.Options.concat([_filler(pkg, 1100), opts, _filler(pkg, 1100)]), y)
        _check(oracle, opts, y, got[1100:1124])


@pytest.mark.parametrize("block", [0, 512])
@pytest.mark.parametrize("widths, steps, years", [(np.arange(7, 272, 2), 365, (25, 60)), ([25], 7300, (22, 30))])
def test_tall_columns(pkg, oracle, block, widths, steps, years):
    """Form 1, several steps to a sweep: above and below the 12,050 steps at which scaling
    by 2^-20 for eight of them would lose the range."""
    y = pkg.datasets.synthetic_yield()
    opts = _options(pkg, 47, 64, widths, steps, years)
    cfg = pkg.capi.config(form=pkg.capi.FORM_LANE, block_size=block)
    _check(oracle, opts, y, pkg.capi.price(opts, y, cfg))
