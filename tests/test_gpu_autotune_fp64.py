"""hwt_autotune in FP64 tries what FP64 pricing depends on: the four switches between
mixed mode's kernel arrangements are no candidates there and come back as given."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("given", [0, 2])
def test_fp64_leaves_the_arrangements_alone(pkg, given):
    capi, y = pkg.capi, pkg.datasets.synthetic_yield()
    dev = capi.to_device(pkg.datasets.skewed(seed=59 + given, n=9000 << (given // 2)), y)
    arrangements = capi.FLAG_NO_ROWS | capi.FLAG_NO_FLAT | capi.FLAG_CONCURRENT | capi.FLAG_FUSED
    cfg, rep = capi.autotune(dev, capi.config(flags=given))
    assert rep["cached"] == 0
    # the start, 2 orders, the launch mode, 2 + 2 grids, form 1, and at most two timed again
    assert rep["candidates"] <= 1 + 2 + 1 + 4 + 1 + 2
    assert cfg.flags & arrangements == given & arrangements
    again, rep2 = capi.autotune(dev, capi.config(flags=given))
    assert rep2["cached"] == 1 and again.as_dict() == cfg.as_dict()
