"""hwt_plan_sync reports an execution's counts as often as it is asked, on both sides of
the line between one-kernel batches and the general pipeline."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

COUNTS = ("node_updates", "wide_node_updates", "seq_node_updates", "tasks", "wide_tasks", "wide_step_ops",
          "wide_unit_slots", "wide_plain_slots", "unsupported")


@pytest.mark.parametrize("n", [100, 2048, 2049])
def test_a_second_sync_reports_the_same(pkg, n):
    capi, y = pkg.capi, pkg.datasets.synthetic_yield()
    opts = pkg.datasets.skewed(seed=53, n=n)
    dev = capi.to_device(opts, y)
    plan = capi.Plan(n, y.N)
    for _ in range(2):  # captured, then replayed
        plan.execute(dev)
        first, again = plan.sync(), plan.sync()
        assert first["tasks"] == n and first["wide_step_ops"] > 0
        assert {k: again[k] for k in COUNTS} == {k: first[k] for k in COUNTS}
    # no execution of this plan's before its sync: a smaller batch, then a status alone
    plan.execute(dev, n=n // 2)
    plan.sync()
    assert plan.sync()["tasks"] == n // 2
    plan.close()
