"""The counters that the bench line's roofline divides by a measured time were taken from
the kernel that is in the tree."""
import importlib.util
import json

from conftest import ROOT


def test_counters_belong_to_the_kernel_sources():
    spec = importlib.util.spec_from_file_location("bench", ROOT / "bench.py")
    bench = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(bench)
    counted = json.loads(bench.COUNTERS.read_text())
    assert counted["sources_sha"] == bench.counted_sources_sha(), "profile k_price_tri again (profiles/)"
    fma, mul, add = (counted[f"instructions_{k}_f64"] for k in ("fma", "mul", "add"))
    assert counted["fp64_flop_per_launch"] == 64 * (2 * fma + mul + add)
    assert counted["hbm_bytes_per_launch"] == counted["fetch_bytes"] + counted["write_bytes"]
