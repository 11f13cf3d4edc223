"""The training kernels at the row counts where their loops end differently: one
split of 16 rows, a half residue block of 256, rounds of four and eight 256s with and
without a rest, and a batch that is no multiple of 1,024.  Gradients against the CPU
reference at the bar of test_gpu_surrogate.py."""
import numpy as np
import pytest

import surrogate_ref as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [128, 256, 640, 1152, 2176, 2432])
def test_gradients_at_odd_batches(pkg, rows):
    y = pkg.datasets.synthetic_yield()
    _, dev, prices = pkg.surrogate.training_set(33, 4096, y)
    s = pkg.surrogate.Surrogate(4096, 256, y.N, pkg.surrogate.config(batch=2432, seed=11))
    s.set_training_data(dev, prices)
    at = (np.arange(rows) * 1021 + 3) % 4096
    _, loss, g_gpu = s.eval_rows(1, at)
    x, t = s.get_inputs(at)
    y_cpu, cache = R.forward_bf16(s.get_params()[1].astype(np.float64), x)
    g_cpu = R.backward(cache, y_cpu.astype(np.float64), t.astype(np.float64))
    assert abs(loss - np.mean((y_cpu - t) ** 2)) <= 1e-3 * max(1e-6, loss)
    for name, o in R.OFF.items():
        size = int(np.prod(R.SHAPE[name]))
        a, b = g_gpu[o:o + size].astype(np.float64), g_cpu[o:o + size]
        assert np.linalg.norm(a - b) <= 1e-2 * np.linalg.norm(b) + 1e-12, (name, np.linalg.norm(a - b))
