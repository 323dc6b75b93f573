"""The tuner and the reported shapes where the mixed path runs the matrix-core
kernel, which has one form: one target per lane, whatever was recorded."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_one_form(gpu, tmp_path):
    nt, ns = 13001, 12000
    rng = np.random.default_rng(0)
    d = [gpu.DeviceArray.from_host(rng.random(a)) for a in (3 * nt, 3 * ns, ns, nt)]
    gpu.tune_db_path(str(tmp_path / "t.db"))
    try:
        tpl, cap, ms = gpu.tune_eval(0, d[0], d[1], None, d[2], d[3], precision=gpu.MIXED)
        assert tpl == 1 and cap in (0, 3, 2) and ms > 0
        assert gpu.dense_shape(0, nt, ns, precision=gpu.MIXED) == (tpl, cap)
        gpu.set_dense_shape(0, nt, ns, 4, 0, precision=gpu.MIXED)
        assert gpu.DensePlan(0, d[0], d[1], None, precision=gpu.MIXED).shape() == (gpu.MIXED, 1, 0)
        gpu.set_dense_shape(0, 4000, 4000, 4, 0, precision=gpu.MIXED)  # the FP64 kernels: as recorded
        few = [gpu.DeviceArray.from_host(rng.random(12000)) for _ in range(2)]
        assert gpu.DensePlan(0, few[0], few[1], None, precision=gpu.MIXED).shape() == (gpu.MIXED, 4, 0)
    finally:
        gpu.tune_db_path(None)
    assert gpu.dense_shape(0, 1 << 20, 1 << 20, precision=gpu.MIXED) == (1, 0)
