"""The fused reductions that the row kernel's last workgroup finishes, at the
edges of its counting: one workgroup, 15 to 17 (the counters' 16 lines), 1024
(the last size it is used for) and 1025 (a launch of its own). Every launch
gives the same bits, so the counters are back at zero, and r.r agrees with
numpy's FP64 sum to the pair's 48 bits plus the rounding of n FP64 additions."""
import numpy as np
import pytest

import kutta_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 255, 256, 257, 15 * 256, 16 * 256, 16 * 256 + 1, 17 * 256, 1023 * 256 + 7,
                               1024 * 256, 1024 * 256 + 1])
def test_last_workgroup_finishes(device, n):
    rng = np.random.default_rng(n)
    p, q, r0 = (rng.standard_normal(n).astype(np.float32) for _ in range(3))
    alpha = np.float32(0.375)
    scalars0 = np.zeros(24, np.float32)
    scalars0[8] = alpha
    scalars0[22] = np.float32(3e38)
    dp, dq = device.upload(p), device.upload(q)
    want = r0 - alpha * q
    exact = float(np.sum(want.astype(np.float64) ** 2))
    seen = set()
    for _ in range(4):
        x, r = device.upload(np.zeros(n, np.float32)), device.upload(r0)
        scalars, status = device.upload(scalars0), device.upload(np.zeros(3, np.int32), np.int32)
        device.launch(kutta_amd.Kernel.fused_step_dot_check, n, x, r, dp, dq, scalars, status)
        s = scalars.download()
        assert np.array_equal(r.download(), want)
        assert list(status.download()) == [0, 1, 0]
        assert abs(float(s[18]) + float(s[19]) - exact) <= (2.0 ** -46 + n * 2.0 ** -53) * exact
        seen.add(s[18:20].tobytes())
    assert len(seen) == 1
