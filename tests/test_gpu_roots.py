"""The device's FP64 square root and third against IEEE.  The root's last step adds the exactly formed residual over
2 sqrt(a), whose relative error is about 2^-50, so the result is the rounded root or, next to a tie, its neighbour: 1 ulp.
The third is one correction of the product with the correctly rounded 1/3 by the exact residual (Markstein): the IEEE
quotient.  Below about 1e-290 the residuals are no longer exact."""
import numpy as np
import pytest

import cfd_solver_2d_gpu_amd as F

pytestmark = pytest.mark.gpu


def test_roots_and_thirds():
    print("[gpu-case] device FP64 square root and third against IEEE on 2^20 operands", flush=True)
    rng = np.random.default_rng(77)
    n = 1 << 20
    a = 10.0 ** rng.uniform(-290, 300, n)
    a[: n // 2] = 10.0 ** rng.uniform(-12, 12, n // 2)       # densities, pressures, areas
    a[: n // 8] = np.arange(1, n // 8 + 1, dtype=np.float64)  # with the squares among them
    r, t = F.device_roots(a)
    want = np.sqrt(a)
    assert np.all(np.abs(r - want) <= np.spacing(want))
    assert np.array_equal(t, a / 3.0)
    assert np.array_equal(F.device_roots(-a)[1], -a / 3.0)
    k = np.arange(1, 363, dtype=np.float64)
    assert np.array_equal(F.device_roots(k * k)[0], k)       # exact roots stay exact


def test_special_values():
    print("[gpu-case] device FP64 square root of 0, infinity, NaN and negative numbers", flush=True)
    r, t = F.device_roots(np.array([0.0, -0.0, np.inf, np.nan, -1.0, -np.inf]))
    assert r[0] == 0.0 and r[1] == 0.0 and r[2] == np.inf and np.isnan(r[3:]).all()
    assert t[0] == 0.0 and t[1] == 0.0 and np.isnan(t[3])
