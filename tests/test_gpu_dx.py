"""dT/dx of the mixed form carries two FP32 roundings, no more.

T = 1 + sum_y of one mode at a quarter of the x length, with FP32-exact real
coefficients c(y); rho u = 1/2, everything else zero and Re so large that
lap T / Pe is below a rounding.  Where the x transforms start with a radix-8
pass and are powers of two (a quarter of the length is then a whole number of
that pass's strides), every pass only adds equal or opposite numbers or
multiplies by powers of i: the transforms are exact, and one substep's
increment of T is
-dtgamma/2 ikx c(y) with two roundings: that of ikx c to FP32 as it enters the
x lines and that of the increment as it leaves them.  Against the FP64 run's
increment the relative error is at most 2 * 2^-24, over the rows and over
alpha whose multiples have long mantissas (rounding kx on its own made three).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mgalx", [64, 512, 32])  # the last: the run-time plan
def test_dx_rounding(gpu, mgalx):
    from loma_phd_amd import capi, grid
    my, mgalz = 129, 8
    i0 = mgalx // 4
    y = grid.tanh_mesh(my, 20.0)
    rng = np.random.default_rng(mgalx)
    worst = 0.0
    for alp in (0.1234567891, 0.2718281828, 0.3141592653, 0.7071067811):
        c = rng.uniform(1e-3, 2e-3, my).astype(np.float32).astype(np.float64)
        inc = []
        for precision in (0, 1):
            print(f"dx n={mgalx} alp={alp} precision={precision}", flush=True)
            run = capi.Run(mgalx, my, mgalz, y, 1e12, alp, 0.25, precision=precision)
            zero = np.zeros(run.shape(), np.complex128)
            scal = zero.copy()
            scal[0, 0] = 1.0
            scal[i0, 0, 1:-1] = c[1:-1]
            run.upload(zero, zero, zero, scal, np.full(my, 0.5), np.zeros(my), np.zeros(my))
            before = run.download()["scal"]
            run.substep(1)
            inc.append(run.download()["scal"][i0, 0] - before[i0, 0])
            run.close()
        a, b = inc[1].imag[4:-4], inc[0].imag[4:-4]
        assert np.abs(b).min() > 0.0
        worst = max(worst, float(np.max(np.abs(a / b - 1.0))))
    print(f"dx n={mgalx}: largest relative error {worst / 2.0**-24:.3f} x 2^-24", flush=True)
    assert worst <= 2.0 * 2.0**-24 * (1.0 + 1e-3)
