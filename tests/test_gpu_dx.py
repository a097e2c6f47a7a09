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


# rms error in eps of an FP32 transform with passes of radix 8 first and every
# twiddle power from the first by recursion (the larger of the two directions,
# from a model of the passes with random rows against extended precision)
RMS = {64: 1.06, 96: 0.78, 128: 1.08, 192: 1.05, 256: 1.02, 384: 1.12, 512: 1.40}


@pytest.mark.parametrize("mgalx", sorted(RMS))
def test_row_transform_error(gpu, mgalx):
    """The same product with every x mode in T: one substep's increment goes
    through an inverse and a forward x transform of the mixed form and two
    roundings (each eps / sqrt(12) rms).  Its rms error against the FP64 run
    stays below that of two such transforms as RMS lists."""
    from loma_phd_amd import capi, grid
    my, mgalz = 129, 8
    y = grid.tanh_mesh(my, 20.0)
    rng = np.random.default_rng(mgalx)
    inc = []
    for precision in (0, 1):
        print(f"row transform n={mgalx} precision={precision}", flush=True)
        run = capi.Run(mgalx, my, mgalz, y, 1e12, 0.25, 0.25, precision=precision)
        zero = np.zeros(run.shape(), np.complex128)
        scal = zero.copy()
        scal[0, 0] = 1.0
        if precision == 0:
            c = rng.standard_normal((run.nplanes - 1, my, 2)) * 1e-4
            c[:, :1] = c[:, -1:] = 0.0
            c /= np.arange(1, run.nplanes)[:, None, None]  # dT/dx is white
            c = c.astype(np.float32).astype(np.float64)
        scal[1:, 0] = c[..., 0] + 1j * c[..., 1]
        run.upload(zero, zero, zero, scal, np.full(my, 0.5), np.zeros(my), np.zeros(my))
        run.substep(1)
        inc.append((run.download()["scal"] - scal)[1:, 0, 4:-4])
        run.close()
    err = np.linalg.norm(inc[1] - inc[0]) / np.linalg.norm(inc[0]) / 2.0**-23
    bar = np.sqrt(2.0 * RMS[mgalx] ** 2 + 2.0 / 12.0)
    print(f"row transform n={mgalx}: rms error {err:.3f} eps, bar {bar:.3f}", flush=True)
    assert err <= bar
