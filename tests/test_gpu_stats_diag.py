"""The rho uu, rho vv and rho ww columns of the statistics window carry the
rounding of their own product, however large the other two are.

Short waves under a wide envelope: rho v of order one, rho u and rho w smaller
by the ratio of the wavelength to the envelope (below 1e-2), so that rho uu and
rho ww are below 1e-4 of rho vv.  A mixed run's columns agree with the FP64
run's within the 1e-5 of test_gpu_stats.py, each relative to its own norm: FP32
transforms carry rho u and rho w to some 1e-6 of themselves, and the products
and their sums add a few 6e-8.  (A sum of the transforms of rho uu - rho vv and
rho vv has the rounding of rho vv.)  Lengths of the wavefront-per-row x lines
and of the run-time plan."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mgalx", [64, 48, 192])
def test_diagonal_products(gpu, mgalx):
    from loma_phd_amd import capi, grid
    from loma_phd_amd.stats import STA_COLUMNS
    my, mgalz, k0 = 129, 48, 4.0
    y = grid.tanh_mesh(my, 20.0)
    cols = {}
    for precision in (0, 1):
        print(f"diagonal products n={mgalx} precision={precision}", flush=True)
        run = capi.Run(mgalx, my, mgalz, y, 1e4, k0, k0, precision=precision)
        rng = np.random.default_rng(mgalx)
        n, mz, _ = run.shape()
        amp = (rng.standard_normal((n, mz)) + 1j * rng.standard_normal((n, mz))) * 0.02
        amp[0] = 0.0  # kx > 0 planes only: the others are their conjugates
        kx = k0 * np.arange(n)[:, None]
        kz = k0 * np.r_[np.arange(run.nz + 1), np.arange(-run.nz, 0)][None, :]
        rK = kx**2 + kz**2
        w = 8.0
        v = np.exp(-((y / w) ** 2))
        d2v = (4.0 * y**2 / w**4 - 2.0 / w**2) * v
        phi = amp[:, :, None] * (d2v[None, None] - rK[:, :, None] * v[None, None])
        zero = np.zeros(run.shape(), np.complex128)
        scal = zero.copy()
        scal[0, 0] = 1.0
        run.upload(zero, phi, zero, scal, np.zeros(my), np.zeros(my), np.zeros(my))
        run.stats_config([my // 2])
        run.stats_accumulate(True)
        run.advance(1)
        cols[precision] = run.stats_read()["sta"]
        run.close()
    c = {k: STA_COLUMNS.index(k) for k in ("ruu", "rvv", "rww")}
    norm = {k: np.linalg.norm(cols[0][:, q]) for k, q in c.items()}
    assert max(norm["ruu"], norm["rww"]) < 1e-3 * norm["rvv"], norm
    for k, q in c.items():
        err = np.linalg.norm(cols[1][:, q] - cols[0][:, q]) / norm[k]
        print(f"{k}: norm {norm[k]:.3e} error {err:.2e}", flush=True)
        assert err <= 1e-5, (k, err)
