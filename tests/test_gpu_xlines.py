"""The x-line row kernel at every length it serves, against the FP64 oracle.

One RK3 step at grids whose y sizes leave a remainder in the x-line tile (the
last tile holds one line, an odd number of lines, or all of them), with and
without the passive scalar, in both forms.  The bars are those of the step
tests: 1e-10 per field in FP64 (orders of operations differ), 1e-5 per
physical field in the mixed form (FP32 transforms).
"""
import pytest

from test_gpu_step import _cfg, _compare, _setup

pytestmark = pytest.mark.gpu

# (x points, y points): 64-point tiles hold 32 lines, 512-point ones 4 or 8
SIZES = [(64, 33), (64, 64), (96, 47), (128, 65), (192, 33), (256, 41), (384, 49), (512, 35),
         (100, 37)]


@pytest.mark.parametrize("z", [False, True])
@pytest.mark.parametrize("n,my", SIZES)
def test_step_fp64(gpu, oracle_mod, n, my, z):
    from loma_phd_amd import capi
    run, S, g = _setup(_cfg(n, my, 24, Re=160.0, s=2.0, seed=n), capi.LOMA_FP64, z)
    run.advance(1)
    assert S.step(1) == 0
    _compare(run, S, 1e-10, f"fp64 {n}x{my} z={z}")


@pytest.mark.parametrize("z", [False, True])
@pytest.mark.parametrize("n,my", SIZES)
def test_step_mixed(gpu, oracle_mod, n, my, z):
    from loma_phd_amd import capi, diagnostics, ic
    cfg = _cfg(n, my, 24, Re=160.0, s=2.0, seed=n)
    run, S, g = _setup(cfg, capi.LOMA_MIXED, z)
    run.advance(1)
    assert S.step(1) == 0
    errs = diagnostics.field_errors(run.download(), S.get(), ic.HostOps(cfg.y()), cfg.alp, cfg.bet)
    print(f"mixed {n}x{my} z={z}", errs, flush=True)
    for f, e in errs.items():
        assert e < 1e-5, (f, e)
