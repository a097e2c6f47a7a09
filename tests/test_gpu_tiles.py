"""Tuned tiles change the schedule, not the result: a run made with
LOMA_FLAG_AUTOTUNE ends bit for bit where the same run without it ends, at
lengths of the wavefront-per-row x lines (whose tile the tuner keeps) and of
the run-time plan (every tile the same kernel).  Small grids, where a smaller
tile would fill the chip better and win a timing."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ("vor", "phi", "psi", "scal", "u00", "v00", "w00")


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("mgalx,my,mgalz", [
    (64, 33, 24), (64, 129, 64), (96, 129, 32), (128, 65, 24), (192, 49, 24), (256, 33, 12),
    (384, 17, 12), (512, 33, 12), (100, 65, 24)])
def test_tuned_run_equals_untuned(gpu, mgalx, my, mgalz, precision):
    from loma_phd_amd import capi, ic
    from loma_phd_amd.grid import MixingLayerConfig
    cfg = MixingLayerConfig(mgalx=mgalx, my=my, mgalz=mgalz, s=3.0, Re=200.0, seed=mgalx)
    st = ic.initial_condition(cfg)
    got, tiles = [], []
    for flags in (0, capi.LOMA_FLAG_AUTOTUNE):
        print(f"tiles {mgalx}x{my}x{mgalz} precision={precision} flags={flags}", flush=True)
        run = capi.Run(mgalx, my, mgalz, st["y"], cfg.Re, cfg.alp, cfg.bet, cfg.pr, cfg.cfl,
                       cfg.ncfl, cfg.dt0, precision, flags)
        run.upload(st["vor"], st["phi"], st["psi"], st["scal"], st["u00"], st["v00"], st["w00"])
        run.advance(1)
        got.append(run.download())
        tiles.append(run.tiles())
        run.close()
    print("tiles", tiles, flush=True)
    for f in FIELDS:
        assert np.array_equal(got[0][f], got[1][f]), (f, tiles)
