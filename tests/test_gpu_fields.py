"""The transform fields of a step against those of foup2 and of a statistics step.

A step derives dT/dx in the x lines and transforms ruu - rvv and rww - rvv;
foup2 takes dT/dx as given and returns the nine products; a statistics step
transforms rvv beside the step's fields.  Row-kernel lengths (64: no first
radix, 96: six entries a lane, 512: eight rows) and run-time lengths, with
the bars of test_gpu_foup2.py (2e-6, FP32 storage) and test_gpu_stats.py.
"""
import ctypes

import numpy as np
import pytest

from conftest import rel_l2
from test_gpu_foup2 import _dp, _fp, _inputs, _ref_layout
from test_gpu_stats import _cfg, _check, _gpu_windows, _oracle_windows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [64, 96, 512])
def test_foup2_row_lengths(gpu, oracle_mod, n):
    from loma_phd_amd import capi
    from loma_phd_amd.grid import MixingLayerConfig
    print(f"foup2 {n}", flush=True)
    cfg = MixingLayerConfig(mgalx=n, my=35, mgalz=24, Re=300.0, s=3.0, seed=2, scalar_z=False)
    g = oracle_mod.Grid(n, cfg.my, cfg.mgalz, cfg.y(), cfg.Re, cfg.alp, cfg.bet, cfg.pr)
    rng = np.random.default_rng(n)
    ins = np.stack([_ref_layout(f, cfg.mgalz) for f in _inputs(g, rng, cfg)])
    ins[4] *= 1.5  # dT/dx is foup2's own input, not taken from T
    rhst = 1e-3 * rng.standard_normal((cfg.my, cfg.mgalz, n))
    S = oracle_mod.State(g, dt0=0.0123, cfl=cfg.cfl, ncfl=1, flags=0)
    S.set_rhst(rhst)
    want, _ = S.foup2(ins[:, :, :g.mz].astype(np.complex128), 1, 0.0123)
    run = capi.Run(n, cfg.my, cfg.mgalz, cfg.y(), cfg.Re, cfg.alp, cfg.bet, cfg.pr, cfg.cfl, 1,
                   0.0123, capi.LOMA_FP64, 0)
    up1, up2, up3, lap, tx, ty, tz, t = [np.ascontiguousarray(a) for a in ins]
    t11, t33, tn = np.zeros_like(up1), np.zeros_like(up1), np.zeros_like(up1)
    fn = capi.lib().loma_foup2
    fn.argtypes = [ctypes.c_void_p] + [_fp] * 6 + [_dp] + [_fp] * 5 + [ctypes.c_int,
                                                                       ctypes.c_double, _dp]
    f = lambda a: a.view(np.float32).ctypes.data_as(_fp)
    dtr = np.zeros(1)
    assert fn(run._h, f(up1), f(up2), f(up3), f(t11), f(lap), f(t33), rhst.ctypes.data_as(_dp),
              f(t), f(tn), f(tx), f(ty), f(tz), 1, 0.0123, dtr.ctypes.data_as(_dp)) == 0
    run.close()
    for q, a in enumerate((up1, up2, up3, t11, lap, t33, tx, ty, tz, t, tn)):
        e = rel_l2(a[:, :g.mz, :], want[q])
        assert e < 2e-6, (q, e)


@pytest.mark.parametrize("shape,mixed", [((72, 65, 45), False), ((72, 65, 45), True),
                                         ((96, 65, 48), True)])
def test_statistics_step_fields(gpu, oracle_mod, shape, mixed):
    from loma_phd_amd import capi, ic
    print(f"statistics fields {shape} mixed={mixed}", flush=True)
    cfg = _cfg(*shape)
    st = ic.initial_condition(cfg)
    prec = capi.LOMA_MIXED if mixed else capi.LOMA_FP64
    gw, a = _gpu_windows(cfg, st, prec)
    _, b = _gpu_windows(cfg, st, prec, stats=False)
    for f in ("vor", "phi", "psi", "scal", "u00", "v00", "w00"):
        assert np.array_equal(a[f], b[f]), f
    _check(gw, _oracle_windows(oracle_mod, cfg, st), 1e-5 if mixed else 1e-9, "fields",
           floor=1e-3 if mixed else 1e-9)
