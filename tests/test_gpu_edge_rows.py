"""The edge rows of the first derivative's right-hand side, where they lie.

B1 comes from scalar registers with its first and last three rows apart; the
last three start at any row of a lane's chunk and run on into the next lane,
or end with lane 63.  Every chunk size M, the two starts that cross lanes and
the full grid of 64 M rows, against the oracle with the bars of
test_gpu_columns.py (1e-11) and test_gpu_xlines.py (1e-5, mixed).
"""
import numpy as np
import pytest

from conftest import rel_l2
from test_gpu_columns import _dev
from test_gpu_step import _cfg, _setup

pytestmark = pytest.mark.gpu

CHUNKS = [3, 4, 5, 6, 7, 8, 9, 10, 12, 14, 16]


def _sizes(M):
    big = range(64 * M, 64 * M - 2 * M, -1)
    return [64 * M] + [next(my for my in big if (my - 3) % M == M - q) for q in (1, 2)]


@pytest.mark.parametrize("my", [my for M in CHUNKS for my in _sizes(M)])
def test_first_derivative(gpu, oracle_mod, my):
    from loma_phd_amd import capi, grid
    print(f"first derivative my={my}", flush=True)
    y = grid.tanh_mesh(my, 20.0)
    run = capi.Run(48, my, 48, y, 300.0, 0.25, 0.25)
    g = oracle_mod.Grid(48, my, 48, y, 300.0, 0.25, 0.25)
    rng = np.random.default_rng(my)
    u = rng.standard_normal((3, my)) + 1j * rng.standard_normal((3, my))
    import torch
    ud, vd = _dev(torch, u), _dev(torch, np.zeros_like(u))
    run.deryr2_dev(ud.data_ptr(), vd.data_ptr(), 3)
    v, want = vd.cpu().numpy(), g.deryr2(u)
    assert rel_l2(v, want) < 1e-11
    assert rel_l2(v[:, -6:], want[:, -6:]) < 1e-11 and rel_l2(v[:, :6], want[:, :6]) < 1e-11


@pytest.mark.parametrize("my", _sizes(4)[1:] + _sizes(5)[1:])
def test_mixed_step(gpu, oracle_mod, my):
    from loma_phd_amd import capi, diagnostics, ic
    print(f"mixed step my={my}", flush=True)
    cfg = _cfg(64, my, 24, Re=160.0, s=2.0, seed=my)
    run, S, g = _setup(cfg, capi.LOMA_MIXED, False)
    run.advance(1)
    assert S.step(1) == 0
    errs = diagnostics.field_errors(run.download(), S.get(), ic.HostOps(cfg.y()), cfg.alp, cfg.bet)
    for f, e in errs.items():
        assert e < 1e-5, (f, e)
