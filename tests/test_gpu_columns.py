"""The y operators at every chunk size M (rows per lane) against the oracle.

The coefficient tables are streams of 16-byte vectors whose last vector may be
part filled, by the parity of M and of the row width; rows past the grid's
last row are padding.  One size per M, each with a remainder.  Bars as in
test_gpu_ops.py (orders of operations differ): 1e-11 for derivatives, 1e-10
for solves.
"""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


def _dev(torch, a):
    t = torch.from_numpy(np.ascontiguousarray(a)).cuda()
    torch.cuda.synchronize()
    return t


@pytest.mark.parametrize("my", [16, 63, 131, 250, 320, 383, 447, 453, 575, 611, 700, 830, 1000])
def test_columns(gpu, oracle_mod, my):
    import torch
    from loma_phd_amd import capi, grid
    y = grid.tanh_mesh(my, 20.0)
    run = capi.Run(48, my, 48, y, 300.0, 0.25, 0.25)
    g = oracle_mod.Grid(48, my, 48, y, 300.0, 0.25, 0.25)
    rng = np.random.default_rng(my)
    n = 5
    u = rng.standard_normal((n, my)) + 1j * rng.standard_normal((n, my))
    ud, vd, dd = _dev(torch, u), _dev(torch, np.zeros_like(u)), _dev(torch, np.zeros_like(u))
    print(f"derivatives my={my}", flush=True)
    run.deryr2_dev(ud.data_ptr(), vd.data_ptr(), n)
    assert rel_l2(vd.cpu().numpy(), g.deryr2(u)) < 1e-11
    run.deryyr2_dev(ud.data_ptr(), vd.data_ptr(), n)
    assert rel_l2(vd.cpu().numpy(), g.deryyr2(u)) < 1e-11
    rK = 10 ** rng.uniform(-1, 3, n)
    rd = _dev(torch, rK)
    for name in ("lapvdvhom", "solvepsi"):
        print(f"{name} my={my}", flush=True)
        getattr(run, name + "_dev")(ud.data_ptr(), vd.data_ptr(), dd.data_ptr(), rd.data_ptr(), n)
        v, dv = vd.cpu().numpy(), dd.cpu().numpy()
        for c in range(n):
            vo, dvo = getattr(g, name)(u[c], rK[c])
            assert rel_l2(v[c], vo) < 1e-10, (name, c)
            assert rel_l2(dv[c], dvo) < 1e-10, (name, c)
    du = rng.standard_normal(my)
    x, o = _dev(torch, du), _dev(torch, np.zeros(my))
    run.inty8_dev(x.data_ptr(), o.data_ptr())
    assert rel_l2(o.cpu().numpy(), g.inty8(du)) < 1e-10
