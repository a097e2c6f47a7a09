"""Batched solves larger than the run's workspace (256 MiB of LU tables: 6,553
systems of 1,000 rows, half that for visc, which factors two) go through it in
pieces, and batches of a few, of part of a wavefront and of many systems clear
the rows past the grid in different ways.  A column's arithmetic does not
depend on its batch, so every column of a large batch, a handful repeated with
a period that divides no piece, equals the small batch's bit for bit, whatever
was solved on the run before, and the columns past the batch keep their bytes.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PERIOD = 7


def _tile(torch, a, ncols):
    """ncols columns of a's, and two more of sevens behind them"""
    idx = torch.arange(ncols + 2) % PERIOD
    t = a[idx].cuda()
    t[ncols:] = 7.0
    return t.contiguous()


@pytest.mark.parametrize("my,ncols", [(1000, 6600), (129, 70), (129, 300), (63, 7), (17, 40)])
def test_pieces(gpu, my, ncols):
    import torch
    from loma_phd_amd import capi, grid
    run = capi.Run(48, my, 48, grid.tanh_mesh(my, 20.0), 300.0, 0.25, 0.25)
    g = torch.Generator().manual_seed(my)
    f = torch.randn(PERIOD, my, 2, dtype=torch.float64, generator=g)
    rK = 10.0 ** (torch.rand(PERIOD, dtype=torch.float64, generator=g) * 4.0 - 1.0)

    def solve(kind, n):
        x, k = _tile(torch, f, n), _tile(torch, rK, n)
        v, dv = torch.full_like(x, 7.0), torch.full_like(x, 7.0)
        torch.cuda.synchronize()
        if kind == "helmholtz":
            run.helmholtz_dev(x.data_ptr(), v.data_ptr(), k.data_ptr(), 3.0, n)
        else:
            getattr(run, kind + "_dev")(x.data_ptr(), v.data_ptr(), dv.data_ptr(),
                                        k.data_ptr(), n)
        return v.cpu(), dv.cpu()

    for kind in ("lapvdvhom", "solvepsi", "helmholtz"):
        print(f"{kind} my={my} columns={ncols}", flush=True)
        small = solve(kind, PERIOD)
        big = solve(kind, ncols)
        again = solve(kind, PERIOD)
        for s, b, a in zip(small, big, again):
            assert torch.equal(s, a)
            assert torch.isfinite(b).all()
            assert torch.equal(b[:ncols], s[torch.arange(ncols) % PERIOD])
            assert (b[ncols:] == 7.0).all()
    run.close()


@pytest.mark.parametrize("my,ncols", [(1000, 3300), (129, 70), (17, 40)])
def test_visc_pieces(gpu, my, ncols):
    import torch
    from loma_phd_amd import capi, grid
    run = capi.Run(48, my, 48, grid.tanh_mesh(my, 20.0), 300.0, 0.25, 0.25)
    g = torch.Generator().manual_seed(my)
    f = [torch.randn(PERIOD, my, 2, dtype=torch.float64, generator=g) for _ in range(6)]
    rK = [10.0 ** (torch.rand(PERIOD, dtype=torch.float64, generator=g) * 3.0) for _ in range(2)]

    def visc(n):
        a, k = [_tile(torch, x, n) for x in f], [_tile(torch, x, n) for x in rK]
        torch.cuda.synchronize()
        run.visc_dev(*[x.data_ptr() for x in a], *[x.data_ptr() for x in k], 0.3, 0.2, 0.1, n)
        return [x.cpu() for x in a]

    print(f"visc my={my} columns={ncols}", flush=True)
    small, big, again = visc(PERIOD), visc(ncols), visc(PERIOD)
    for s, b, a in zip(small, big, again):
        assert torch.equal(s, a)
        assert torch.isfinite(b).all()
        assert torch.equal(b[:ncols], s[torch.arange(ncols) % PERIOD])
        assert (b[ncols:] == 7.0).all()
    run.close()


def test_null_wavenumbers_are_refused(gpu):
    """No wavenumbers: an error of the call, nothing launched; no columns: nothing
    to do."""
    import torch
    from loma_phd_amd import capi, grid
    run = capi.Run(48, 17, 48, grid.tanh_mesh(17, 20.0), 300.0, 0.25, 0.25)
    x = torch.ones(3, 17, 2, dtype=torch.float64, device="cuda")
    v = torch.full_like(x, 7.0)
    torch.cuda.synchronize()
    for call in (run.lapvdvhom_dev, run.solvepsi_dev):
        with pytest.raises(capi.LomaError):
            call(x.data_ptr(), v.data_ptr(), v.data_ptr(), None, 3)
        call(x.data_ptr(), v.data_ptr(), v.data_ptr(), None, 0)
    with pytest.raises(capi.LomaError):
        run.helmholtz_dev(x.data_ptr(), v.data_ptr(), None, 1.0, 3)
    assert (v.cpu() == 7.0).all()
    run.close()
