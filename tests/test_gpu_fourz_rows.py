"""fourz over batches of rows: the lengths of the wavefront-per-row kernel and
lengths of the run-time plan, with row counts that leave the last workgroup
(and its last wavefront) part filled.  Rows in FP64, at most 2^9 points and
four radix passes: a relative L2 error of a few 1e-16, bar 1e-12 as in
test_gpu_ops.py; rows past the batch keep their bytes.
"""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [64, 96, 128, 192, 256, 384, 512, 8, 36, 45, 90, 100, 270, 500])
def test_fourz_rows(gpu, n):
    import torch
    from loma_phd_amd import capi, grid
    run = capi.Run(48, 17, n, grid.tanh_mesh(17, 20.0), 300.0, 0.25, 0.25)
    rng = np.random.default_rng(n)
    for nrows in (1, 3, 67, 613):
        c = rng.standard_normal((nrows + 2, n)) + 1j * rng.standard_normal((nrows + 2, n))
        for iopt in (-1, 1):
            print(f"fourz n={n} rows={nrows} iopt={iopt}", flush=True)
            d = torch.from_numpy(c.copy()).cuda()
            torch.cuda.synchronize()
            run.fourz_dev(d.data_ptr(), nrows, iopt)
            torch.cuda.synchronize()
            got = d.cpu().numpy()
            ref = np.fft.fft(c, axis=1) / n if iopt < 0 else np.fft.ifft(c, axis=1) * n
            assert rel_l2(got[:nrows], ref[:nrows]) < 1e-12
            assert np.array_equal(got[nrows:], c[nrows:])
