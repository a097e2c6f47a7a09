"""fourz over large batches at lengths of the run-time plan: several rows share a
workgroup from 2,048 rows on (as many as the length leaves room for), and the
last workgroup is part filled.  FP64 rows of at most four radix passes: a few
1e-16 relative, bar 1e-12 as in test_gpu_ops.py; rows past the batch keep
their bytes."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,counts", [
    (8, (2049, 5003, 140001)), (36, (2049, 5003, 50001)), (45, (2049, 5003, 50001)),
    (90, (2047, 2049, 30001)), (250, (3073, 5003)), (500, (2049, 5003)), (540, (2049,))])
def test_fourz_batches(gpu, n, counts):
    import torch
    from loma_phd_amd import capi, grid
    run = capi.Run(48, 17, n, grid.tanh_mesh(17, 20.0), 300.0, 0.25, 0.25)
    rng = np.random.default_rng(n)
    for nrows in counts:
        c = rng.standard_normal((nrows + 3, n)) + 1j * rng.standard_normal((nrows + 3, n))
        for iopt in (-1, 1):
            print(f"fourz n={n} rows={nrows} iopt={iopt}", flush=True)
            d = torch.from_numpy(c.copy()).cuda()
            torch.cuda.synchronize()
            run.fourz_dev(d.data_ptr(), nrows, iopt)
            torch.cuda.synchronize()
            got = d.cpu().numpy()
            ref = np.fft.fft(c, axis=1) / n if iopt < 0 else np.fft.ifft(c, axis=1) * n
            assert rel_l2(got[:nrows], ref[:nrows]) < 1e-12
            # every row, not only the batch's norm
            e = np.linalg.norm(got[:nrows] - ref[:nrows], axis=1)
            assert (e <= 1e-12 * np.linalg.norm(ref[:nrows], axis=1)).all()
            assert np.array_equal(got[nrows:], c[nrows:])
    run.close()
