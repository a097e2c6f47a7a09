"""Batched banded solves where a chunk of rows or a group of systems is part
filled: n around 8 and 16 (the chunk and the pair of chunks), system counts
around the three group sizes (16 to 4096 systems, 32 to 8192, 64).  The band
entries outside the matrix are NaN (they are not read into a result), and the
systems after the batch keep their bytes.  Diagonally dominant systems, FP64
arithmetic: errors of a few 1e-16, bar 1e-12 as in test_gpu_band.py.
"""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nsys", [(3, 1), (4, 17), (7, 64), (8, 15), (9, 33), (15, 16), (16, 5),
                                    (17, 70), (24, 31), (31, 3), (32, 18), (33, 130), (40, 2),
                                    (48, 9), (100, 40), (17, 4096), (19, 4099), (16, 8192),
                                    (18, 8250)])
@pytest.mark.parametrize("fp32", [False, True])
def test_band_edges(gpu, n, nsys, fp32):
    import torch
    from loma_phd_amd import capi
    print(f"band n={n} nsys={nsys} fp32={fp32}", flush=True)
    rng = np.random.default_rng(1000 * n + nsys)
    band = rng.uniform(-1.0, 1.0, (nsys, n, 5))
    band[:, :, 2] = 2.5 * np.abs(band[:, :, [0, 1, 3, 4]]).sum(axis=2) + 0.1
    A = np.zeros((nsys, n, n))
    for d in range(5):
        for j in range(n):
            if 0 <= j - 2 + d < n:
                A[:, j, j - 2 + d] = band[:, j, d]
            else:
                band[:, j, d] = np.nan
    rhs = rng.standard_normal((nsys, n)) + 1j * rng.standard_normal((nsys, n))
    if fp32:
        rhs = rhs.astype(np.complex64)
    ref = np.linalg.solve(A, rhs.astype(np.complex128)[..., None])[..., 0]
    b, r = torch.from_numpy(band).cuda(), torch.from_numpy(rhs).cuda()
    x = torch.full((nsys + 1, n), 3.0, dtype=torch.complex128, device="cuda")
    torch.cuda.synchronize()
    capi.band5_solve_dev(b.data_ptr(), r.data_ptr(), x.data_ptr(), n, nsys, rhs_fp32=fp32)
    got = x.cpu().numpy()
    assert rel_l2(got[:nsys], ref) < 1e-12
    assert np.all(got[nsys] == 3.0)
    assert np.array_equal(r.cpu().numpy(), rhs)
    if not fp32:  # in place
        capi.band5_solve_dev(b.data_ptr(), r.data_ptr(), None, n, nsys)
        assert np.array_equal(r.cpu().numpy(), got[:nsys])
