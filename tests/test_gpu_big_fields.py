"""Transform fields of more than 4 GiB (512x1024x1620, FP64: 4.5 GB each, some
170 GB a run): the row x lines with 64-bit offsets.

The z modes are multiples of 45, so every z line repeats with a period of 36
points, and the run does what one of 36 z points and 45 times the spanwise
wavenumber does: 1620 / 3 - 1 = 539 and 36 / 3 - 1 = 11 = 539 / 45 modes are
kept, so the truncations agree too.  One substep of both, FP64, from random
modes; the z transforms of 1620 and of 36 points round differently, a few
1e-16 of a field's size, and the second derivatives of the y operators amplify
that by up to 1 / dy^2: bars 1e-9 for Omega_y and phi, 1e-12 for T."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

P = 45


def test_big_fields(gpu):
    import torch
    from loma_phd_amd import capi, grid
    mgalx, my = 512, 1024
    if torch.cuda.mem_get_info()[0] < 1.05 * capi.footprint(mgalx, my, 36 * P):
        pytest.skip("needs some 170 GB of device memory")
    y = grid.tanh_mesh(my, 20.0)
    rng = np.random.default_rng(1)
    small = capi.Run(mgalx, my, 36, y, 400.0, 0.25, 0.25 * P, dt0=1e-3)
    n, mz, _ = small.shape()
    nz = small.nz
    f = {k: np.zeros((n, mz, my), np.complex128) for k in ("vor", "phi", "scal")}
    env = np.exp(-((y / 5.0) ** 2))
    nx = 40  # x modes: all products stay below the truncation's noise
    for k, a in (("vor", 1e-2), ("phi", 1e-1), ("scal", 1e-3)):
        c = rng.standard_normal((nx, mz, 2)) @ np.array([1.0, 1.0j])
        f[k][1:nx + 1] = a * c[:, :, None] * env
    f["scal"][0, 0] = 1.0 + 0.2 * np.tanh(y)
    u00 = 0.5 * np.tanh(2.0 * y)
    got = {}
    names = ("vor", "phi", "scal")
    for mgalz, step in ((36, 1), (36 * P, P)):
        print(f"big fields, {mgalz} z points", flush=True)
        run = small if step == 1 else capi.Run(mgalx, my, mgalz, y, 400.0, 0.25, 0.25, dt0=1e-3)
        if step > 1:
            assert run.nplanes * mgalz * 1024 * 16 > 1 << 32
            assert run.nz // P == nz
        kz = np.r_[np.arange(nz + 1), np.arange(-nz, 0)] * step
        full = {}
        for k in names:
            full[k] = np.zeros(run.shape(), np.complex128)
            full[k][:, kz % run.mz] = f[k]
        zero = np.zeros(run.shape(), np.complex128)  # pages are not touched
        p = lambda a: a.ctypes.data_as(ctypes.c_void_p)
        z1 = np.zeros(my)
        capi.check(capi.lib().loma_upload(run.handle, p(full["vor"]), p(full["phi"]), p(zero),
                                          p(full["scal"]), capi._d(u00), capi._d(z1), capi._d(z1),
                                          1))
        print("uploaded", flush=True)
        run.substep(1)
        print("substep done", flush=True)
        capi.check(capi.lib().loma_download(run.handle, *[p(full[k]) if k != "psi" else None
                                                          for k in ("vor", "phi", "psi", "scal")],
                                            None, None, None, 1))
        got[step] = {k: full[k][:, kz % run.mz].copy() for k in names}
        if step > 1:  # nothing in the modes between
            for k in names:
                between = np.ones(run.mz, bool)
                between[kz % run.mz] = False
                top = max(float(np.abs(full[k][i, between]).max()) for i in (0, 1, 20, 100, n - 1))
                assert top <= 1e-9 * np.abs(got[step][k]).max(), (k, top)
        run.close()
    for k, bar in (("vor", 1e-9), ("phi", 1e-9), ("scal", 1e-12)):
        inc = [got[s][k] - f[k] for s in (1, P)]
        e = np.linalg.norm(inc[1] - inc[0]) / np.linalg.norm(got[1][k])
        print(f"{k}: {e:.2e}", flush=True)
        assert np.linalg.norm(inc[0]) > 0.0
        assert e <= bar, (k, e)
