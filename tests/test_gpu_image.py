"""Images of a run as host arrays: fields smaller than a slot of the host
staging, of a few slots and of all sixteen (more than one thread copies), with
some of the fields left out.  Uploaded numbers come back as they were, and the
FP32 image is each number rounded to nearest: equal bits, no tolerance.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ("vor", "phi", "psi", "scal")


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("shape", [(12, 17, 8), (48, 65, 48), (60, 131, 64), (192, 131, 96)])
def test_image(gpu, shape, precision):
    from loma_phd_amd import capi, grid
    mgalx, my, mgalz = shape
    print(f"image {shape} precision {precision}", flush=True)
    run = capi.Run(mgalx, my, mgalz, grid.tanh_mesh(my, 20.0), 300.0, 0.25, 0.25,
                   precision=precision, flags=capi.LOMA_FLAG_SCALAR_Z)
    rng = np.random.default_rng(my)
    s = run.shape()
    f = {k: (rng.standard_normal(s) + 1j * rng.standard_normal(s)) * 10.0 ** rng.uniform(-40, 6, s)
         for k in FIELDS + ("z",)}
    f["scal"][0, 0] = 1.0  # upload takes a positive mean T only
    m = rng.standard_normal((3, my))
    run.upload(*[f[k] for k in FIELDS], *m, z=f["z"])
    got = run.download()
    for k, v in f.items():
        assert np.array_equal(got[k], v), k
    for k, v in zip(("u00", "v00", "w00"), m):
        assert np.array_equal(got[k], v), k
    p = lambda a: None if a is None else a.ctypes.data_as(ctypes.c_void_p)
    out = {k: np.full(s, 7.0, np.complex64) for k in f}
    for leave in ((), ("vor",), ("phi", "scal"), FIELDS):
        a = [None if k in leave else out[k] for k in FIELDS]
        capi.check(capi.lib().loma_download(run.handle, *[p(q) for q in a], None, None, None, 0))
        for k in FIELDS:
            want = np.full(s, 7.0, np.complex64) if k in leave else f[k].astype(np.complex64)
            assert np.array_equal(out[k], want), (k, leave)
            out[k][...] = 7.0
    capi.check(capi.lib().loma_download_z(run.handle, p(out["z"]), 0))
    assert np.array_equal(out["z"], f["z"].astype(np.complex64))
