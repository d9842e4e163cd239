"""Fields reach the host whole at the sizes where their way changes: below one
piece of pinned memory (1 MiB), across pieces with a remainder, and, for large
fields (the last size's in both precisions), in four parts.  The populations
come back as they were uploaded (FP64 storage: to the last bits of
f = w + (f - w)), and a field downloaded twice, or reduced on the device,
agrees with itself.
"""
import numpy as np
import pytest

from komegafoulingmodel_amd import channel, lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nX,nY", [(100, 8), (130, 75), (1025, 129), (1500, 467),
                                   (2049, 1030)])
@pytest.mark.parametrize("storage", ["f32", "f64"])
def test_fields_come_back_whole(nX, nY, storage):
    w = channel.flat_channel(nX, nY, seed=nX)
    L = lib.Lattice(nX, nY, storage=storage)
    L.set_params(w.tau0, w.Fval, w.nu)
    L.build_geometry(w.C0, w.BL, **w.geom_params())
    inside = (L.geometry("nType").astype(np.int32) & 1) == 0
    inside &= np.arange(w.D) % w.XF < nX
    rng = np.random.default_rng(nX)
    f = np.array([4 / 9] + 4 * [1 / 9] + 4 * [1 / 36])[:, None] + rng.uniform(-1e-2, 1e-2, (9, w.D))
    f[:, ~inside] = 0.0
    L.upload_state(f.reshape(-1))
    got = L.download("f").reshape(9, -1)
    # FP64: two roundings of values below 1; FP32: one of a deviation below 2^-6
    assert np.max(np.abs(got - f)) <= (2.0 ** -52 if storage == "f64" else 2.0 ** -30)
    rho = L.download("rho")
    assert np.array_equal(rho, L.download("rho"))
    assert np.max(np.abs(rho[inside] - f.sum(0)[inside])) < 1e-6
    assert L.reduce("ux", lib.RED_MAX) == L.download("ux").max()
    L.close()
