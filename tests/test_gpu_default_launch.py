"""The launch that plain steps take when no shape is set, at widths where the
last two-step tile of a row is cut to one column, to all but one, or not at
all, and on lattices of each size class; populations, macros and the wall
shear are bit-identical to one step per pass.  41 steps: an eager first step,
a captured block of 32, then pairs.
"""
import numpy as np
import pytest

from komegafoulingmodel_amd import channel, lib

pytestmark = pytest.mark.gpu


def _run(w, storage, one_step):
    L = lib.Lattice(w.nX, w.nY, storage=storage)
    if one_step:
        L.set_launch(256, 1, 1088, 1)
    L.set_params(w.tau0, w.Fval, w.nu)
    L.build_geometry(w.C0, w.BL, **dict(w.geom_params(), wall_d_search_rad=1))
    L.init_state(*w.initial_velocity(L.geometry("nType")))
    L.step(41, lib.OPTION_SAVE_MACRO_FIELDS)
    L.step(2)
    L.step(3, lib.OPTION_SAVE_MACRO_FIELDS)
    L.wall_shear()
    out = {f: L.download(f) for f in ("f", "ux", "uy", "rho", "tau_node")}
    L.close()
    return out


@pytest.mark.parametrize("nX,nY,storage", [
    (65, 40, "f32"), (127, 33, "f64"), (129, 50, "f16"),     # below 50,000 nodes
    (1281, 45, "f32"), (1343, 52, "bf16"), (705, 90, "f64"),  # below 600,000
    (1985, 310, "f32"), (1857, 330, "f64"),                   # above
    (2049, 490, "f16"), (2112, 480, "f16"), (2112, 480, "bf16"),  # 16-bit, above a million
    (4096, 980, "f32")])                                      # node pairs of 128 x 12
def test_default_launch_matches_one_step_per_pass(nX, nY, storage):
    w = channel.fouled_channel(nX, nY, Fval=1e-5, seed=nX, amp=(0.0, 8.0 * nY / 1024.0))
    a, b = _run(w, storage, False), _run(w, storage, True)
    for f in a:
        assert np.array_equal(a[f], b[f]), f


def test_autotune_keeps_the_bits_on_an_odd_width():
    w = channel.fouled_channel(333, 60, Fval=1e-5, seed=5, amp=(0.0, 0.5))
    ref = _run(w, "f32", True)
    L = lib.Lattice(w.nX, w.nY)
    L.set_params(w.tau0, w.Fval, w.nu)
    L.build_geometry(w.C0, w.BL, **dict(w.geom_params(), wall_d_search_rad=1))
    block, npt, pad, _, spp = L.autotune(20)
    L.init_state(*w.initial_velocity(L.geometry("nType")))
    L.step(46)
    assert np.array_equal(L.download("f"), ref["f"])
    L.set_launch(block, npt, pad, spp)  # what it returns can be set
    L.close()


@pytest.mark.parametrize("nX,storage", [(20, "f32"), (65, "f32"), (129, "f64"), (333, "f16")])
@pytest.mark.parametrize("tile", [512, 640, 832, 1856])
def test_two_step_tiles_can_be_set_on_any_width(nX, storage, tile):
    """Rows whose last tile (64 or 128 columns) has 1 to 77 of them."""
    w = channel.flat_channel(nX, 45, Fval=1e-5, seed=nX)
    f = []
    for shape in ((256, 1, 1088, 1), (tile, 1, 64, 2)):
        L = lib.Lattice(w.nX, w.nY, storage=storage)
        L.set_params(w.tau0, w.Fval, w.nu)
        L.build_geometry(w.C0, w.BL, **dict(w.geom_params(), x_release_pos=min(10.0, nX / 10)))
        L.set_launch(*shape)
        L.init_state(*w.initial_velocity(L.geometry("nType")))
        L.step(43, lib.OPTION_SAVE_MACRO_FIELDS)
        f.append((L.download("f"), L.download("ux")))
        if shape[3] == 2:
            for pairs in (1024, 1536, 1664, 3584):  # node pairs need whole tiles
                with pytest.raises(lib.KofmError):
                    L.set_launch(pairs, 1, 64, 2)
        L.close()
    assert np.array_equal(f[0][0], f[1][0]) and np.array_equal(f[0][1], f[1][1])


def test_autotune_returns_the_shape_it_keeps_on_an_odd_width():
    """2001 x 203, where two steps per pass take half the time of one (5.4
    against 10.8 us a step): the shape that is returned has two and can be set."""
    w = channel.flat_channel(2001, 203, Fval=1e-5, seed=1)
    L = lib.Lattice(w.nX, w.nY)
    L.set_params(w.tau0, w.Fval, w.nu)
    L.build_geometry(w.C0, w.BL, **dict(w.geom_params(), wall_d_search_rad=1))
    L.init_state(*w.initial_velocity(L.geometry("nType")))
    block, npt, pad, ms, spp = L.autotune(40)
    print(block, npt, pad, ms, spp, flush=True)
    assert spp == 2
    L.set_launch(block, npt, pad, spp)
    L.step(41)
    L.close()
