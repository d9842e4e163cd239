"""The implicit solves at the lattice sizes where their blocks can go wrong:
widths one below, at and one above a block's 256 columns and a narrow lattice,
heights that leave a partial last group of rows, and a lattice tall enough
that a block walks several groups.  Three steps of a flat channel with k-omega
and temperature, FP64, against the FP64 oracle with both solved to the
rounding floor: 1e-10 of each field's largest value, the bound the same
comparison keeps over 500 steps elsewhere.
"""
import numpy as np
import pytest

from komegafoulingmodel_amd import channel, lib
from pairs import fluid_mask, make_pair, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nX,nY", [(40, 12), (255, 13), (256, 16), (257, 19), (513, 70),
                                   (300, 1031)])
def test_solves_match_the_oracle(nX, nY):
    nu, Re, H = 0.01, 500.0, nY - 2.0
    w = channel.wavy_channel(nX, nY, H=H, amp=0.0, period=128.0, nu=nu, Re=Re,
                             Fval=channel.turbulent_forcing(H, nu, Re), seed=nX)
    L, orc = make_pair(w, "f64", solver_rtol=1e-15, solver_maxit=2000)
    tp = dict(alpha_fluid=nu / 0.708, alpha_foul=0.004, pr_turb=0.9, t_in=2.0, t_initial=0.5)
    L.thermal_init(**tp, rel_tol=1e-13, abs_tol=0.0, max_iters=2000)
    orc.init_thermal(**tp, rtol=1e-13, atol=0.0, maxit=2000)
    for _ in range(3):
        L.step(1, lib.OPTION_SAVE_MACRO_FIELDS)
        L.thermal_step(1)
        orc.step(1)
        orc.t_step(1)
    # the lattice's own columns: the padding to a multiple of 128 is not compared
    m = fluid_mask(orc.nType) & (np.arange(w.D) % w.XF < nX)
    errs = {f: rel_err(L.download(f)[m], a[m])
            for f, a in (("k", orc.K), ("omega", orc.O), ("T", orc.T), ("ux", orc.ux))}
    print(nX, nY, {k: f"{v:.2e}" for k, v in errs.items()}, flush=True)
    assert all(v < 1e-10 for v in errs.values()), errs
    L.close()
