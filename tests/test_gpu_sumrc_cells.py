"""SUMRC adds the cells I, K, L >= 2, J <= NT-1 (src/ModRamRun.f90:246-255);
what the others hold, NaN and infinities too, must not reach the energy
records.  A run whose K=1 cells are NaN gives bit for bit the records of the
run in which they are not: no operator carries them to other cells."""
import numpy as np
import pytest

from conftest import gpu_available
from helpers import random_problem
from ramgpu import inputs, species as sp
from ramgpu.capi import RamGpu

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="no GPU")]

RECORDS = ("setrc", "lsdr", "lscha", "lsatm", "lswae", "lscoe", "lscsc")


def _runs(p, set_up):
    """The records and F2 of one step from p, and from p with K=1 NaN."""
    out = []
    for spoil in (False, True):
        f = p.f2.copy(order="F")
        if spoil:
            f[:, :, :, 0, :] = np.nan
        g = RamGpu.from_problem(p)
        set_up(g)
        g.put_f2(f)
        out.append((g.ram_run(1), g.get_f2()))
        g.close()
    return out


# one thread per line (69120 lines), lines in chunks (1225 lines)
@pytest.mark.parametrize("grid", [(4, 30, 48, 48), (5, 7, 7, 25)], ids=lambda g: "x".join(map(str, g)))
def test_setrc_leaves_out_the_first_energy(grid):
    p = random_problem(*grid, species=(sp.HYDROGEN,), seed=3)
    (ra, fa), (rb, fb) = _runs(p, lambda g: None)
    np.testing.assert_array_equal(fa[:, :, :, 1:], fb[:, :, :, 1:])
    assert np.isfinite(ra[0]["setrc"])
    assert rb[0]["setrc"] == ra[0]["setrc"]


@pytest.mark.parametrize("coul,pitch", [(True, False), (False, True), (True, True)])
def test_records_of_optional_processes_leave_out_the_first_energy(coul, pitch):
    p = random_problem(5, 6, 12, 20, species=(sp.ELECTRON, sp.OXYGEN, sp.HYDROGEN, sp.HELIUM), seed=4)
    p.wave = inputs.wave_inputs(p.grid, p.kp, wpi=[0, 1, 0, 0])
    if coul:
        p.coulomb = inputs.CoulombInputs(inputs.plasmasphere_density(p.grid, p.kp), 600.0)
    d = inputs.pitch_diffusion_coef(p.grid, p.geom, scale=1e-5, seed=1)

    def set_up(g):
        if pitch:  # He+ takes none of them
            g.set_wpadif(1, d, None, True, False)
            g.set_wpadif(3, d, None, False, True)
            g.set_flc(2, d)

    (ra, fa), (rb, fb) = _runs(p, set_up)
    np.testing.assert_array_equal(fa[:, :, :, 1:], fb[:, :, :, 1:])
    for s in range(4):
        for k in RECORDS:
            assert rb[s][k] == ra[s][k] and np.isfinite(ra[s][k]), (s, k, ra[s][k], rb[s][k])
