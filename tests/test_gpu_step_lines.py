"""The plane kernel of a step with Coulomb collisions, WPADIF and FLCscatter at
the edges of its mapping (lines that end in a chunk's first rows, one wave and
many, one chunk and many).  One ram_run step is compared bit for bit with the
same step taken operator by operator (other kernels), and its energy records
with the SUMRCs between those operators."""
import numpy as np
import pytest

from conftest import gpu_available
from helpers import random_problem
from ramgpu import inputs, species as sp
from ramgpu.capi import RamGpu

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="no GPU")]

RTOL = 1e-12  # of SETRC: the sums' order
KIND = ("lsdr", "lscha", "lsatm", "lswae", "lscoe", "lscsc")

# (NR, NT, NE, NPA), Coulomb collisions, FLCscatter acting
CASES = [((4, 4, 4, 4), False, True), ((5, 6, 4, 5), False, True), ((4, 5, 7, 120), True, True),
         ((6, 5, 63, 20), True, True), ((5, 6, 64, 17), True, False), ((4, 5, 65, 33), True, True),
         ((5, 4, 31, 61), False, True), ((5, 5, 16, 13), True, True), ((20, 8, 35, 72), True, True),
         ((6, 40, 48, 90), True, True), ((5, 30, 64, 90), False, True)]


def _set_up(p, flc_on):
    """e-: WPADIF at the WPI positions; O+: WAVELO, FLCscatter; H+: EMIC, FLCscatter; He+: none."""
    g = RamGpu.from_problem(p)
    d = [inputs.pitch_diffusion_coef(p.grid, p.geom, scale=sc, seed=n) for n, sc in enumerate((1e-5, 3e-6, 5e-6))]
    g.set_time(600.0)
    g.set_wpadif(1, d[0], d[1], True, False)
    g.set_wpadif(3, d[1], None, False, True)
    for s in (2, 3):
        g.set_flc(s, d[2], dt_bc=300.0 if flc_on else 900.0)
    return g


def _step_by_operators(g, p, coul):
    """src/ModRamRun.f90:64-201 through the entry points of single operators,
    with a SUMRC after each but FLCscatter."""
    rec = []
    for s, spc in enumerate(p.grid.species, start=1):
        r = dict.fromkeys(KIND, 0.0)

        def op(name, book=None, s=s, r=r):
            getattr(g, name)(s)
            if book:
                r[book] += g.sumrc(s)[1]

        wpi = {1: ["wpadif"], 2: ["wavelo"]}.get(s, [])
        half = [(n, "lswae") for n in wpi] + ([("wpadif", "lswae")] if s == 3 else []) + \
            ([("charexchange", "lscha")] if spc.cex else []) + ([("flcscatter", None)] if s in (2, 3) else [])
        for n in ("driftr", "driftp", "drifte"):
            op(n)
        op("driftmu", "lsdr")
        if coul:
            op("coulen", "lscoe")
            op("coulmu", "lscsc")
        for n, b in half + [("atmol", "lsatm")] * 2 + half[::-1]:
            op(n, b)
        if coul:
            op("coulmu", "lscsc")
            op("coulen", "lscoe")
        for n in ("driftmu", "drifte", "driftp"):
            op(n)
        op("driftr", "lsdr")
        r["setrc"] = g.sumrc(s)[0]
        rec.append(r)
    f = g.get_f2()
    f[:, :, p.grid.nt - 1] = f[:, :, 0]
    f[:, np.asarray(p.geom.outside_mgnp) == 1] = 1e-31
    return f, rec


@pytest.mark.parametrize("grid,coul,flc_on", CASES, ids=lambda v: "x".join(map(str, v)) if type(v) is tuple else str(v))
def test_step_with_optional_processes_at_mapping_edges(grid, coul, flc_on):
    p = random_problem(*grid, species=(sp.ELECTRON, sp.OXYGEN, sp.HYDROGEN, sp.HELIUM), seed=sum(grid))
    p.wave = inputs.wave_inputs(p.grid, p.kp, wpi=[0, 1, 0, 0])
    if coul:
        p.coulomb = inputs.CoulombInputs(inputs.plasmasphere_density(p.grid, p.kp), 600.0)
    a, b = _set_up(p, flc_on), _set_up(p, flc_on)
    for s in range(1, 5):  # SETRC of the start, for the first ELORC
        a.sumrc(s)
        b.sumrc(s)
    out = a.ram_run(1)
    fused = a.get_f2()
    ref, rec = _step_by_operators(b, p, coul)
    diff = np.argwhere(fused != ref)
    assert diff.size == 0, f"{len(diff)} cells differ, first at {diff[0]}"
    for s in range(4):
        for k in rec[s]:
            assert abs(out[s][k] - rec[s][k]) <= RTOL * abs(rec[s]["setrc"]), (s, k, out[s][k], rec[s][k])
    a.close()
    b.close()
