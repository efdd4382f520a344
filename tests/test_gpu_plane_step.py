"""The fused step's plane kernel at the edges of its mapping: rows per thread
that divide NPA or leave a ragged last chunk, chunks that straddle waves or
fill them, one wave and many, few and many planes per CU.  One fused step is
compared bit for bit with the same step taken operator by operator (other
kernels), and with the oracle."""
import numpy as np
import pytest

from conftest import gpu_available
from helpers import max_rel_err, random_problem
from oracle.oracle import Oracle
from ramgpu import inputs, species as sp
from ramgpu.capi import RamGpu

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="no GPU")]

RTOL = 1e-12  # the step's tolerance (tests/test_gpu_parity.py): the loss factors' exponentials

# (NR, NT, NE, NPA)
GRIDS = [(4, 4, 4, 4), (5, 6, 4, 5), (6, 7, 8, 16), (5, 5, 16, 13), (6, 5, 63, 20), (5, 6, 64, 17),
         (4, 5, 65, 33), (5, 4, 31, 61), (4, 4, 7, 120), (20, 6, 35, 72), (6, 40, 48, 90), (5, 30, 64, 90)]


def _step_by_operators(g, p):
    """src/ModRamRun.f90:64-201 through the entry points of single operators."""
    for s, spc in enumerate(p.grid.species, start=1):
        for op in ("driftr", "driftp", "drifte", "driftmu"):
            getattr(g, op)(s)
        losses = ([g.wavelo] if p.wave is not None and p.wave.wpi[s - 1] else []) + \
            ([g.charexchange] if spc.cex else []) + [g.atmol]
        for op in losses + losses[::-1]:
            op(s)
        for op in ("driftmu", "drifte", "driftp", "driftr"):
            getattr(g, op)(s)
    f = g.get_f2()
    f[:, :, p.grid.nt - 1] = f[:, :, 0]
    f[:, np.asarray(p.geom.outside_mgnp) == 1] = 1e-31
    return f


@pytest.mark.parametrize("grid", GRIDS, ids=lambda g: "x".join(map(str, g)))
def test_fused_step_at_mapping_edges(grid):
    p = random_problem(*grid, species=(sp.ELECTRON, sp.OXYGEN), seed=sum(grid))
    p.wave = inputs.wave_inputs(p.grid, p.kp)
    a, b = RamGpu.from_problem(p), RamGpu.from_problem(p)
    out = a.ram_run(1)
    fused = a.get_f2()
    diff = np.argwhere(fused != _step_by_operators(b, p))
    assert diff.size == 0, f"{len(diff)} cells differ, first at {diff[0]}"
    o = Oracle(p)
    o.ram_run()
    assert max_rel_err(fused, o.f2) <= RTOL
    for s in range(p.grid.ns):
        for k in ("setrc", "lsdr", "lscha", "lsatm", "lswae"):
            assert abs(out[s][k] - o.arr(k)[s]) <= RTOL * abs(o.arr("setrc")[s]), (s, k)
        for n, k in enumerate(("dtdrift_r", "dtdrift_p", "dtdrift_e", "dtdrift_mu")):
            ref = o.dtdrift()[s, n]
            assert abs(out[s][k] - ref) <= RTOL * abs(ref), (s, k)
    a.close()
    b.close()
