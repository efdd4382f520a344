"""The plane adjoint of a step at the edges of its mapping: chunks that divide
NPA or leave a ragged last one, columns that straddle waves or fill them, one
wave and many.  The adjoint of one fused step is compared with the adjoints of
its operators one after the other (other kernels) at the states between them,
which the fused step passes bit for bit."""
import numpy as np
import pytest

from conftest import gpu_available
from helpers import random_problem
from ramgpu import species as sp
from ramgpu.capi import RamGpu

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="no GPU")]

# both sides add the same products, a cell's few in another order
RTOL = 1e-12  # of the largest adjoint of the species

# (NR, NT, NE, NPA)
GRIDS = [(4, 4, 4, 4), (5, 6, 4, 5), (6, 7, 8, 16), (5, 5, 16, 13), (6, 5, 63, 20), (5, 6, 64, 17), (4, 5, 65, 33),
         (5, 4, 31, 61), (4, 4, 7, 120), (20, 6, 35, 72), (6, 40, 41, 60), (5, 30, 60, 29)]


@pytest.mark.parametrize("grid", GRIDS, ids=lambda g: "x".join(map(str, g)))
def test_step_adjoint_at_mapping_edges(grid):
    p = random_problem(*grid, species=(sp.ELECTRON, sp.OXYGEN), seed=sum(grid), spiky=True)
    g = RamGpu.from_problem(p)
    x = g.get_f2()
    rng = np.random.default_rng(sum(grid))
    ybar = np.asfortranarray(rng.standard_normal(x.shape))
    ybar[:, :, -1] = 0.0  # the seam and the mask are DRIFTR's last sweep's
    ybar[:, np.asarray(p.geom.outside_mgnp) == 1] = 0.0
    got, got_b = g.ram_run_bwd(ybar)
    ref, ref_b = ybar, np.zeros_like(got_b)
    for s, spc in enumerate(p.grid.species, start=1):
        half = ["charexchange"] if spc.cex else []
        ops = ["driftr", "driftp", "drifte", "driftmu"] + half + ["atmol", "atmol"] + half + \
            ["driftmu", "drifte", "driftp", "driftr"]
        g.put_f2(x)
        states = []
        for op in ops:
            states.append(g.get_f2())
            getattr(g, op)(s)
        for op, f in zip(ops[::-1], states[::-1]):
            g.put_f2(f)
            if op == "driftr":
                ref, ref_b = g.op_bwd(op, s, ref, ref_b)
            else:
                ref = g.op_bwd(op, s, ref)
    for a, b, what in ((got, ref, "F2"), (got_b, ref_b, "FGEOS")):
        for s in range(2):
            err = np.abs(a[s] - b[s]).max()
            assert err <= RTOL * np.abs(b[s]).max(), (what, s, err)
    g.close()
