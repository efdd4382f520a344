"""DRIFTR and DRIFTP with a line's cells cut into chunks, at the edges of the
mapping: one chunk and many, a ragged last chunk, a chunk of the line's last
two cells, waves partly filled, lines too long for chunks.  Each operator is
compared bit for bit with the oracle, the last sweep of a step (seam, mask,
SUMRC) through ram_run."""
import numpy as np
import pytest

from conftest import gpu_available
from helpers import max_rel_err, random_problem
from oracle.oracle import Oracle
from ramgpu import species as sp
from ramgpu.capi import RamGpu

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="no GPU")]

RTOL = 1e-12  # the step's tolerance (tests/test_gpu_parity.py): the loss factors' exponentials

# (NR, NT, NE, NPA)
GRIDS = [(4, 4, 4, 4), (5, 5, 4, 5), (6, 7, 7, 9), (8, 9, 8, 8), (9, 8, 5, 13), (10, 13, 11, 17), (17, 16, 8, 10),
         (33, 25, 4, 16), (32, 33, 5, 13), (41, 49, 4, 6), (12, 129, 16, 8), (127, 12, 4, 5), (130, 11, 5, 4),
         (11, 130, 16, 8)]


@pytest.mark.parametrize("grid", GRIDS, ids=lambda g: "x".join(map(str, g)))
def test_line_sweeps_at_mapping_edges(grid):
    p = random_problem(*grid, species=(sp.ELECTRON, sp.OXYGEN), seed=sum(grid), spiky=True)
    g = RamGpu.from_problem(p)
    o = Oracle(p)
    for s in (1, 2):
        o.call("cepara", s)
        o.call("driftpara", s)
        for op in ("driftr", "driftp", "driftp", "driftr"):
            o.call(op, s)
            dt = getattr(g, op)(s)
            diff = np.argwhere(g.get_f2() != o.f2)
            assert diff.size == 0, f"{op}(S={s}): {len(diff)} cells differ, first at {diff[0]}"
            assert dt == o.dtdrift()[s - 1, ["driftr", "driftp"].index(op)], (op, s)
    g.close()
    g, o = RamGpu.from_problem(p), Oracle(p)
    out = g.ram_run(1)
    o.ram_run()
    assert max_rel_err(g.get_f2(), o.f2) <= RTOL
    for s in range(2):
        for k in ("setrc", "lsdr"):
            assert abs(out[s][k] - o.arr(k)[s]) <= RTOL * abs(o.arr("setrc")[s]), (s, k)
    g.close()


def test_recording_out_of_place_sweep_keeps_every_species_limit():
    # out of place (the taped step), DRIFTP's launch has more blocks than any
    # other kernel, those that copy the I=1 rows; the CFL maxima it records
    # must be the in-place sweep's
    p = random_problem(4, 48, 64, 90, species=(sp.ELECTRON, sp.HYDROGEN, sp.HELIUM, sp.OXYGEN), seed=7)
    a, b = RamGpu.from_problem(p), RamGpu.from_problem(p)
    a.ram_run_bwd(np.ones_like(p.f2))  # records the limits on its taped step
    ra, rb = a.ram_run(1), b.ram_run(1)
    for s in range(4):
        for k in ("dtdrift_r", "dtdrift_p", "dtdrift_e", "dtdrift_mu"):
            assert ra[s][k] == rb[s][k], (s, k)
    a.close()
    b.close()
