"""F2's two layouts at the edges of the transposing tiles (at most 2048
cells, 128 rows of species and rings, 64 energies): less than a tile, whole
tiles, one row or energy more.
A sweep of one species between put and get, compared with the oracle bit for
bit: an error that both directions share would show."""
import numpy as np
import pytest

from conftest import gpu_available
from helpers import random_problem
from oracle.oracle import Oracle
from ramgpu import species as sp
from ramgpu.capi import RamGpu

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="no GPU")]

ALL = (sp.ELECTRON, sp.HYDROGEN, sp.HELIUM, sp.OXYGEN)
# species, (NR, NT, NE, NPA)
CASES = [(1, (4, 4, 4, 4)), (2, (32, 4, 32, 4)), (2, (33, 4, 31, 5)), (4, (32, 4, 5, 4)), (3, (43, 6, 6, 5)),
         (4, (8, 5, 64, 5)), (4, (33, 6, 65, 6)), (1, (5, 4, 129, 4))]


@pytest.mark.parametrize("n,grid", CASES, ids=lambda x: "x".join(map(str, x)) if isinstance(x, tuple) else str(x))
def test_layouts_at_tile_edges(n, grid):
    p = random_problem(*grid, species=ALL[:n], seed=n + sum(grid), spiky=True)
    g, o = RamGpu.from_problem(p), Oracle(p)
    np.testing.assert_array_equal(g.get_f2(), o.f2)
    o.call("cepara", n)
    o.call("driftpara", n)
    o.call("driftr", n)
    g.driftr(n)
    np.testing.assert_array_equal(g.get_f2(), o.f2)
    g.close()
