"""F2's two layouts on both sides of the rule that chooses between tiles and a
thread per cell (NS*NR*NE of 320; 1.2 MB out, 4.4 MB in; 13 MB for planes of a
multiple of 2048 cells): a get after a put returns the array, and DRIFTR between them equals the oracle's bit for bit."""
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
# species, (NR, NT, NE, NPA): rows of 316 and 320 cells; 1.17, 1.23, 4.35, 4.49 MB; 12.8 and 13.1 MB
CASES = [(1, (4, 48, 79, 60)), (1, (4, 48, 80, 60)), (2, (5, 24, 32, 19)), (2, (5, 24, 32, 20)), (4, (4, 29, 32, 37)),
         (4, (4, 29, 33, 37)), (4, (7, 28, 32, 64)), (4, (8, 25, 32, 64)), (1, (4, 4, 4, 4))]


@pytest.mark.parametrize("n,grid", CASES, ids=lambda x: "x".join(map(str, x)) if isinstance(x, tuple) else str(x))
def test_layouts_at_the_rule(n, grid):
    p = random_problem(*grid, species=ALL[:n], seed=n + sum(grid))
    g, o = RamGpu.from_problem(p), Oracle(p)
    np.testing.assert_array_equal(g.get_f2(), o.f2)
    o.call("cepara", n)
    o.call("driftpara", n)
    o.call("driftr", n)
    g.driftr(n)
    np.testing.assert_array_equal(g.get_f2(), o.f2)
    g.close()
