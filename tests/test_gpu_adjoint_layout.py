"""The arrays in which adjoint_run returns dL/dFGEOS: one C-contiguous
(nsteps,NS,NT,NE,NPA) array from RamGpu, Fortran-ordered steps from RamBatch,
both with the values of the C ABI's Fortran-ordered ones (to 1e-12: two runs
add the stale ghosts' terms atomically, in any order); at the edges of the
reordering tiles (64 columns S,J,K by 32 L) and with more steps than the tape
holds at a time (10 NR a step of a segment)."""
import ctypes as C

import numpy as np
import pytest

from conftest import gpu_available
from helpers import random_problem
from ramgpu import species as sp
from ramgpu.capi import RamBatch, RamGpu, _p

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="no GPU")]

TOL = 1e-12

# species, (NR, NT, NE, NPA), steps: less than a tile, whole tiles, one more in each direction; more than 80 steps of NR = 4
CASES = [(1, (5, 4, 4, 5), 3), (1, (4, 8, 8, 32), 9), (2, (4, 5, 13, 33), 4), (3, (5, 7, 9, 64), 11), (2, (6, 8, 20, 13), 2),
         (1, (4, 4, 5, 6), 83)]


@pytest.mark.parametrize("ns,grid,nsteps", CASES, ids=lambda v: "x".join(map(str, v)) if type(v) is tuple else str(v))
def test_fgeos_gradient_layout(ns, grid, nsteps):
    p = random_problem(*grid, species=(sp.HYDROGEN, sp.OXYGEN, sp.HELIUM)[:ns], seed=sum(grid))
    # a point at every (S, J, K) of the outer ring, which the boundary feeds
    nr, nt, ne, npa = grid
    pts = np.array([(s + 1, nr, j + 1, k + 1) for s in range(ns) for j in range(nt) for k in range(ne)], dtype=np.int32)
    w = np.random.default_rng(1).uniform(0.5, 1.5, (len(pts), npa))
    target = np.zeros((nsteps, len(pts)))

    g = RamGpu.from_problem(p)
    loss, gf, gb = g.adjoint_run(nsteps, pts, w, target, ckpt_every=2)
    assert gb.shape == (nsteps, ns) + grid[1:]
    assert gb.flags.c_contiguous and gb.flags.owndata and gb.flags.writeable

    g.put_f2(p.f2)
    flat = np.full(gb.size, np.nan)
    l2, gf2 = C.c_double(), np.zeros(g.dims, order="F")
    assert g.lib.ramgpu_adjoint_run(g.h, nsteps, 2, None, None, len(pts), pts.ctypes.data_as(C.POINTER(C.c_int)), _p(w),
                                    _p(target), C.byref(l2), _p(gf2), _p(flat)) == 0
    ref = np.stack([a.reshape(gb.shape[1:], order="F") for a in np.split(flat, nsteps)])
    assert abs(loss - l2.value) <= TOL * abs(loss)
    assert np.count_nonzero(ref) > 0
    for a, b in ((gf, gf2), (gb, ref)):
        assert np.linalg.norm((a - b).ravel()) <= TOL * np.linalg.norm(b.ravel())
        assert np.array_equal(a == 0, b == 0)

    g.put_f2(p.f2)
    g.set_kp(p.kp)
    b = RamBatch([g])
    _, _, gbs = b.adjoint_run(nsteps, [pts], [w], [target], np.full((nsteps, 1), p.kp), ckpt_every=2)
    assert all(a.flags.f_contiguous for a in gbs[0])
    b.close()
    g.close()
