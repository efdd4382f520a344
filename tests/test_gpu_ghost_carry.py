"""DRIFTR's outer ghost carried over more (K,L) planes than a block of the
carry's kernel covers: the only inflow lines are low-energy ones at one local
time, and every outflow line reads the ghost the last of them left."""
import numpy as np
import pytest

from conftest import gpu_available
from helpers import random_problem
from oracle.oracle import Oracle
from ramgpu import species as sp
from ramgpu.capi import RamGpu

JS = 3  # the local time with inflow


def _problem(nr, nt, ne, npa):
    """C(NR) = CR + q1*P4(K)/..: CR > 0 and C(NR-1) < 0 but at JS, where a small
    CR < 0 is outdone by the gradient drift (growing with energy) beyond K=1."""
    p = random_problem(nr, nt, ne, npa, species=(sp.HYDROGEN,), seed=nr + npa, mgnp_frac=0.0)
    g, r = p.geom, p.grid
    p.vt[:] = 0.0
    for a in (g.fnhs, g.fnis):
        a[:] = a[:, :1, :]
    g.bnes[:] = g.bnes[:, :1]
    g.fnis[:, JS + 1, :] += 0.05
    g.eip[:] = 0.01
    g.eip[nr - 2, :] = -0.1
    i = nr - 1
    bsum = g.bnes[i, JS] + g.bnes[i + 1, JS]
    q1 = 0.1 / (g.fnhs[i, JS] + g.fnhs[i + 1, JS])
    p4 = p.dts * r.ekev[0] * 1000.0 * (r.grel[0, 0] + 1.0) / r.grel[0, 0] / r.dphi / r.mdr
    c1 = (q1 * p4 / 2 / bsum / (r.rlz[i] + 0.5 * r.mdr)).max()
    g.eip[i:, JS] = -c1 * bsum / 2 * r.mdr / p.dts
    # cells and boundary of one size, so that the limiter lets the ghost through
    rng = np.random.default_rng(1)
    p.f2[:] = rng.uniform(1.0, 2.0, p.f2.shape)
    p.fgeos[:] = rng.uniform(1.0, 2.0, p.fgeos.shape) / (r.conf1 * g.fnhs[nr - 1][None, :, None, :])
    return p


def _driftr(p):
    o = Oracle(p)
    o.call("driftpara", 1)
    o.call("driftr", 1)
    return o


DIMS = [(6, 8, 24, 64), (5, 9, 70, 30)]


@pytest.mark.parametrize("dims", DIMS, ids=lambda d: "x".join(map(str, d)))
def test_case_is_what_it_says(dims):
    p, q = _problem(*dims), _problem(*dims)
    q.fgeos[0, JS] *= 1.3
    f, h = _driftr(p).f2[0], _driftr(q).f2[0]
    seen = (f != h).any(axis=0)[JS].any(axis=1)  # energies whose lines at JS see their own boundary
    assert seen[0] and (f[:, :JS, -1] != h[:, :JS, -1]).any()
    low = _problem(*dims)
    low.fgeos[0, JS, :8] *= 1.3
    assert np.array_equal(_driftr(low).f2, _driftr(q).f2)  # no inflow beyond K=8


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="no GPU")
@pytest.mark.parametrize("dims", DIMS, ids=lambda d: "x".join(map(str, d)))
def test_carry_reaches_back_over_blocks(dims):
    p = _problem(*dims)
    o, g = _driftr(p), RamGpu.from_problem(p)
    dt = g.driftr(1)
    diff = np.argwhere(g.get_f2() != o.f2)
    assert diff.size == 0, f"{len(diff)} cells differ, first at {diff[0]}"
    assert dt == o.dtdrift()[0, 0]
    g.close()
