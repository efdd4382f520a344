"""Ensembles whose members take kernels of several shapes: the members' lines
together few (all in chunks) and many (the first sweeps by one thread per line,
the last one and the members' own runs in chunks, one member's lines too many
for chunks even alone), planes from one wave to the widest block in one launch,
and persistent grids whose blocks pass from one member's layout to another's.
ram_run must give every member's own F2, records and limits bit for bit, the
adjoint its own gradients to 1e-12 (the misfit and the stale ghosts add
atomically, in any order)."""
import numpy as np
import pytest

from conftest import gpu_available
from helpers import random_problem
from ramgpu import inputs, species as sp
from ramgpu.capi import RamBatch, RamGpu

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="no GPU")]

TOL = 1e-12
H, HO, EH = (sp.HYDROGEN,), (sp.HYDROGEN, sp.OXYGEN), (sp.ELECTRON, sp.HYDROGEN)
FEW = [(H, (4, 4, 4, 4)), (H, (5, 6, 64, 17)), (H, (9, 8, 31, 61)), (HO, (6, 7, 16, 13)), (H, (8, 9, 35, 71))]
MANY = [(H, (4, 30, 48, 48)), (HO, (14, 19, 31, 46)), (H, (5, 6, 64, 90)), (EH, (6, 7, 12, 20)), (H, (17, 9, 20, 33))]
NSTEPS = 3
CAPS = [(0, 0, 0), (37, 41, 29)]


def _problems(members):
    return [random_problem(*grid, species=s, seed=sum(grid)) for s, grid in members]


def _context(p, kp):
    g = RamGpu.from_problem(p)
    g.set_kp(kp)
    return g


def _same_state(g, alone, out, ref, what):
    np.testing.assert_array_equal(g.get_f2(), alone.get_f2(), err_msg=what)
    for s, (a, b) in enumerate(zip(out, ref)):
        assert a == b, (what, s, a, b)


@pytest.mark.parametrize("members", [FEW, MANY], ids=["few", "many"])
def test_steps_equal_members_alone(members):
    probs = _problems(members)
    kp = np.random.default_rng(3).uniform(1.0, 6.0, (NSTEPS, len(probs)))
    alone = [_context(p, 3.0) for p in probs]
    mem = [_context(p, 3.0) for p in probs]
    b = RamBatch(mem)
    b.autotune(reps=1)
    for caps in CAPS:
        b.set_shapes(*caps)
        out = b.ram_run_schedule(kp)
        for m, g in enumerate(alone):
            _same_state(mem[m], g, out[m], g.ram_run_schedule(kp[:, m]), f"member {m}, caps {caps}")
    b.close()
    for g in alone + mem:
        g.close()


@pytest.mark.parametrize("retape", [False, True])
@pytest.mark.parametrize("members", [FEW, MANY], ids=["few", "many"])
def test_adjoint_equals_members_alone(members, retape, monkeypatch):
    if retape:
        monkeypatch.setenv("RAMGPU_ADJOINT_RETAPE", "1")
    probs = _problems(members)
    rng = np.random.default_rng(4)
    kp = rng.uniform(1.0, 6.0, (NSTEPS, len(probs)))
    sats = [inputs.satellite_points(p, 5, seed=m) for m, p in enumerate(probs)]
    pts, w = [s[0] for s in sats], [s[1] for s in sats]
    tgt = [np.log(inputs.satellite_flux(p.f2, *s))[None, :] + 0.1 * rng.standard_normal((NSTEPS, 5))
           for p, s in zip(probs, sats)]
    mem = [_context(p, 3.0) for p in probs]
    b = RamBatch(mem)
    if retape:
        b.set_shapes(*CAPS[1])
    loss, gf, gb = b.adjoint_run(NSTEPS, pts, w, tgt, kp, ckpt_every=2)
    for m, p in enumerate(probs):
        g = _context(p, 3.0)
        l1, f1, b1 = g.adjoint_run(NSTEPS, pts[m], w[m], tgt[m], ckpt_every=2, kp=kp[:, m])
        assert abs(loss[m] - l1) <= TOL * abs(l1), m
        for x, y in ((gf[m], f1), (gb[m], b1)):
            assert np.max(np.abs(x - y)) <= TOL * max(np.max(np.abs(y)), 1e-300), m
        np.testing.assert_array_equal(mem[m].get_f2(), g.get_f2(), err_msg=f"member {m}")
        g.close()
    b.close()
    for g in mem:
        g.close()
