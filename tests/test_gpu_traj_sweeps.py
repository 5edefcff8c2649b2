"""The parallel-in-s RK4 with one thread per point (blocks of 256 points per
chain) against the FP64 oracle's serial RK4, at chain lengths around the block
size and with uneven splits at ct = 0.  Tolerance as in test_gpu_traj.py:
1e-9 of each component's magnitude, above the rounding of the summation order
(1e-11) and far below the RK4 truncation error (1e-7)."""
import numpy as np
import pytest

from srw_amd import workloads as W
from tests import oracle_lib as oracle
from tests.test_gpu_traj import REL, _arrays, _traj

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [16, 255, 256, 257, 258, 511, 513, 1025])
@pytest.mark.parametrize("ct0,ct1", [(-0.2, 0.2), (-0.003, 0.3), (-0.3, 0.003), (-0.3, 0.0), (0.0, 0.3)])
def test_chain_lengths_around_a_block(n, ct0, ct1):
    from srw_amd import srwlpy
    print("case:", n, ct0, ct1, flush=True)
    mag = W.planar_undulator()
    kw = dict(x=2e-6, xp=3e-6, y=-1e-6, yp=1e-6)
    tg, to = _traj(n, ct0, ct1, **kw), _traj(n, ct0, ct1, **kw)
    srwlpy.CalcPartTraj(tg, mag)
    assert oracle.calc_traj(to, mag) == 0
    g, o = _arrays(tg), _arrays(to)
    scale = np.maximum(np.max(np.abs(o), axis=1), 1e-30)[:, None]
    assert float(np.max(np.abs(g - o) / scale)) < REL


def _run(n, ct0, ct1, E_GeV, y=0., yp=0., nper=100):
    """The same trajectory by the parallel and the serial kernels, and the sweeps of the two chains."""
    from srw_amd import srwlpy
    mag = W.planar_undulator(nper=nper)
    out = []
    for serial in (False, True):
        t = _traj(n, ct0, ct1)
        t.partInitCond = W.electron_beam(E_GeV, 0.5, 0., 0., y, yp).partStatMom1
        srwlpy.set_traj_serial(serial)
        try:
            srwlpy.CalcPartTraj(t, mag)
        finally:
            srwlpy.set_traj_serial(False)
        if not serial:
            sweeps = srwlpy.last_traj_sweeps()
        out.append(_arrays(t))
    return out[0], out[1], sweeps


# Low energies focus so strongly that the fixed point needs more sweeps than
# are launched.
@pytest.mark.parametrize("E_GeV,ct0,ct1,handed", [
    (3.0, -1.08, 1.08, (False, False)),
    (0.05, -1.08, 1.08, (True, True)),
    (0.05, -0.05, 1.08, (False, True)),
    (0.02, -1.08, 0.05, (True, False)),
])
def test_chains_the_sweeps_leave_unconverged(E_GeV, ct0, ct1, handed):
    """Both chains, or one of them, still moving after the last sweep are
    finished by the one-workgroup solver: the serial kernel's positions."""
    print("case: %g GeV, ct %g to %g" % (E_GeV, ct0, ct1), flush=True)
    g, s, sweeps = _run(4001, ct0, ct1, E_GeV, y=1e-4)
    print("sweeps of the two chains:", sweeps, flush=True)
    assert tuple(k == 0 for k in sweeps) == handed
    scale = np.maximum(np.max(np.abs(s), axis=1), 1e-30)[:, None]
    assert float(np.max(np.abs(g - s) / scale)) < REL


def test_iterates_that_overflow_leave_the_chain_to_the_solver():
    """An electron that leaves the gap: the field's growth off axis overflows
    the iterates and, later, the orbit itself.  Both kernels give the same orbit
    up to where it ends; before it overflows the steps across the last periods
    magnify roundings, so the comparison stops at 5 mm off axis, with 1e-6 of
    each component's magnitude there."""
    print("case: 0.05 GeV, 0.1 rad, ct -0.02 to 1.08", flush=True)
    g, s, sweeps = _run(4001, -0.02, 1.08, 0.05, yp=0.1)
    print("sweeps of the two chains:", sweeps, "finite points:", int(np.isfinite(s).all(0).sum()), flush=True)
    assert sweeps[1] == 0
    assert not np.isfinite(s).all()
    assert np.array_equal(np.isfinite(g), np.isfinite(s))
    ends = np.where(np.isfinite(s).all(0) & (np.abs(s[2]) > 5e-3))[0]
    near = slice(0, int(ends[ends > 100].min()))
    assert near.stop > 200
    scale = np.max(np.abs(s[:, near]), axis=1)[:, None] + 1e-30
    assert float(np.max(np.abs(g[:, near] - s[:, near]) / scale)) < 1e-6
