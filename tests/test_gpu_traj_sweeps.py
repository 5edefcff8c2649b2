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
