"""The integrals of the squared angles are zero at the electron's initial
position, interpolated where that lies between two trajectory points (an even
number of points, or a range that is not symmetric about it); their constant is
a phase of the whole field.  Against the FP64 oracle, both components of a field
of several meshes together.

Tolerance: the fields agree to about 1e-6 where the trajectory resolves the
undulator (50 points a period and more); a term of the sums left out is a phase
of 1e-3 and more at these steps, 1e-5 tells them apart.  Every range ends outside
the field: the reference takes the middle of the last interval but one for that
of the last (srtrjdat.cpp:1724-1805), the device the last one's own."""
from array import array

import numpy as np
import pytest

from srw_amd import workloads as W
from srw_amd.srwlib import SRWLMagFldC, SRWLMagFldH, SRWLMagFldU
from tests import oracle_lib as oracle
from tests.util import cfield, clone_wfr

pytestmark = pytest.mark.gpu

TOL = 1e-5


# points, centre of the undulator (its field reaches 0.1 m to both sides), range
CASES = [(1001, 0., None), (1002, 0., None), (1300, 0., None), (1003, 0., (-0.12, 0.1)), (1537, 0., (-0.1, 0.1211)),
         (1026, -0.12, (-0.22, 0.0003)), (1026, 0.12, (-0.0003, 0.22)), (1540, -0.12, (-0.22, 0.)),
         (1541, 0.12, (0., 0.22))]


@pytest.mark.parametrize("meth", [0, 1])
@pytest.mark.parametrize("sym", [1, -1])
@pytest.mark.parametrize("n,zc,lim", CASES)
def test_phase_with_the_origin_between_points(n, zc, lim, sym, meth):
    from srw_amd import srwlpy
    print("case:", n, zc, lim, sym, meth, flush=True)
    per, nper = 0.01, 12
    half = per * (0.5 * nper + 4)
    und = SRWLMagFldU([SRWLMagFldH(1, 'v', W.undulator_B(1.5, per), 0, sym, 1)], per, nper)
    mag = SRWLMagFldC([und], array('d', [0]), array('d', [0]), array('d', [zc]))
    beam = W.electron_beam(x=1e-5, y=-2e-5, yp=3e-6)
    e = 0.9 * W.first_harmonic_eV(beam.partStatMom1.gamma, 1.5, per)
    a, b = lim if lim else (-half, half)
    prec = array('d', [meth, 0.005 if meth else (b - a) / (n - 0.5), lim[0] if lim else 0, lim[1] if lim else 0, n, 1, 0])
    for nx, ny in ((4, 3), (40, 36)):
        w = W.wavefront(beam, 1, e, e, nx, ny, 3e-4, 3e-4, 20.)
        wg, wo = clone_wfr(w), clone_wfr(w)
        srwlpy.CalcElecFieldSR(wg, 0, mag, prec)
        assert oracle.calc_field(wo, mag, prec) <= 0
        g, o = (np.stack([cfield(v.arEx, v), cfield(v.arEy, v)]) for v in (wg, wo))
        err = np.linalg.norm(g - o) / np.linalg.norm(o)
        print("%d x %d rel-L2 %.2e" % (nx, ny, err), flush=True)
        assert err < TOL
