"""The field and its slope at the integration limits, which the terminating
terms of low photon energies follow: a limit inside the magnet where the field
crosses zero keeps its slope, and outside the magnet the rounding of the
trajectory's interpolation counts as no field, at any offset and step.

Tolerance: the path's contract, 1e-4 rel-L2 of both components together.  The
crossing edge is compared with the oracle as it is, the field-free ones with
the oracle's edge fields set to zero (their own values are rounding too)."""
import ctypes as C
from array import array

import numpy as np
import pytest

from srw_amd import workloads as W
from srw_amd.srwlib import SRWLMagFldC, SRWLMagFldH, SRWLMagFldU
from tests import oracle_lib as oracle
from tests.util import cfield, clone_wfr

pytestmark = pytest.mark.gpu

TOL = 1e-4


def _error(w, mag, prec, edge_scale=1.):
    from srw_amd import srwlpy
    wg, wo = clone_wfr(w), clone_wfr(w)
    srwlpy.CalcElecFieldSR(wg, 0, mag, prec)
    knob = C.c_double.in_dll(oracle.lib, "orc_edge_field_scale")
    try:
        knob.value = edge_scale
        assert oracle.calc_field(wo, mag, prec) <= 0   # warnings: end terms not computed everywhere
    finally:
        knob.value = 1.
    d = n = 0.
    for c in ("arEx", "arEy"):
        g, o = cfield(getattr(wg, c), wg), cfield(getattr(wo, c), wo)
        d += np.linalg.norm(g - o) ** 2
        n += np.linalg.norm(o) ** 2
    return float(np.sqrt(d / n))


@pytest.mark.parametrize("meth", [0, 1])
@pytest.mark.parametrize("frac", [1e-3, 1e-2])
@pytest.mark.parametrize("n", [1001, 10801, 40001])
def test_limit_where_the_field_crosses_zero(meth, frac, n):
    """An undulator of sine phase integrated from its centre: B = 0 and dB/ds =
    252 T/m at the left limit."""
    print("case: method %d, %g of the first harmonic, %d points" % (meth, frac, n), flush=True)
    und = SRWLMagFldU([SRWLMagFldH(1, 'v', W.undulator_B(1.5, 0.02), 0, -1, 1)], 0.02, 100)
    mag = SRWLMagFldC([und], array('d', [0]), array('d', [0]), array('d', [0]))
    beam = W.electron_beam()
    e = frac * W.first_harmonic_eV(beam.partStatMom1.gamma, 1.5, 0.02)
    w = W.wavefront(beam, 1, e, e, 9, 9)
    err = _error(w, mag, array('d', [meth, 0.01 if meth else 0.108 / (n - 1), 0, 0.108, n, 1, 0]))
    print("rel-L2 %.2e" % err, flush=True)
    assert err < TOL


@pytest.mark.parametrize("x0,y0", [(0., 0.), (1e-4, 0.), (1e-3, 0.), (2e-5, -3e-4)])
@pytest.mark.parametrize("n", [2001, 10001, 100001])
def test_field_free_limits_follow_no_rounding(x0, y0, n):
    print("case: electron at %g, %g m, %d points" % (x0, y0, n), flush=True)
    w = W.wavefront(W.electron_beam(x=x0, y=y0), 1, 0.5, 0.5, 11, 11, 5e-3, 5e-3)
    err = _error(w, W.planar_undulator(), W.traj_prec(n), edge_scale=0.)
    print("rel-L2 %.2e" % err, flush=True)
    assert err < TOL
