"""The matrix-product SR kernel (64 x 64 point tiles of four 32 x 32 parts,
integration points in groups of 8 and units of 32) against the FP64 oracle, at
mesh sizes around the tile, at integration ranges around the group and the
unit, and on both sides of the rule that chooses it.

Tolerance: a term carries about 2e-7 of its magnitude (phase, sine, FP16 pair)
and the terms add like a random walk, so a field that is not far below the sum
of its terms agrees to about 1e-6; 1e-5 rel-L2 of both components together
leaves a factor of 10 and is a tenth of the path's contract (1e-4)."""
import numpy as np
import pytest

from srw_amd import workloads as W
from tests import oracle_lib as oracle
from tests.util import cfield, clone_wfr

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _error(w, mag, prec):
    from srw_amd import srwlpy
    wg, wo = clone_wfr(w), clone_wfr(w)
    srwlpy.CalcElecFieldSR(wg, 0, mag, prec)
    assert oracle.calc_field(wo, mag, prec) == 0
    d = n = 0.
    for c in ("arEx", "arEy"):
        g, o = cfield(getattr(wg, c), wg), cfield(getattr(wo, c), wo)
        d += np.linalg.norm(g - o) ** 2
        n += np.linalg.norm(o) ** 2
    return float(np.sqrt(d / n))


def _case(nx, ny, ne=1, nper=12, np_traj=1201, tilt=False):
    kw = dict(x=2e-5, xp=3e-6, y=-1e-5, yp=1e-6) if tilt else {}
    beam = W.electron_beam(**kw)
    e = W.first_harmonic_eV(beam.partStatMom1.gamma, 1.5, 0.02)
    w = W.wavefront(beam, ne, 0.99 * e, 1.01 * e if ne > 1 else 0.99 * e, nx, ny, 1e-3, 0.7e-3, 20.)
    return w, W.planar_undulator(1.5, 0.02, nper), W.traj_prec(np_traj, nper=nper)


@pytest.mark.parametrize("nx,ny", [(32, 32), (33, 65), (64, 64), (65, 63), (128, 31), (40, 97), (16, 16), (200, 5),
                                   (22, 23), (23, 23), (12, 300)])
def test_mesh_sizes_around_a_tile(nx, ny):
    """16 x 16, 200 x 5 and 22 x 23 fill less than an eighth of their tiles: the
    one-lane kernel."""
    print("case:", nx, ny, flush=True)
    e = _error(*_case(nx, ny, tilt=True))
    print("rel-L2 %.2e" % e, flush=True)
    assert e < TOL


@pytest.mark.parametrize("n", [9, 31, 33, 35, 65, 67, 129])
def test_integration_points_around_a_unit(n):
    """n integration points: the step lies between the values at which the
    count changes, where its rounding would decide the count."""
    print("case:", n, flush=True)
    w, mag, prec = _case(48, 40, nper=1, np_traj=301, tilt=True)
    prec[1] = 2. * (0.5 * 0.02 + 4 * 0.02) / (n - 0.5)
    e = _error(w, mag, prec)
    print("rel-L2 %.2e" % e, flush=True)
    assert e < TOL


@pytest.mark.parametrize("ne", [3, 8, 11])
def test_several_energies_and_mirror_symmetry(ne):
    print("case:", ne, flush=True)
    e = _error(*_case(70, 45, ne=ne))
    print("rel-L2 %.2e" % e, flush=True)
    assert e < TOL


def test_batch_mixes_both_kernels():
    """Requests on both sides of the rule in one batch, against single calls."""
    from srw_amd import srwlpy
    ws, ms, prec = [], [], None
    for nx, ny in ((64, 40), (12, 9), (33, 100), (150, 2)):
        w, m, prec = _case(nx, ny, tilt=True)
        ws.append(w)
        ms.append(m)
    wb = [clone_wfr(w) for w in ws]
    srwlpy.CalcElecFieldSRBatch(wb, ms, prec)
    for w, m, b in zip(ws, ms, wb):
        srwlpy.CalcElecFieldSR(w, 0, m, prec)
        g, o = cfield(b.arEx, b), cfield(w.arEx, w)
        assert np.linalg.norm(g - o) < 1e-6 * np.linalg.norm(o)


@pytest.mark.parametrize("nx,ny,ne", [(64, 64, 1), (70, 45, 11), (150, 93, 3)])
def test_agrees_with_one_lane_per_point(nx, ny, ne):
    """The same mesh with the kernel on and off.  Tolerance: twice TOL's share of
    a kernel, 1e-6 of rounding each (see above), with the factor of 10 shared."""
    from srw_amd import srwlpy
    print("case:", nx, ny, ne, flush=True)
    w, mag, prec = _case(nx, ny, ne=ne, tilt=True)
    got = []
    for on in (True, False):
        wg = clone_wfr(w)
        srwlpy.set_mesh_kernel(on)
        try:
            srwlpy.CalcElecFieldSR(wg, 0, mag, prec)
        finally:
            srwlpy.set_mesh_kernel(True)
        got.append(np.stack([cfield(wg.arEx, wg), cfield(wg.arEy, wg)]))
    d = np.linalg.norm(got[0] - got[1]) / np.linalg.norm(got[1])
    print("rel-L2 %.2e" % d, flush=True)
    assert 0 < d < TOL


@pytest.mark.parametrize("harm,step,half", [(1, 16, 1e-4), (5, 4, 1e-4), (9, 2, 1e-4), (9, 4, 1e-4), (15, 2, 1e-5),
                                            (9, 4, 1e-3)])
def test_errors_no_larger_than_one_lane_per_point(harm, step, half):
    """Harmonics and steps at which the phase turns by 0.5 to 3 revolutions over 4
    steps: the errors against FP64 at most 1.2 of those with the kernel off."""
    from srw_amd import srwlpy
    print("case: harmonic %d, step x %d, half %g m" % (harm, step, half), flush=True)
    beam = W.electron_beam(x=2e-6, y=1e-6)
    e = harm * 0.995 * W.first_harmonic_eV(beam.partStatMom1.gamma, 1.5, 0.02)
    w = W.wavefront(beam, 1, e, e, 48, 40, half, half, 20.)
    prec = W.traj_prec(10001)
    prec[1] *= step
    got = []
    for on, tol in ((True, 0.), (False, 0.), (True, 1e-12)):
        wg = clone_wfr(w)
        srwlpy.set_mesh_kernel(on)
        srwlpy.set_cond_tol(tol)
        try:
            srwlpy.CalcElecFieldSR(wg, 0, W.planar_undulator(), prec)
        finally:
            srwlpy.set_mesh_kernel(True)
            srwlpy.set_cond_tol(1e-4)
        got.append(np.stack([cfield(wg.arEx, wg), cfield(wg.arEy, wg)]))
    mesh, lane = (np.linalg.norm(g - got[2]) / np.linalg.norm(got[2]) for g in got[:2])
    print("kernel on %.2e, off %.2e" % (mesh, lane), flush=True)
    assert mesh <= 1.2 * lane


@pytest.mark.parametrize("small,ne", [((1, 1), 1), ((1, 3), 9), ((9, 1), 1)])
def test_small_request_among_meshes_keeps_the_parts(small, ne):
    """One request off the mesh kernel in a batch of large meshes: the partial
    sums, which hold every point of the batch once per part of the s-range, stay
    within 16384 blocks of 256 points."""
    from srw_amd import srwlpy
    print("case: 6 meshes of 256 x 256 and one of %d x %d x %d" % (small[0], small[1], ne), flush=True)
    reqs = [_case(256, 256, ne if k % 2 else 1, tilt=True, np_traj=4001) for k in range(6)]
    reqs.append(_case(small[0], small[1], ne, tilt=True, np_traj=4001))
    ws, ms, prec = [r[0] for r in reqs], [r[1] for r in reqs], reqs[0][2]
    wb = [clone_wfr(w) for w in ws]
    srwlpy.CalcElecFieldSRBatch(wb, ms, prec)
    st = srwlpy.stats()
    print("%d blocks in %d parts" % (st["sr_blocks"], st["sr_split"]), flush=True)
    assert st["sr_blocks"] * st["sr_split"] <= 16384
    for k in (0, 1, 6):
        srwlpy.CalcElecFieldSR(ws[k], 0, ms[k], prec)
        g, o = cfield(wb[k].arEx, wb[k]), cfield(ws[k].arEx, ws[k])
        assert np.linalg.norm(g - o) < 1e-6 * np.linalg.norm(o)


@pytest.mark.parametrize("nx,ny,ne", [(70, 300, 60), (33, 600, 64), (300, 65, 70), (64, 130, 140)])
def test_streamed_tile_rows_equal_one_pass(nx, ny, ne):
    """Fields of 16 MB or more, without mirror symmetry: the sums launched by
    tile rows with the finished rows' copies beside them, against one launch
    and one copy.  The s-range is cut alike, so the fields are the same bits.
    33 x 600 reaches so far off axis that the points recomputed in FP64 are more
    than the streamed copy patches, and the whole field is copied again."""
    from srw_amd import srwlpy
    print("case: %d x %d x %d streamed tile rows" % (nx, ny, ne), flush=True)
    w, mag, prec = W.single_electron(n=nx, ne=ne, de_rel=0.02)
    p = w.partBeam.partStatMom1
    p.x, p.y, p.xp, p.yp = 20e-6, 10e-6, 3e-6, 2e-6
    span = w.mesh.yFin - w.mesh.yStart
    w.allocate(ne, nx, ny)
    w.mesh.yFin = w.mesh.yStart + span * ny / nx * 0.5
    got = []
    for bands in (1, 0):
        wg = clone_wfr(w)
        srwlpy.set_bands(bands)
        try:
            srwlpy.CalcElecFieldSR(wg, 0, mag, prec)
        finally:
            srwlpy.set_bands(0)
        fp64 = int(srwlpy.stats()["sr_fp64_points"])
        print("bands %d: streamed %s, FP64 points %d" % (bands, srwlpy.last_streamed(), fp64), flush=True)
        overflow = fp64 > 1 << 18
        assert overflow == ((nx, ny) == (33, 600))
        assert srwlpy.last_streamed() == (bands == 0 and not overflow)
        got.append([np.frombuffer(getattr(wg, c), np.float32) for c in ("arEx", "arEy")])
    for a, b in zip(*got):
        assert np.isfinite(a).all() and np.abs(a).max() > 0
        assert np.array_equal(a, b)


@pytest.mark.parametrize("e_ev,step,half", [(1e6, 40, 1e-5), (1e6, 10, 1e-5), (1e7, 10, 1e-5), (1e5, 40, 1e-5),
                                            (1e5, 2, 1e-5), (1e5, 1, 1e-4), (1e6, 40, 1e-3), (1.6e3, 1, 5e-2)])
def test_coarse_steps_keep_the_phase(e_ev, step, half):
    """Photon energies and steps at which the phase turns by 1 to 2000
    revolutions over 4 steps, on both sides of the rule that takes the kernel,
    and a mesh far off axis: every point against its own FP64 recomputation.
    Tolerance: the condition check's, 1e-4 of a point's field."""
    from srw_amd import srwlpy
    print("case: %g eV, step x %g, half %g m" % (e_ev, step, half), flush=True)
    w = W.wavefront(W.electron_beam(x=2e-6, y=1e-6), 1, e_ev, e_ev, 40, 40, half, half, 20.)
    prec = W.traj_prec(10001)
    prec[1] *= step
    got = []
    for tol in (1e-4, 1e-12):
        wg = clone_wfr(w)
        srwlpy.set_cond_tol(tol)
        try:
            srwlpy.CalcElecFieldSR(wg, 0, W.planar_undulator(), prec)
        finally:
            srwlpy.set_cond_tol(1e-4)
        got.append(np.stack([cfield(wg.arEx, wg), cfield(wg.arEy, wg)]))
    err = np.sqrt((np.abs(got[0] - got[1]) ** 2).sum(0) / (np.abs(got[1]) ** 2).sum(0))
    print("worst %.2e, rel-L2 %.2e" % (err.max(), np.linalg.norm(got[0] - got[1]) / np.linalg.norm(got[1])), flush=True)
    assert err.max() < 1e-4
