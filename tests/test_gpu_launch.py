"""Edges of the phase launches: side and interior tiles in one launch on grids
where a tile's rows, columns or planes run out (absorbers of one to twelve
cells, slabs closer together than a tile is tall, a single interior column,
k chunks of one plane up to the default), and the Cerjan taper applied by the
update itself.  Bit for bit against the FP32 oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.gpu_helpers import compare_fields, gpu_from_model, small_config

pytestmark = pytest.mark.gpu
MT = dict(x=0.1, y=-0.1, z=1.6, t0=0.0, tr=0.4, mo=1e15, strike=30.0, dip=60.0, rake=90.0)
BF = dict(x=0.1, y=-0.1, z=1.6, t0=0.0, tr=0.4, fx=0.3, fy=-1.0, fz=0.7)


def _model(**kw):
    cfg = small_config(nt=12, zbeg=-1.0, stations=[], wav_flags=0, **kw)
    return O.build_model(cfg)


def _same(g, run, label):
    for n, (ulp, rel) in compare_fields(g, run).items():
        assert ulp == 0, (label, n, ulp, rel)


@pytest.mark.parametrize("kchunk", [0, 1, 5])
@pytest.mark.parametrize("nx,ny,nz,na", [(13, 70, 14, 6), (70, 13, 14, 6), (9, 9, 12, 4), (67, 66, 12, 1),
                                         (150, 31, 24, 12)])
def test_tile_edges(orc, nx, ny, nz, na, kchunk):
    m = _model(nx=nx, ny=ny, nz=nz, na=na, nm=2, sources=[MT])
    run = O.OracleRun(m, 32)
    run.run(12)
    g = gpu_from_model(m, kchunk=kchunk)
    g.step(1, 12, use_graph=True, block=5)
    _same(g, run, f"{nx}x{ny}x{nz} na={na} kchunk={kchunk}")


@pytest.mark.parametrize("force", [False, True])
@pytest.mark.parametrize("nx,ny,nz,kchunk", [(33, 30, 27, 0), (65, 18, 9, 1), (64, 21, 16, 4), (129, 9, 11, 3)])
def test_taper_applied_by_the_update(orc, nx, ny, nz, kchunk, force):
    m = _model(nx=nx, ny=ny, nz=nz, na=4, nm=1, abc="cerjan", sources=[BF if force else MT], bf_mode=force)
    run = O.OracleRun(m, 32)
    run.run(12)
    g = gpu_from_model(m, kchunk=kchunk)
    g.step(1, 12)
    _same(g, run, "steps")
    # the fused routines against the reference's separate ones
    h = gpu_from_model(m, kchunk=kchunk)
    for it in range(1, 13):
        if it % 2:
            h.update_stress()
        else:
            h.kernel_update_stress()
            h.absorb_update_stress()
        h.source_stressglut(it)
        if it % 2:
            h.kernel_update_vel()
            h.absorb_update_vel()
        else:
            h.update_vel()
        h.source_bodyforce(it)
    for n in O.FIELDS_V + O.FIELDS_S:
        assert np.array_equal(h.get_field(n), g.get_field(n)), n


@pytest.mark.parametrize("nx,ny,nz,na", [(40, 36, 32, 8), (67, 13, 14, 6), (9, 70, 12, 4)])
def test_profiles_replaced_between_steps(orc, nx, ny, nz, na):
    """The auxiliaries of an axis that does not damp a cell are left alone,
    unless they have moved under earlier profiles: a context whose profiles
    are set again after an update of a field at rest takes every auxiliary
    from then on, and both forms agree before and after the damping moves to
    other cells."""
    m = _model(nx=nx, ny=ny, nz=nz, na=na, nm=1, sources=[MT])
    run = O.OracleRun(m, 32)
    run.run(12)
    prof = [m.gxc, m.gxe, m.gyc, m.gye, m.gzc, m.gze]
    moved = [np.roll(p, 3 * 4) for p in prof]   # four numbers a cell
    g, h = gpu_from_model(m), gpu_from_model(m)
    h.update_stress()
    h.set_pml(*prof)
    for c in (g, h):
        c.step(1, 12)
        _same(c, run, f"{nx}x{ny}x{nz} na={na}")
        c.set_pml(*moved)
        c.step(1, 6)
    for n in O.FIELDS_V + O.FIELDS_S:
        assert np.array_equal(h.get_field(n), g.get_field(n)), n


@pytest.mark.parametrize("by,variant", [(0, -1), (2, -1), (0, 0)])
@pytest.mark.parametrize("flags,sections", [(1 | 2 | 8, ["xy_v", "fs_u", "ob_v", "yz_u"]), (15, ["fs_v"]), (3, ["xz_ps", "fs_v"]),
                                            (8, [])])
def test_outputs_in_the_stress_launch(orc, flags, sections, by, variant):
    """Receivers, sections and Green's-function cells, more than one block of
    each, taken by the stress update's launch or beside it, against the same
    step made of the single routines: step blocks in a graph, more than one
    block of them, and the steps left over."""
    nt = 11
    rng = np.random.default_rng(3)
    st = [(float(x), float(y), 0.0, "fsb") for x, y in rng.uniform(-3.0, 3.0, (300, 2))]
    m = O.build_model(small_config(nt=nt, nx=37, ny=34, nz=24, na=5, nm=1, zbeg=-1.0, stations=st, wav_flags=flags, ntdec_w=2,
                                   sources=[MT]))
    cells = [rng.integers(3, n - 2, 290) for n in (37, 34, 24)]
    stf = rng.standard_normal(nt).astype(np.float32)

    def make(**kw):
        g = gpu_from_model(m, **kw)
        if sections:
            g.set_snapshots(sections, m.kfs, k0_xy=5, i0_yz=17, j0_xz=15, ntdec_s=3, nframe=4, M0=m.M0, UC=m.UC)
        g.set_green(*cells, 18, 16, 9, "z", True, 2, 6, stf)
        return g

    g, h = make(by=by, variant=variant), make()
    g.step(1, nt, use_graph=True, block=4)
    for it in range(1, nt + 1):
        h.green_store(it)
        h.wav_store(it)
        if sections:
            h.snap_write(it)
        h.update_stress()
        h.source_stressglut(it)
        h.update_vel()
        h.source_bodyforce(it)
        h.green_source(it)
    kinds = [k for k, bit in (("vel", 1), ("disp", 2), ("stress", 4), ("strain", 8)) if flags & bit]
    for k in kinds:
        assert np.any(h.seismograms(k) != 0)
        assert np.array_equal(g.seismograms(k), h.seismograms(k)), k
    for s in sections:
        for f in range(4):
            assert np.array_equal(g.snapshot(s, f), h.snapshot(s, f)), (s, f)
        if s[:2] in ("fs", "ob") and s[3:] != "ps":
            assert np.array_equal(g.snap_max(s), h.snap_max(s)), s
    assert np.any(h.green() != 0) and np.array_equal(g.green(), h.green())
    for n in O.FIELDS_V + O.FIELDS_S:
        assert np.array_equal(g.get_field(n), h.get_field(n)), n


@pytest.mark.parametrize("at", [None, (0, 0, 0), (12, 20, 18), (-1, -1, -1)])
def test_relaxation_times_without_memory_variables(orc, at):
    """taup and taus are read where one of them is not zero anywhere, halo
    included, and no longer once they are zero again"""
    m = _model(nx=33, ny=30, nz=22, na=5, nm=0, sources=[MT])
    run = O.OracleRun(m, 32)
    run.run(12)
    g = gpu_from_model(m)
    if at is not None:
        for q in (m.taup, m.taus):
            h = gpu_from_model(m)
            tau = [np.zeros_like(m.taup), np.zeros_like(m.taus)]
            tau[0 if q is m.taup else 1][at] = 0.25
            h.set_medium(m.rho, m.lam, m.mu, *tau, m.kfs_top, m.kfs_bot, m.kob_top, m.kob_bot, m.kob)
            h.step(1, 12)
            inside = at == (12, 20, 18)
            assert inside == any(not np.array_equal(h.get_field(n), run.field(n)) for n in O.FIELDS_S)
            h.close()
        g.set_medium(m.rho, m.lam, m.mu, *tau, m.kfs_top, m.kfs_bot, m.kob_top, m.kob_bot, m.kob)
        g.set_medium(m.rho, m.lam, m.mu, m.taup, m.taus, m.kfs_top, m.kfs_bot, m.kob_top, m.kob_bot, m.kob)
    g.step(1, 12)
    _same(g, run, f"tau at {at}")
