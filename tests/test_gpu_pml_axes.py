"""When the updates leave the PML auxiliaries of undamped axes alone: only
steps that ran and profiles that undamp an axis of a cell take every auxiliary
from then on; making a batch, tuning it or setting the same profiles again do
not.  Both forms give the oracle's bits."""
import numpy as np
import pytest

from oracle import oracle as O
from gpu_helpers import compare_fields, gpu_from_model, small_config

pytestmark = pytest.mark.gpu


def _model(nx=41, ny=35, nz=29, na=7):
    return O.build_model(small_config(nx=nx, ny=ny, nz=nz, na=na, nt=10, nm=1, wav_flags=1))


def _profiles(m):
    return [m.gxc, m.gxe, m.gyc, m.gye, m.gzc, m.gze]


def _undamped(p, n):
    """the profiles with cell n (from 0) of the x axis undamped"""
    q = [a.copy() for a in p]
    for a in q[:2]:
        a.reshape(-1, 4)[n] = (1.0, 0.0, 0.0, 0.0)
    return q


def _same(g, run, label):
    for n, (ulp, rel) in compare_fields(g, run).items():
        assert ulp == 0, (label, n, ulp, rel)


def test_filled_arguments_move_nothing(orc):
    from openswpc_amd.gpu import SwpcBatch
    m = _model()
    run = O.OracleRun(m, 32)
    run.run(10)
    sims = [gpu_from_model(m) for _ in range(2)]
    batch = SwpcBatch(sims)                  # builds the members' arguments and tables
    for s in sims:
        s.set_pml(*_undamped(_profiles(m), 2))
        assert s.pml_axes_skipped()          # nothing has been stepped
        s.set_pml(*_profiles(m))
    batch.tune(1)
    for s in sims:
        s.set_pml(*_profiles(m))
        assert s.pml_axes_skipped()          # the same profiles
    batch.step(1, 10)
    batch.synchronize()
    for s in sims:
        s.set_pml(*_profiles(m))
        assert s.pml_axes_skipped()
        _same(s, run, "batch")
    batch.close()


@pytest.mark.parametrize("by_graph", [False, True])
def test_undamped_after_a_step_takes_them_all(orc, by_graph):
    m = _model()
    run = O.OracleRun(m, 32)
    run.run(10)
    p = _profiles(m)
    more = _undamped(p, 0)                   # x damps in cells 1 to na: one less
    g, h = gpu_from_model(m), gpu_from_model(m)
    h.update_stress()                        # of a field at rest
    h.set_pml(*more)
    assert not h.pml_axes_skipped()
    h.set_pml(*p)
    assert not h.pml_axes_skipped()          # until a gradient starts from rest
    for c, skipped in ((g, True), (h, False)):
        c.step(1, 10, use_graph=by_graph, block=3)
        assert c.pml_axes_skipped() == skipped
        _same(c, run, skipped)
        c.set_pml(*more)                     # the auxiliaries of cell 1 are not zero
        assert not c.pml_axes_skipped()
        c.step(1, 7, use_graph=by_graph, block=3)
    for n in O.FIELDS_V + O.FIELDS_S:
        assert np.array_equal(g.get_field(n), h.get_field(n)), n
    obs = np.zeros((m.nst, 3, m.ntw), np.float32)
    J = [c.adjoint_gradient(10, obs, ckp=4)[0] for c in (g, h)]
    assert J[0] == J[1] > 0
    for c in (g, h):
        assert c.pml_axes_skipped()
        c.set_pml(*more)                     # damped in no step since the gradient started
        assert c.pml_axes_skipped()
        c.set_pml(*p)
        c.set_pml(*p)
        assert c.pml_axes_skipped()


def test_damping_more_keeps_them_skipped(orc):
    m = _model()
    p = _profiles(m)
    g = gpu_from_model(m)
    g.set_pml(*_undamped(p, 1))
    g.step(1, 5)
    g.set_pml(*p)                            # an axis more than the steps ran with
    assert g.pml_axes_skipped()
    g.set_pml(*_undamped(p, 1))
    assert g.pml_axes_skipped()              # no step ran with it
    g.set_pml(*p)
    g.step(6, 5)
    g.set_pml(*_undamped(p, 1))
    assert not g.pml_axes_skipped()


def test_no_pml_has_none(orc):
    m = O.build_model(small_config(nx=30, ny=28, nz=26, na=5, nt=4, nm=0, abc="cerjan", wav_flags=0, stations=[]))
    assert not gpu_from_model(m).pml_axes_skipped()
