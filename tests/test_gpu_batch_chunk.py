"""The k chunk of batched members: one depth for all that have the default, by
the tiles of the whole batch; a depth set for a member holds; the members' own
launches keep theirs.  Bit for bit under every packing, with PML and Cerjan
members together and the stress streams' accesses of either kind."""
import numpy as np
import pytest

from oracle import oracle as O
from gpu_helpers import compare_fields, gpu_from_model, small_config
from openswpc_amd.gpu import SwpcBatch

pytestmark = pytest.mark.gpu
MT = dict(x=0.3, y=-0.6, z=4.2, t0=0.05, tr=0.8, mo=1e15, strike=30.0, dip=60.0, rake=90.0)
BF = dict(x=-0.7, y=0.4, z=3.3, t0=0.0, tr=0.6, fx=0.3, fy=-1.0, fz=0.5)


@pytest.mark.parametrize("by,variant", [(4, 0), (2, 4), (1, 1)])
@pytest.mark.parametrize("packing", [0, 1, 2])
def test_mixed_members(orc, packing, by, variant):
    nt = 11
    models = [O.build_model(small_config(nt=nt, nm=1, **kw)) for kw in (
        dict(nx=39, ny=35, nz=31, na=7, sources=[MT]), dict(nx=34, ny=29, nz=26, na=5, abc="cerjan", sources=[BF], bf_mode=True),
        dict(nx=66, ny=27, nz=24, na=4, sources=[MT]))]
    sims = [gpu_from_model(m, by=by, variant=variant) for m in models]
    sims[2].set_tuning(5, 0, -1)
    own = [s.tuning() for s in sims]
    batch = SwpcBatch(sims)
    batch.set_packing(packing)
    assert batch.kchunks() == [1, 1, 5] and [s.tuning() for s in sims] == own
    batch.step(1, 8, use_graph=True, block=3)
    sims[0].set_tuning(3, 0, -1)             # a new depth rebuilds the batch's tables
    batch.step(9, nt - 8)
    batch.synchronize()
    assert batch.kchunks() == [3, 1, 5]
    for m, s in zip(models, sims):
        run = O.OracleRun(m, 32)
        run.run(nt)
        for n, (ulp, rel) in compare_fields(s, run).items():
            assert ulp == 0, (n, ulp, rel)
        assert np.array_equal(s.seismograms("vel"), run.wav["vel"])
    batch.close()


@pytest.mark.parametrize("nm,members,depth", [(1, 1, 1), (1, 4, 2), (0, 4, 4)])
def test_depth_by_the_whole_batch(nm, members, depth):
    nt = 9
    m = O.build_model(small_config(nx=128, ny=128, nz=128, na=20, nm=nm, nt=nt, wav_flags=1, sources=[MT]))
    alone = gpu_from_model(m)
    alone.step(1, nt)
    sims = [gpu_from_model(m) for _ in range(members)]
    batch = SwpcBatch(sims)
    assert batch.kchunks() == [depth] * members
    batch.step(1, nt, use_graph=True, block=4)
    batch.synchronize()
    for s in sims:
        assert s.tuning() == alone.tuning()
        for n in O.FIELDS_V + O.FIELDS_S:
            assert np.array_equal(s.get_field(n), alone.get_field(n)), n
    batch.close()
