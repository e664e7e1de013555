"""Chunk boundaries of the interior columns, which weigh a plane of the bottom
absorber against an interior one by what each moves: absorbers thinner and
thicker than the planes above them, every depth that divides them and not, in
step blocks, in the fused launch, by the separate routines and timed (where the
bottom band and the side columns are launches of their own).  Bit for bit against the FP32 oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from gpu_helpers import compare_fields, gpu_from_model, small_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nm", [0, 1, 3])
@pytest.mark.parametrize("nz,na", [(16, 10), (13, 4), (37, 9)])
def test_boundaries(orc, nm, nz, na):
    nt = 8
    m = O.build_model(small_config(nx=35, ny=31, nz=nz, na=na, nm=nm, nt=nt, zbeg=-1.0, wav_flags=1,
                                   sources=[dict(x=0.1, y=-0.1, z=1.1, t0=0.0, tr=0.4, mo=1e15, strike=30.0, dip=60.0, rake=90.0)],
                                   stations=[(1.1, -0.7, 0.0, "fsb")]))
    run = O.OracleRun(m, 32)
    run.run(nt)
    for kchunk in (2, 3, 4, 7, 16, nz + 5):
        for variant in (1, 129):
            g = gpu_from_model(m, kchunk=kchunk, variant=variant)
            g.step(1, 5, use_graph=True, block=5)
            g.wav_store(6)                   # step 6 by the separate routines: the band and the side columns alone
            g.kernel_update_stress()
            g.absorb_update_stress()
            g.source_stressglut(6)
            g.kernel_update_vel()
            g.absorb_update_vel()
            g.source_bodyforce(6)
            g.step_timed(7, nt - 6)
            for n, (ulp, rel) in compare_fields(g, run).items():
                assert ulp == 0, (kchunk, variant, n, ulp, rel)
            assert np.array_equal(g.seismograms("vel"), run.wav["vel"])
            g.close()
