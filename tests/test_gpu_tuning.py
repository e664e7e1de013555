"""The launch shape in use: what swpc_get_tuning reports, and that the fused
launch takes a depth of its own by default (each of its chunks computes the
velocities of four planes more than it updates) and the caller's otherwise."""
import numpy as np
import pytest

from openswpc_amd import gpu
from oracle import oracle as O
from gpu_helpers import compare_fields, gpu_from_model, small_config

CUS = 256   # of an MI355X


def test_null_context_has_no_tuning():
    L = gpu.load_library()
    assert L.swpc_get_tuning(None, None, None, None, None) == -1
    assert L.swpc_pml_axes_skipped(None) == -1


def _fused_default(nx, ny, nz, na, rows):
    tiles = -(-(nx - 2 * na) // 60) * -(-(ny - 2 * na) // rows)
    kc = 16
    while kc > 1 and tiles * -(-(nz - na) // kc) < (5 if rows == 8 else 7) / 4 * CUS:
        kc //= 2
    return kc


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny,nz,na,nm", [(20, 19, 17, 4, 0), (96, 96, 96, 10, 2), (128, 128, 128, 20, 3),
                                            (256, 200, 160, 20, 0)])
def test_fused_launch_has_its_own_default_depth(nx, ny, nz, na, nm):
    g = gpu.SwpcGPU(nx, ny, nz, na, nm)
    kc = g.tuning()[0]
    four, eight = (_fused_default(nx, ny, nz, na, rows) for rows in (4, 8))
    assert g.tuning() == (kc, 4, 1, four) and 1 <= kc <= 16
    if (nx, nm) == (128, 3):
        assert (kc, four) == (2, 8)      # 3 velocity planes per stress plane at 2
    g.set_tuning(0, 2, 128 | 256 | 1)
    assert g.tuning() == (kc, 2, 385, eight)
    g.set_tuning(5, 0, -1)
    assert g.tuning() == (5, 2, 385, 5)
    g.set_tuning(-1, 4, 1)
    assert g.tuning() == (kc, 4, 1, four)
    g.close()


@pytest.mark.gpu
@pytest.mark.parametrize("variant", [129, 385])
@pytest.mark.parametrize("nx,ny,nz,na", [(40, 36, 32, 8), (131, 23, 45, 5)])
def test_fused_steps_at_the_default_depth(orc, nx, ny, nz, na, variant):
    m = O.build_model(small_config(nx=nx, ny=ny, nz=nz, na=na, nm=1, nt=13, wav_flags=1))
    run = O.OracleRun(m, 32)
    run.run(13)
    g = gpu_from_model(m, variant=variant)
    g.step(1, 13, use_graph=True, block=5)
    for n, (ulp, rel) in compare_fields(g, run).items():
        assert ulp == 0, (n, ulp, rel)
    assert np.array_equal(g.seismograms("vel"), run.wav["vel"])
