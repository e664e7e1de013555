"""Launch variants: the flags that select something (bits 0, 2, 4, 7, 8) with
fewer rows per tile and with outputs to take, and the retired ones (bits 1, 3,
5 and 6), which are accepted and change nothing.  Every form gives the same
bits; the default form is compared with the oracle elsewhere."""
import numpy as np
import pytest

from oracle import oracle as O
from gpu_helpers import gpu_from_model, small_config

pytestmark = pytest.mark.gpu
NT = 9
SECTIONS = ["xy_v", "fs_u", "xz_ps"]


@pytest.fixture(scope="module")
def base(orc):
    rng = np.random.default_rng(5)
    st = [(float(x), float(y), 0.0, "fsb") for x, y in rng.uniform(-3.0, 3.0, (270, 2))]
    m = O.build_model(small_config(nt=NT, nx=45, ny=33, nz=23, na=5, nm=1, zbeg=-1.0, stations=st, wav_flags=11,
                                   sources=[dict(x=0.1, y=-0.1, z=1.6, t0=0.0, tr=0.4, mo=1e15, strike=30.0, dip=60.0, rake=90.0)]))
    cells = [rng.integers(3, n - 2, 280) for n in (45, 33, 23)]
    stf = rng.standard_normal(NT).astype(np.float32)
    return m, cells, stf, _outputs(m, cells, stf)


def _outputs(m, cells, stf, by=0, variant=-1):
    g = gpu_from_model(m, by=by, variant=variant)
    g.set_snapshots(SECTIONS, m.kfs, k0_xy=5, j0_xz=15, ntdec_s=4, nframe=3, M0=m.M0, UC=m.UC)
    g.set_green(*cells, 18, 16, 9, "y", True, 2, 5, stf)
    assert variant < 0 or g.tuning()[1:3] == (by or 4, variant)
    g.step(1, NT, use_graph=True, block=4)
    out = {n: g.get_field(n) for n in O.FIELDS_V + O.FIELDS_S}
    out.update({k: g.seismograms(k) for k in ("vel", "disp", "strain")})
    out.update({(s, f): g.snapshot(s, f) for s in SECTIONS for f in range(3)})
    out.update(green=g.green(), fs=g.snap_max("fs_u"))
    g.close()
    return out


@pytest.mark.parametrize("by,variant", [(1, 0), (2, 0), (1, 1), (4, 4), (2, 4), (1, 5), (2, 5 | 128), (1, 16 | 256),
                                        (4, 1 | 2), (4, 1 | 8), (4, 1 | 32 | 64), (2, 2 | 4 | 8 | 32)])
def test_every_form_gives_the_same_bits(base, by, variant):
    m, cells, stf, want = base
    got = _outputs(m, cells, stf, by, variant)
    for k, v in want.items():
        assert np.any(v != 0) or k[1:] == (0,), k    # frames 0 are taken before the source fires
        assert np.array_equal(got[k], v), k
