"""The adjoint kernels where their tiles, their neighbour words and their
shared densities change kind: ragged grids around the 64-cell tile width, one
to three interior cells between the absorbing zones, a seawater band, and a
different spacing along each axis; against the FP64 oracle adjoint.

Tolerance, set before the first run: the FP32 gradient is a sum over nt = 40
steps of products of fields that each carry the rounding of as many steps,
about nt * 2^-24 = 2.4e-6 of the largest value with a factor of some tens for
the nine-term sums; 1e-4 of the largest value, as for the other gradients.
"""
import numpy as np
import pytest

from oracle import oracle as O
from gpu_helpers import gpu_from_model
from test_oracle_adjoint import OCEAN, _cfg, _visco

pytestmark = pytest.mark.gpu

OFF = O.OFF


@pytest.mark.parametrize("nx,ny,nz,na,nm,ocean", [
    (67, 21, 18, 5, 0, True), (63, 13, 19, 5, 3, True), (64, 11, 15, 4, 0, False),
    (66, 9, 17, 4, 1, False), (10, 68, 16, 4, 2, False),
])
def test_gradient_at_tile_and_zone_edges(orc, nx, ny, nz, na, nm, ocean):
    nt = 40
    kw = dict(nx=nx, ny=ny, nz=nz, na=na, nt=nt, wav_flags=1, dt=0.02, dx=0.5, dy=0.45, dz=0.55)
    if ocean:
        kw.update(OCEAN)
    m = O.build_model(_cfg(**kw) if nm == 0 else _visco(nm=nm, **kw))
    rng = np.random.default_rng(11)
    d = O.OracleAdjoint(m, 64).forward(nt, keep=False)
    d_obs = d * (1 + 0.3 * rng.standard_normal(d.shape)) + 0.1 * np.abs(d).max() * rng.standard_normal(d.shape)
    J, g, _ = O.misfit_and_gradient(m, nt, d_obs)
    obs = np.ascontiguousarray(d_obs.transpose(1, 2, 0), np.float32)
    gpu = gpu_from_model(m)
    Jg, *got = gpu.adjoint_gradient(nt, obs, ckp=11)
    gpu.close()
    assert abs(Jg - J) <= 1e-4 * J
    cells = (slice(OFF + 1, OFF + 1 + nz), slice(OFF + 1, OFF + 1 + nx), slice(OFF + 1, OFF + 1 + ny))
    for name, a, b in zip(("lam", "mu", "rho"), got, g):
        a, b = a.astype(np.float64), np.asarray(b, np.float64)
        assert np.abs(b).max() > 0.0
        err = np.abs(a - b).max() / np.abs(b).max()
        assert err < 1e-4, (name, err)
