"""The gradient's record store after a call that ran out of memory: the store
it left behind holds what earlier arrays left in the arena, and the next call
has to start from a cleared one."""
import numpy as np
import pytest

from oracle import oracle as O
from gpu_helpers import gpu_from_model, small_config

pytestmark = pytest.mark.gpu
GRAN = 256 << 20


def test_store_of_a_failed_call_is_cleared(orc):
    import torch

    from openswpc_amd.gpu import SwpcError, SwpcGPU, stripe_release, stripe_reserve
    nt, ckp = 12, 5
    m = O.build_model(small_config(nx=24, ny=22, nz=20, na=4, nt=nt, nm=0, wav_flags=1))
    obs = np.zeros((m.nst, 3, m.ntw), np.float32)
    good = gpu_from_model(m)
    want = good.adjoint_gradient(nt, obs, ckp=ckp)
    good.close()
    assert np.any(want[1])

    # a trace as large as the rest of the card's memory: its copy cannot be allocated beside it
    total = torch.cuda.mem_get_info()[1]
    nst = 8
    ntw = int(0.55 * total / (12 * nst)) + 1
    assert ntw < 2**31 and 2 * 12 * nst * ntw > total
    stripe_reserve(2 * GRAN)
    try:
        dirty = SwpcGPU(200, 200, 160, 4, 0)
        for n in ("Vx", "Vy", "Vz", "Sxx", "Syy", "Szz", "Syz", "Sxz", "Sxy"):
            dirty.set_field(n, np.full_like(dirty.get_field(n), 7.0))
        dirty.close()
        g = gpu_from_model(m)
        at = np.full(nst, 9, np.int32)
        g.set_receivers(at, at, at, 1, 1, ntw, m.M0, m.UC)
        with pytest.raises(SwpcError, match="device memory for the checkpoints"):
            g.adjoint_accumulate(nt, obs, ckp)
        g.set_receivers(m.ist, m.jst, m.kst, 1, 1, m.ntw, m.M0, m.UC)
        got = g.adjoint_gradient(nt, obs, ckp=ckp)
        g.close()
    finally:
        stripe_release()
    assert got[0] == want[0]
    for a, b in zip(got[1:], want[1:]):
        assert np.array_equal(a, b)
