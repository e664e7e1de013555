"""Arena ranges that stay mapped after they are freed: a context of the same
size takes them again, one of another size or many small arrays get their
granules, nothing of an earlier context shows, and the free bytes read as if
every range had been unmapped."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
GRAN = 256 << 20


def _free():
    from openswpc_amd.gpu import stripe_free_bytes
    return [stripe_free_bytes(0, r) for r in range(3)]


def _use(dims, whole):
    """create a context, check that its fields start at zero and hold what is put there"""
    from openswpc_amd.gpu import SwpcGPU
    free0 = _free()
    g = SwpcGPU(*dims, 4, 0)
    taken = sum(free0) - sum(_free())
    assert taken > 0
    if whole:
        assert taken >= 0.9 * g.device_bytes()
    for n in ("Vx", "Sxy"):
        f = g.get_field(n)
        assert not np.any(f)
        f[2, 2::3, 5] = 1.5
        f[-4, 3, 2::7] = -2.0
        g.set_field(n, f)
        assert np.array_equal(g.get_field(n), f)
    g.close()
    assert _free() == free0
    return taken


def test_ranges_are_taken_again_and_given_up():
    from openswpc_amd.gpu import stripe_release, stripe_reserve
    two, three, small = (512, 512, 400), (640, 512, 480), (96, 80, 64)
    stripe_reserve(16 * GRAN)
    try:
        a = _use(two, True)
        assert _use(two, True) == a        # the same ranges again
        b = _use(three, True)              # more granules than were never mapped
        assert b > a
        _use(small, False)
        assert _use(two, True) == a
        assert _use(three, True) == b
    finally:
        stripe_release()
    stripe_reserve(GRAN)                   # every granule went back to the device
    stripe_release()
