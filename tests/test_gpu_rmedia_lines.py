"""Random media through the line transforms and through hipFFT at the edges of
both: prime, odd and power-of-two lengths, lines that leave a block's last
columns or rows empty, lengths for which a block takes eight, four, two or
one lines, and lengths that no block takes; against the same algorithm in float64
on the host with the same noise.

Tolerance, set before the first run: both transforms are in double precision,
and a whitened value moves by the transform's rounding over its size before
whitening, about 1e-15 * sqrt(cells) * 1e3 for the smallest of a few 1e5
values; the field is rounded to float32, 6e-8 of its largest value.  1e-6 of
the largest value.
"""
import numpy as np
import pytest

from openswpc_amd.gpu import rmedia_3d

pytestmark = pytest.mark.gpu


def _mix(z):
    with np.errstate(over="ignore"):
        z = z + np.uint64(0x9E3779B97F4A7C15)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        return z ^ (z >> np.uint64(31))


def _host(ptype, shape, d, a, eps, kappa, seed):
    n1, n2, n3 = shape
    q = np.arange(n1 * n2 * n3, dtype=np.uint64)
    noise = (_mix(_mix(np.array([seed], np.uint64)) ^ q) >> np.uint64(11)).astype(np.float64) * 2.0 ** -53
    b = np.fft.rfftn(noise.reshape(n3, n2, n1))
    f32 = [float(np.float32(v)) for v in (*d, *a)]
    k3, k2 = (2 * np.pi * np.fft.fftfreq(n, h) for n, h in ((n3, f32[2]), (n2, f32[1])))
    k1 = 2 * np.pi * np.fft.rfftfreq(n1, f32[0])
    q2 = (k3 * f32[5])[:, None, None] ** 2 + (k2 * f32[4])[None, :, None] ** 2 + (k1 * f32[3])[None, None, :] ** 2
    p = {1: np.exp(-q2 / 4), 2: (1 + q2) ** -2, 3: (1 + q2) ** -(float(np.float32(kappa)) + 1.5)}[ptype]
    b *= np.sqrt(p) / np.abs(b)
    b[0, 0, 0] = 0.0
    x = np.fft.irfftn(b, s=(n3, n2, n1), axes=(0, 1, 2))
    x -= x.mean()
    return x * (float(np.float32(eps)) / np.sqrt(np.mean(x * x)))


@pytest.mark.parametrize("ptype,shape", [
    (3, (198, 26, 23)), (2, (25, 36, 49)), (1, (64, 17, 131)), (3, (7, 600, 3)), (2, (5, 3, 1150)),
    (3, (262, 2, 9)), (2, (1201, 4, 5)), (3, (16, 128, 64)), (2, (3, 2, 2)), (3, (2000, 4, 3)),
    (1, (3, 3300, 2)), (3, (4, 3, 4000)), (2, (4801, 3, 2)),
])
def test_same_field_as_the_host(ptype, shape):
    args = (ptype, shape, (0.5, 0.4, 0.3), (2.0, 1.5, 1.0), 0.05, 0.5)
    want = _host(*args, seed=5)
    got = rmedia_3d(*args, seed=5)
    assert got.shape == want.shape
    assert np.abs(got - want).max() <= 1e-6 * np.abs(want).max()
