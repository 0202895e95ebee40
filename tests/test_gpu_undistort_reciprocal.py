"""The undistortion's reciprocal where a division goes astray first: a radial
factor of exactly zero, next to zero on both sides, negative, infinite and NaN,
and random coefficients of every size, equal to the oracle (which divides)."""
import numpy as np
import pytest

from oracle import oracle
from parity_util import say

pytestmark = pytest.mark.gpu


def check(name, uv, prm):
    from nav24_amd.undistort import PinholeRadTanHip
    got, ref = PinholeRadTanHip(prm).UndistortKeyPoints(uv), oracle.kp_undistort(uv, prm)
    say(f"{name}: {np.isfinite(ref).mean():.2f} finite")
    assert np.array_equal(got, ref, equal_nan=True), name


def test_radial_factor_zero_and_around():
    # fx = 64, cx = 0: u = 64 has r^2 = 1, where 1 + k1 r^2 is 0 for k1 = -1
    u = np.float32(64) + np.arange(-64, 65, dtype=np.float32) * np.float32(2.0 ** -17)
    uv = np.concatenate([np.stack([u, np.zeros_like(u)], 1), np.stack([np.zeros_like(u), -u], 1)])
    for k1, k2 in ((-1.0, 0.0), (-2.0, 1.0), (0.0, -1.0), (-1.0, 1e30), (1e30, -1e30)):
        check(f"k1 {k1}, k2 {k2}", uv, [64.0, 64.0, 0.0, 0.0, k1, k2, 0.0, 0.0])


@pytest.mark.parametrize("seed", range(4))
def test_random_coefficients_of_every_size(seed):
    r = np.random.default_rng(seed)
    for _ in range(8):
        k = r.choice([-1, 1], 4) * 10.0 ** r.uniform(-12, 12, 4) * (r.uniform(0, 1, 4) < 0.8)
        uv = (r.choice([-1, 1], (2000, 2)) * 10.0 ** r.uniform(-6, 9, (2000, 2))).astype(np.float32)
        check(f"seed {seed}, k {k}", uv, [450.0, 440.0, 320.0, 240.0, *k])
