"""How a convolution is cut into launches, on the CPU: every position and channel is
covered once and no launch exceeds the device's limits, over the sizes that the entry
points accept (positions times taps up to 2^31)."""
import random

import pytest

from tests.conv_plan import plan

SIZES = [
    # positions, taps, channels per group, (image, group) pairs
    (1, 1, 1, 1), (67108864, 31, 4, 1), (2**31 - 1, 1, 1, 1), (2**31 - 1, 1, 300, 1),
    (2**28, 7, 256, 1), (2**26 + 1, 29, 70, 1), (33000000, 65, 8, 1), (2**22, 500, 64, 1),
    (49, 9, 1, 65535), (3136, 9, 1, 384), (2**14, 33024, 3, 1), (1, 64, 1 << 23, 1),
]


def check(P, K, N, z):
    p = plan(P, K, N, z)
    assert 0 < p["gx"] and p["gx"] * p["threads"] < 2**32, p
    assert 0 < p["gy"] <= 65535 and z <= 65535, p
    assert 0 < p["step"] < 2**31 + 64, p
    if p["taps"]:
        assert K <= 4 * p["nw"] and p["step"] == P, p
        assert p["gy"] * p["nper"] >= N > (p["gy"] - 1) * p["nper"], p
        # the stride over positions stays clear of 2^32
        assert P + p["gx"] * p["threads"] < 2**32, p
    else:
        assert p["step"] % p["pt"] == 0 and p["gx"] * p["pt"] == p["step"], p
        assert p["cw"] in (1, 2, 4, 8, 16), p
        assert p["gy"] * 16 * p["cw"] >= N > (p["gy"] - 1) * 16 * p["cw"], p
        # a workgroup's first position is a 32-bit integer
        assert (P - 1) // p["step"] * p["step"] + (P - 1) % p["step"] < 2**31, p


@pytest.mark.parametrize("size", SIZES)
def test_limits(size):
    check(*size)


def test_limits_of_random_sizes():
    rng = random.Random(1)
    for _ in range(4000):
        K = int(2 ** rng.uniform(0, 15))
        P = max(1, int(2 ** rng.uniform(0, 31)) // K)
        check(P, K, int(2 ** rng.uniform(0, 12)), int(2 ** rng.uniform(0, 15.9)))
