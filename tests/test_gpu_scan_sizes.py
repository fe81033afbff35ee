"""Exclusive scan around the sizes at which it changes its launches: one block
(up to 16384 items), partition sums added up by the last kernel (up to 256
partitions of 4096) and scanned by one of their own; against the oracle."""

import numpy as np
import pytest

import oracle
from conftest import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [0, 1, 15, 16, 16383, 16384, 16385, 20_480, 256 * 4096 - 1, 256 * 4096, 256 * 4096 + 1])
@pytest.mark.parametrize("modulus", [16, 0])  # 0: whole 32-bit values, the sum wraps
def test_exclusive_scan_sizes(gpu, n, modulus):
    import splattar_amd as sa
    announce(f"scan n={n} modulus={modulus}")
    scan = sa.PrefixSum(gpu, max(n, 1))
    vals = oracle.xorshift32(n + 3, max(n, 1), modulus)[:n]
    if n:
        scan.data().write(vals)
    scan.encode(n)
    want, total = oracle.exclusive_scan(vals)
    if n:
        assert np.array_equal(scan.data().read(n), want)
    assert int(scan.total().read()[0]) == total
    scan.close()
