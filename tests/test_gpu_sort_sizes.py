"""Radix sort around the sizes at which it changes its split: one workgroup
(up to 4096 pairs), few partitions without a scan (up to 2^17) and partitions of
1024, 2048 and 4096 keys; against numpy's stable sort."""

import numpy as np
import pytest

import oracle
from conftest import announce

pytestmark = pytest.mark.gpu


def _check(s, n, bits, lo, hi, digit, distinct):
    keys = oracle.xorshift32(n + 17, max(n, 1), distinct)[:n].astype(np.uint32 if bits == 32 else np.uint64)
    if bits == 64:
        keys = (keys << np.uint64(29)) | oracle.xorshift32(n + 5, max(n, 1), 3)[:n].astype(np.uint64)
    pay = np.arange(n, dtype=np.uint32)
    s.keys().write(keys)
    s.payloads().write(pay)
    s.counts().write(np.array([n], np.uint32))
    s.encode(begin_bit=lo, end_bit=hi, digit_bits=digit)
    mask = np.uint64((1 << hi) - (1 << lo))
    order = np.argsort(keys.astype(np.uint64) & mask, kind="stable")
    assert np.array_equal(s.keys().read(n), keys[order]), (n, distinct)
    assert np.array_equal(s.payloads().read(n), pay[order]), (n, distinct)


# (capacity, counts): the capacity selects the kernels, the count the split.
@pytest.mark.parametrize("bits,cap,counts", [
    (32, 4096, (0, 1, 63, 64, 1023, 1024, 1025, 4095, 4096)),
    (32, 8192, (0, 1, 63, 64, 1023, 1024, 1025, 4097, 8191, 8192)),
    (64, 4096, (0, 1, 65, 1024, 1025, 4095, 4096)),
    (64, 1 << 17, (0, 1, 1025, (1 << 16) + 1, 1 << 17)),
    (32, 1 << 19, (0, 1, 1024, 1025, 8193, (1 << 17) - 1, 1 << 17, (1 << 17) + 1, (1 << 18) + 1, 1 << 19)),
    (64, 1 << 19, (1, 4097, (1 << 17) + 1, (1 << 18) + 1, (1 << 19) - 3)),
    (32, (1 << 22) + 3, (0, 1, 5000, 1 << 20, (1 << 20) + 1, 1 << 22, (1 << 22) + 3)),
    (64, (1 << 20) + 5, (0, 1025, 1 << 20, (1 << 20) + 5)),
])
@pytest.mark.parametrize("digit", [8, 4])
def test_sort_sizes(gpu, bits, cap, counts, digit):
    import splattar_amd as sa
    s = sa.RadixSorter(gpu, cap, key_bits=bits)
    for n in counts:
        announce(f"sort{bits} capacity={cap} n={n} digit={digit}")
        _check(s, n, bits, 0, bits if cap <= 8192 else 16, digit, 1 << 16)
        _check(s, n, bits, 4, 20, digit, 1)                # one key: the input order stays
        _check(s, n, bits, 3, 19, digit, 0xFFFFFFFF)       # whole digits: bits outside the range are ignored
    s.close()


def test_sort_more_partitions_than_the_upsweep_has_workgroups(gpu):
    import splattar_amd as sa
    n = 8192 * 4096 + 5
    announce(f"sort32 n={n}")
    s = sa.RadixSorter(gpu, n, key_bits=32)
    keys = oracle.xorshift32(99, n, 1 << 16)
    s.keys().write(keys)
    s.payloads().write(np.arange(n, dtype=np.uint32))
    s.counts().write(np.array([n], np.uint32))
    s.encode(end_bit=16)
    order = np.argsort(keys.astype(np.uint16), kind="stable")
    assert np.array_equal(s.keys().read(n), keys[order])
    assert np.array_equal(s.payloads().read(n), order.astype(np.uint32))
    s.close()
