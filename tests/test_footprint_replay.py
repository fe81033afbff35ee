"""The footprint tests of the rasterizer leave out no pixel that the hit
evaluation accepts: the product's own device code compiled for the host, over
every pixel of every record's rect (oracle/footprint_replay.cpp). The tests
allow 1/32 px (1/8 px by rows), so rounding of thin, edge-on and far-off
ellipses is what could break this."""

import pytest

import oracle


KINDS = {"usual": 0, "thin": 1, "edge-on": 2, "opacity at the threshold": 3, "large and near": 4, "mixed": 5}


# Odd sizes, one below a tile, a large one (centres far from the origin).
@pytest.mark.parametrize("kind", list(KINDS))
@pytest.mark.parametrize("n,size", [(40_000, (203, 131)), (30_000, (15, 9)), (4_000, (3839, 2161))])
def test_no_accepted_pixel_is_left_out(kind, n, size):
    if kind == "large and near":
        n //= 10
    r = oracle.footprint_replay(11, n, *size, KINDS[kind])
    assert r["hits"] > (n // 50 if kind != "opacity at the threshold" else 0)
    assert r["misses"] == dict.fromkeys(oracle.FOOTPRINT_TESTS, 0)
    assert r["bounded"] > 0
    if kind in ("usual", "edge-on") and size == (203, 131):
        assert r["kept"] < 0.2  # the tests do leave out what a record does not reach


def test_disk_radius_has_no_error_beyond_its_rounding():
    """Logarithm and root of the opacity bound are taken in double."""
    for kind in KINDS.values():
        assert oracle.footprint_replay(12, 5_000, 203, 131, kind)["radius_err"] == 0.0
