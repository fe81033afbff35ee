"""The one-workgroup sort writes over its input after an even number of passes,
so its buffers may not be declared as free of aliases (results of a compiler
that used such a promise would be wrong only now and then)."""

import os
import re

from conftest import ROOT


def _params(src, name):
    """The parameter lists of the functions called `name` that sort.hip defines."""
    found = re.findall(r"\b%s\(((?:[^()]|\([^()]*\))*)\)\s*\{" % name, src)
    assert found, name
    return found


def test_in_place_sort_promises_no_restrict():
    with open(os.path.join(ROOT, "splattar_amd", "csrc", "sort.hip")) as f:
        src = f.read()
    for name in ("small_sort", "small_sort_kernel"):
        for params in _params(src, name):
            for buf in ("kin", "vin", "kout", "vout"):
                for p in params.split(","):
                    if re.search(r"\b%s\b" % buf, p):
                        assert "__restrict__" not in p, f"{name}: {p.strip()}"
    # The passes of several workgroups go from one pair of buffers to the other.
    assert "__restrict__" in _params(src, "downsweep_kernel")[0]
