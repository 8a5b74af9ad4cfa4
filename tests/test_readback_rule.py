"""Which destinations of a download one kernel may write (tpm_readback.hpp), host code: arrays that lie in one
page-locked allocation each, aligned and apart from each other; anything else takes the copies."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
#include <cstdio>
#include "tpm_readback.hpp"
int main() {
    int count;
    long long n;
    while (std::scanf("%d %lld", &count, &n) == 2) {
        tpm_readback_dst d[11];
        for (int k = 0; k < count; k++) {
            int host;
            unsigned long long dev, base, size;
            if (std::scanf("%d %d %llu %llu %llu", &d[k].bytes, &host, &dev, &base, &size) != 5) return 1;
            d[k].host = host != 0;
            d[k].dev = dev;
            d[k].base = base;
            d[k].size = size;
        }
        std::printf("%d\n", (int)tpm_readback_direct(d, count, n));
    }
    return 0;
}
"""

P = 0x4fff00000000  # a page-locked allocation
TOP = 2 ** 64 - 4096
CASES = {
    "whole allocation": (100, [(4, 1, P, P, 400)], 1),
    "inside an allocation": (100, [(4, 1, P + 64, P, 464)], 1),
    "bytes at an odd address": (100, [(1, 1, P + 1, P, 101)], 1),
    "two arrays side by side": (100, [(4, 1, P, P, 800), (4, 1, P + 400, P, 800)], 1),
    "two allocations": (100, [(4, 1, P, P, 400), (1, 1, P + 4096, P + 4096, 100)], 1),
    "no array": (100, [], 1),
    "at the top of the address space": (100, [(4, 1, TOP, TOP, 400)], 1),
    "pageable": (100, [(4, 0, 0, 0, 0)], 0),
    "one pageable among others": (100, [(4, 1, P, P, 400), (4, 0, 0, 0, 0), (1, 1, P + 400, P, 500)], 0),
    # both ends may be page-locked: another allocation holds the last byte, and what lies between is not known
    "past the end of its allocation": (100, [(4, 1, P, P, 396)], 0),
    "a hole between two allocations": (10000, [(4, 1, P, P, 4096)], 0),
    "an allocation that holds the first entry alone": (100, [(4, 1, P + 396, P, 400)], 0),
    "before its allocation": (100, [(4, 1, P - 4, P, 4096)], 0),
    "misaligned": (100, [(4, 1, P + 2, P, 4096)], 0),
    "the same buffer twice": (100, [(4, 1, P, P, 400), (4, 1, P, P, 400)], 0),
    "overlapping by one byte": (100, [(4, 1, P, P, 800), (1, 1, P + 399, P, 800)], 0),
    "overlapping the other way round": (100, [(1, 1, P + 399, P, 800), (4, 1, P, P, 800)], 0),
}


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    d = tmp_path_factory.mktemp("readback")
    (d / "r.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror",
                    "-I" + os.path.join(ROOT, "tigerpm_amd", "csrc"), str(d / "r.cpp"), "-o", str(d / "r")], check=True)
    return str(d / "r")


@pytest.mark.parametrize("name", CASES)
def test_rule(driver, name):
    n, arrays, want = CASES[name]
    text = "%d %d\n" % (len(arrays), n) + "".join("%d %d %d %d %d\n" % a for a in arrays)
    out = subprocess.run([driver], input=text, capture_output=True, text=True, check=True).stdout
    assert int(out) == want
