"""Sizes of the query blocks of a kNN search by hit bits, from the formulas the library compiles in:
whole groups of 256 queries, all workspaces of a block within the bytes given, none if not even one
group fits."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r"""
#include "launch.hpp"
#include <cstdio>
using namespace dagpu;
int main() {
    for (long long nq : {1ll, 255ll, 256ll, 257ll, 20000ll, 1000000ll, 2147483647ll})
        for (int n : {8192, 8193, 200000, 2000000, 33000000, 100000000})
            for (int d : {1, 32, 33, 128})
                for (size_t most : {(size_t)1, (size_t)1 << 20, (size_t)16 << 20, (size_t)1 << 30,
                                    (size_t)16 << 30})
                    std::printf("%lld %d %d %zu %zu %d\n", nq, n, d, most, bits_query_bytes(n, d),
                                bits_block(nq, n, d, most));
}
"""


@pytest.fixture(scope="module")
def blocks(tmp_path_factory):
    d = tmp_path_factory.mktemp("blocks")
    (d / "b.cpp").write_text(SRC)
    inc = os.path.join(ROOT, "aocl-data-analytics_amd", "csrc", "kernels")
    subprocess.check_call(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", inc, "-I",
                           "/opt/rocm/include", str(d / "b.cpp"), "-o", str(d / "b")])
    out = subprocess.check_output([str(d / "b")], text=True)
    return [tuple(int(v) for v in line.split()) for line in out.splitlines()]


def test_blocks_fit(blocks):
    assert len(blocks) == 7 * 6 * 4 * 5
    for nq, n, d, most, each, block in blocks:
        # bits, 2,048 columns, 256 minima, operand row, norm and limit, threshold and count
        assert each == (n + 511) // 512 * 64 + 2048 * 4 + 256 * 4 + (d + 31) // 32 * 64 + 24
        assert block % 256 == 0 and 0 <= block <= (nq + 255) // 256 * 256
        assert block * each <= most
        # no more groups would be of use or fit
        assert block >= nq or (block + 256) * each > most
