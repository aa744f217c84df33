"""The parts that agx_trace_rays cuts a call into: every ray once, in order, up
to the largest count the interface takes (a 32-bit position would pass 2^32 at
the last part and start again).
"""
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "atrc_amd" / "csrc"

PROGRAM = r"""
#include "agx_chunks.h"
#include <cstdio>
#include <cstdlib>
int main(int, char **argv) {
    const uint32_t n = uint32_t(std::strtoull(argv[1], nullptr, 10)), chunk = uint32_t(std::strtoull(argv[2], nullptr, 10));
    unsigned long long next = 0, calls = 0, limit = n / chunk + 3ull;
    const int r = agx::for_each_chunk(n, chunk, [&](size_t first, uint32_t count) {
        if (first != next || count == 0 || count > chunk || ++calls > limit) return 1;
        next += count;
        return 0;
    });
    std::printf("%d %llu %llu\n", r, next, calls);
}
"""


@pytest.fixture(scope="module")
def chunks(tmp_path_factory):
    d = tmp_path_factory.mktemp("chunks")
    (d / "chunks.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{CSRC}", "-o", str(d / "chunks"), str(d / "chunks.cpp")], check=True)
    return lambda n, chunk: [int(x) for x in subprocess.run([str(d / "chunks"), str(n), str(chunk)], check=True,
                                                             capture_output=True, timeout=20).stdout.split()]


CASES = [(n, c) for n in (0, 1, 2, 7) for c in (1, 3)] + \
    [(n, 1 << 22) for n in (0, 1, (1 << 22) - 1, 1 << 22, (1 << 22) + 1, (1 << 32) - (1 << 22),
                            (1 << 32) - (1 << 22) + 1, (1 << 32) - 1)]


@pytest.mark.parametrize("n,chunk", CASES)
def test_every_ray_once(chunks, n, chunk):
    assert chunks(n, chunk) == [0, n, -(-n // chunk)]
