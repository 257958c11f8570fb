"""The bounds on a resident loop's waits (csrc/fd_wait.h), compiled for the host: their length on the
100 MHz clock, for a neighbour's message (one limit) and for one that has no room to start yet
(kRoomWaits limits), from no wait at all to the longest one."""
import subprocess

import pytest

from swit_amd.build import CSRC

SOURCE = r"""
#include <cstdio>
#include <cstdlib>
#include "fd_wait.h"
using namespace swit::rk;
// ticks, to the unit of the limit, from the first look at the clock to the end of a wait
int main(int argc, char **argv) {
    const unsigned limit = wait_limit(atoi(argv[1])) * (argv[2][0] == 'r' ? kRoomWaits : 1);
    const unsigned long long start = atoll(argv[3]), unit = 1ull << kWaitShift;
    unsigned long long from = 0, n = 0;
    if (!wait_over(start, from, limit)) {
        unsigned long long lo = 0, hi = 1ull << 40;         // in units: over at hi, not at lo
        while (hi - lo > 1) {
            const unsigned long long mid = lo + (hi - lo) / 2;
            if (wait_over(start + mid * unit, from, limit)) hi = mid;
            else lo = mid;
        }
        n = hi;
    }
    if (from != start) return 1;
    printf("%llu %u %d\n", n * unit, kRoomWaits, kMaxWaitMs);
}
"""


@pytest.fixture(scope="module")
def ticks(tmp_path_factory):
    d = tmp_path_factory.mktemp("wait")
    (d / "wait.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, str(d / "wait.cpp"), "-o", str(d / "wait")], check=True)
    return lambda *a: [int(v) for v in subprocess.run([str(d / "wait"), *map(str, a)], check=True,
                                                      capture_output=True, timeout=60).stdout.split()]


@pytest.mark.parametrize("start", [1, 12345, 2**45 + 7])
@pytest.mark.parametrize("what,limits", [("message", 1), ("room", 20)])
@pytest.mark.parametrize("ms", [0, 1, 1000, 30000, 10**8])
def test_length(ticks, ms, what, limits, start):
    t, room, longest = ticks(ms, what, start)
    assert room == 20 and longest == 10**8
    assert ms * 100000 * limits - limits * 2**16 < t <= ms * 100000 * limits
