"""The bound on a resident loop's waits (csrc/fd_wait.h), compiled for the host: a wave gives
a neighbour that runs the limit, counts that from the time its whole group is known to run, and ends
in any case.  The waits are stepped with a clock of one tick."""
import subprocess

import pytest

from swit_amd.build import CSRC

SOURCE = r"""
#include <cstdio>
#include <cstdlib>
#include "fd_wait.h"
using namespace swit::rk;
// ticks from the start of a wait, at clock `start`, to its end; the group runs from clock `runs_at`
int main(int argc, char **argv) {
    const unsigned long long start = atoll(argv[1]), limit = atoll(argv[2]), runs_at = atoll(argv[3]);
    Wait w;
    for (unsigned long long now = start;; ++now)
        if (wait_over(now, limit, w, [&] { return now >= runs_at; })) {
            printf("%llu\n", now - start);
            return 0;
        }
}
"""


@pytest.fixture(scope="module")
def ticks(tmp_path_factory):
    d = tmp_path_factory.mktemp("wait")
    (d / "wait.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, str(d / "wait.cpp"), "-o", str(d / "wait")], check=True)
    return lambda *a: int(subprocess.run([str(d / "wait"), *map(str, a)], check=True, capture_output=True,
                                         timeout=60).stdout)


def test_a_neighbour_that_runs_gets_the_limit(ticks):
    assert ticks(7, 1000, 0) == 2000        # a limit to ask whether the group runs, a limit from there


@pytest.mark.parametrize("runs_at", [1500, 5000, 19000])
def test_waiting_for_room_does_not_count(ticks, runs_at):
    """A group that starts late, behind another launch, has the whole limit from then on."""
    assert ticks(1, 1000, runs_at) == runs_at - 1 + 1000


def test_a_group_that_never_starts_ends(ticks):
    assert ticks(1, 1000, 10**9) == 20 * 1000


def test_no_limit_ends_at_once(ticks):
    assert ticks(1, 0, 0) == 0 and ticks(1, 0, 10**9) == 0
