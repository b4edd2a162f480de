"""The waits of the solve sweeps end: csrc/rv_poll.h, which the device code compiles, run on the CPU
with words that never arrive, a failure elsewhere, and words that arrive late."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rivrs-linalg_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "rv_poll.h"

// near, limit, poll at which the last word / every word / the error word is set (-1: never)
int main(int, char **v) {
    const bool near = std::atoi(v[1]);
    const int limit = std::atoi(v[2]);
    const long last_at = std::atol(v[3]), all_at = std::atol(v[4]), err_at = std::atol(v[5]);
    long polls = 0;
    auto past = [&](long at) { return at >= 0 && polls >= at; };
    auto poll = [&](long at) {
        if (++polls > 1000000) {
            std::printf("endless\n");
            std::exit(1);
        }
        return !past(at);
    };
    rv::SpinBudget budget{limit};
    bool unset = poll(all_at);
    const bool ok = rv::wait_words(
        near, [&] { return unset; }, [&] { return poll(last_at); }, [&] { unset = poll(all_at); },
        [&] { return budget.spent([&] { return past(err_at); }); });
    std::printf("%ld %d %d\n", polls, (int)unset, (int)!ok);
    return 0;
}
"""


@pytest.fixture(scope="module")
def waiter(tmp_path_factory):
    d = tmp_path_factory.mktemp("poll")
    src, exe = str(d / "poll.cpp"), str(d / "poll")
    with open(src, "w") as f:
        f.write(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", CSRC, src, "-o", exe], check=True)

    def run(near, limit, last_at, all_at, err_at):
        r = subprocess.run([exe] + [str(int(x)) for x in (near, limit, last_at, all_at, err_at)], capture_output=True,
                           text=True, timeout=60)
        assert r.returncode == 0, r.stdout
        polls, unset, gave_up = (int(x) for x in r.stdout.split())
        return polls, bool(unset), bool(gave_up)

    return run


@pytest.mark.parametrize("near", [True, False])
@pytest.mark.parametrize("limit", [0, 63, 64, 1000])
def test_words_that_never_arrive(waiter, near, limit):
    polls, unset, gave_up = waiter(near, limit, -1, -1, -1)
    assert unset and gave_up and polls <= limit + 2 * 64


@pytest.mark.parametrize("near", [True, False])
@pytest.mark.parametrize("err_at", [0, 1, 64, 500])
def test_a_failure_elsewhere_ends_the_wait(waiter, near, err_at):
    polls, unset, gave_up = waiter(near, 1 << 22, -1, -1, err_at)
    assert unset and gave_up and polls <= err_at + 2 * 64


# the polled word is there, another of the block never comes
def test_a_block_that_stays_incomplete(waiter):
    polls, unset, gave_up = waiter(False, 1000, 10, -1, -1)
    assert unset and gave_up and polls <= 2 * (1000 + 2 * 64)


@pytest.mark.parametrize("near", [True, False])
@pytest.mark.parametrize("at", [0, 1, 2, 63, 64, 65, 900])
def test_words_that_arrive_are_taken(waiter, near, at):
    _, unset, gave_up = waiter(near, 1 << 22, at, at + 3, -1)
    assert not unset and not gave_up
