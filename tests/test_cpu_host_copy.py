"""The host's part of copies through pinned slots (copy_crew.h) without a GPU,
under the host's sanitizers: every byte arrives, once, for arrays of any size
and alignment, on one CPU and with fewer threads than asked for."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SLOT = 1 << 16   # the check's slots and pages


@pytest.fixture(scope="module", params=["address,undefined", "thread"])
def check(request, tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("copy") / "check")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-g", "-pthread", "-fsanitize=" + request.param,
                           os.path.join(HERE, "copy_crew_check.cpp"), "-o", exe])

    def run(*lines, cpus=None):
        r = subprocess.run([exe], input="\n".join(lines) + "\n", capture_output=True, text=True, timeout=100,
                           preexec_fn=None if cpus is None else lambda: os.sched_setaffinity(0, cpus))
        assert r.returncode == 0, r.stdout[-300:] + r.stderr[-3000:]
    return run


# arrays of floats or doubles, their first byte anywhere in a page
CASES = ["0 %d %d" % (b, a) for b in (4, SLOT - 4, SLOT, 5 * SLOT + 12, 40 * SLOT + 8)
         for a in (0, 1, 3, 4, 15, 16, 4097, SLOT - 15, SLOT - 1)]
CASES += ["0 %d 1 %d 2 %d 0" % (3 * SLOT + 4, 9 * SLOT + 20, 12)]


def test_any_size_and_alignment(check):
    check(*CASES)


def test_one_cpu(check):
    check(*CASES, cpus={min(os.sched_getaffinity(0))})


@pytest.mark.parametrize("refused", [1, 2, 0x80, 0x5A, 0xFF])   # a bit for each thread
def test_threads_that_cannot_be_had(check, refused):
    """Whatever starting a thread throws, the caller does its share."""
    check(*["%d%s" % (refused, c[1:]) for c in CASES[::4]])
