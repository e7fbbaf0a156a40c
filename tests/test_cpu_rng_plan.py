"""The host's part of the device draws (rng_plan.h) without a GPU: plans of
one stream, of many short ones and of ragged lengths, with chunks of 1 to 64
blocks, packed under the host's address and undefined-behaviour sanitizers;
chunk starts from the jump tables against an independent big-integer jump."""
import os
import subprocess

import numpy as np
import pytest

import pyoracle as po
import rng_jump as rj

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("rng_plan") / "check")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
                           "-Wno-unknown-pragmas", os.path.join(HERE, "rng_plan_check.cpp"), "-o", exe])

    def run(*plans):
        text = "\n".join("%d %s" % (len(p), " ".join("%d %d" % s for s in p)) for p in plans)
        r = subprocess.run([exe], input=text, capture_output=True, text=True)
        assert r.returncode == 0, r.stdout[-300:] + r.stderr[-2000:]
        return r.stdout.splitlines()
    return run


def _ragged(n, seed):
    rng = np.random.default_rng(seed)
    return [(int(s), int(2 ** e)) for s, e in zip(rng.integers(0, 2 ** 31, n), rng.uniform(0, 18, n))]


def test_plans_pack_within_their_bytes(check):
    plans = [[(1, 0)], [(5, 1)], [(7, 20011)], [(2 ** 63, 3)], _ragged(2, 1), _ragged(63, 2), _ragged(500, 3),
             [(9, 64)] * 300, [(s, 24 * s * s) for s in range(1, 128)]]
    # lengths on both sides of each change of the chunk length (need = 65536 chunks)
    for q in range(1, 7):
        n = int((65536 * 24.0 * 2 ** q - 4096) / 2.2)
        plans += [[(q, n - 2)], [(q, n + 2)]]
    out = check(*plans)
    kc = [int(s.split()[1]) for s in out if s.startswith("plan")]
    assert len(kc) == len(plans)
    assert kc[-12:] == [0, 1, 1, 2, 2, 3, 3, 4, 4, 5, 5, 6]
    states = [s for s in out if s.startswith("state")]
    for s in states[:60] + states[-36:]:
        v = [int(x) for x in s.split()[1:]]
        want = po.ranlxs_raw_from_state(*rj.state_at_block(v[0], v[1]), 48)
        assert np.array_equal(po.ranlxs_raw_from_state(v[3:], v[2], 48), want), s


@pytest.mark.parametrize("streams", [[(s, 16 ** 3) for s in range(1, 262146)],    # a wavefront of chunks each
                                     [(s, 128 ** 3) for s in range(1, 5601)],
                                     [(77, 12 * 10 ** 9)]])
def test_reach_is_each_streams_own(check, streams):
    """The jump tables reach a chunk of its own stream: draws of any number of
    streams are planned, and a stream of more Gaussians than four base-64
    digits of chunks hold; the furthest chunks are where the stream is."""
    out = check(streams)
    assert int(out[0].split()[2]) >= 262145
    for s in out[1:4] + out[-3:]:
        v = [int(x) for x in s.split()[1:]]
        want = po.ranlxs_raw_from_state(*rj.state_at_block(v[0], v[1]), 48)
        assert np.array_equal(po.ranlxs_raw_from_state(v[3:], v[2], 48), want), s
