"""The scatter pass follows several streams in one wave (streams start on a
multiple of 16 chunks, a wave takes 32): many short streams of each set and
width at once, word for word the oracle's and each stream's alone."""
import hashlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pid", [0, 1, 2])
@pytest.mark.parametrize("which", [1, 2, 3])
@pytest.mark.parametrize("nstreams,ncalls", [(9, 1), (4, 3)])
def test_streams_in_one_wave(gpu, po, pid, which, nstreams, ncalls):
    print(f"[gpu-scatter] set {pid} S{which}: {nstreams} streams x {ncalls}", flush=True)
    ps = gpu.PSet(pid)
    keys = [hashlib.sha256(b"sc%d-%d" % (pid, t)).digest() for t in range(nstreams)]
    nonces = [(977 * t) & 0xffff for t in range(nstreams)]
    got = ps.gauss_sample(keys, nonces, which, ncalls)
    for t in (0, nstreams // 2, nstreams - 1):
        assert np.array_equal(got[t], po.ps_gauss_calls(pid, keys[t], nonces[t], which, ncalls)), t
    for t in range(nstreams):
        assert np.array_equal(got[t], ps.gauss_sample(keys[t:t + 1], nonces[t:t + 1], which, ncalls)[0]), t
