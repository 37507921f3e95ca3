"""The sampler's call boundaries across the walk's windows of 16,384 chunks:
streams that end inside the first window, near its edge and several windows
on, the calls that lie across an edge, two streams of different lengths in one
plan, and compact streams (sample 0 of each call).  Every word equals the
oracle's sequential stream."""
import hashlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def h(t: bytes) -> bytes:
    return hashlib.sha256(t).digest()


# a call takes about 752 (S1), 952 (S2) and 1323 (S3) chunks: the edge lies in
# call 21, 17 and 12
@pytest.mark.parametrize("which,ncalls", [(1, 21), (1, 22), (1, 66), (2, 17), (2, 18), (3, 12), (3, 13), (3, 27)])
def test_calls_across_windows(gpu, po, which, ncalls):
    print(f"[gpu-walk] S{which} x {ncalls}", flush=True)
    key = h(b"w%d-%d" % (which, ncalls))
    want = po.gauss_calls(key, 3, which, ncalls)
    assert np.array_equal(gpu.gauss_sample([key], [3], which, ncalls)[0], want)
    assert np.array_equal(gpu.gauss_sample_first([key], [3], which, ncalls)[0], want[:, :, 0])


@pytest.mark.parametrize("pid,ncalls", [(0, 45), (2, 14)])
def test_other_call_lengths_across_windows(gpu, po, pid, ncalls):
    """2,048 and 8,192 samples a call: shorter and longer spans than 4,096."""
    print(f"[gpu-walk] set {pid} x {ncalls}", flush=True)
    key = h(b"wp%d" % pid)
    for which in (1, 3):
        got = gpu.PSet(pid).gauss_sample([key], [9], which, ncalls)[0]
        assert np.array_equal(got, po.ps_gauss_calls(pid, key, 9, which, ncalls))


def test_streams_of_uneven_lengths_in_one_plan(gpu, po):
    """One message a plan: r and f_0 (two S2 calls, one window) beside l calls of S3."""
    l = 30
    a = po.sample_polya(h(b"wa"))
    mpk, _ = po.setup_from_a(a, h(b"ws"), h(b"we"), l)
    x = np.arange(2 * l, dtype=np.uint32).reshape(2, l) % 5
    got = gpu.encrypt(x, mpk, h(b"w2"), h(b"w3"), nonce0=4)
    for b in range(2):
        assert np.array_equal(got[b], po.encrypt(x[b], mpk, h(b"w2"), h(b"w3"), 4 + b))


@pytest.mark.parametrize("variant", [{}, {"CUFE_AES_REP": "3"}, {"CUFE_GAUSS_WHOLE": "1"}])
@pytest.mark.parametrize("nstreams,which,ncalls", [(1, 1, 1), (1, 2, 2), (3, 3, 5), (40, 2, 2), (5, 3, 90)])
def test_tile_sizes_and_whole_words(gpu, po, monkeypatch, nstreams, which, ncalls, variant):
    """From a few tiles of 16 chunks to several tiles of 64 a wave, with the
    high words deciding and with every candidate from whole words (what a tie
    of the high words takes), and the two-table layout."""
    for k, v in variant.items():
        monkeypatch.setenv(k, v)
    print(f"[gpu-candidates] {nstreams} x S{which} x {ncalls} {variant}", flush=True)
    keys = [h(b"t%d" % t) for t in range(nstreams)]
    nonces = list(range(nstreams))
    got = gpu.gauss_sample(keys, nonces, which, ncalls)
    first = gpu.gauss_sample_first(keys, nonces, which, ncalls)
    for t in {0, nstreams - 1}:
        want = po.gauss_calls(keys[t], nonces[t], which, ncalls)
        assert np.array_equal(got[t], want)
        assert np.array_equal(first[t], want[:, :, 0])
