"""Host copies below, at and past the staged size (4 MiB, in chunks of 2 MiB),
to pageable and pinned arrays, from several threads at once, and device blocks
handed from one call to the next: keys loaded into a context come back word
for word, and a call's result does not depend on the calls before it."""
import hashlib
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 4096
POLY = 3 * N
Q = (16760833, 2147352577, 2130706433)


def h(t: bytes) -> bytes:
    return hashlib.sha256(t).digest()


def keys(seed, l):
    rng = np.random.default_rng(seed)
    return (rng.integers(0, 1 << 24, (l + 1, 3, N), dtype=np.uint32), rng.integers(0, 1 << 24, (l, 3, N), dtype=np.uint32))


# 85 polynomials of 48 KiB are just below 4 MiB, 86 just past it
@pytest.mark.parametrize("l", [1, 84, 85, 86, 128, 171, 785])
def test_keys_round_trip(gpu, l):
    print(f"[gpu-copy] {l} slots", flush=True)
    mpk, msk = keys(l, l)
    ctx = gpu.Context()
    ctx.load_keys(mpk, msk)
    a, b = ctx.get_keys()
    assert np.array_equal(a, mpk) and np.array_equal(b, msk)
    ctx.close()


def test_pinned_and_pageable_arrays_agree(gpu):
    rng = np.random.default_rng(1)
    x = np.stack([rng.integers(0, q, (100, N), dtype=np.uint32) for q in Q], axis=1)
    p = gpu.host_empty(x.shape)
    p[...] = x
    pageable = x.copy()
    lib = gpu.lib()
    assert lib.cufe_ntt_forward(pageable, 100) == 0 and lib.cufe_ntt_forward(p, 100) == 0
    assert np.array_equal(pageable, p)
    assert np.array_equal(gpu.ntt_inverse(p), x)


def test_threads_with_their_own_contexts(gpu):
    """Copies of several threads at once: one holds the copy threads, the others
    go through the runtime, and blocks move between the threads' calls."""
    bad = []

    def one(t):
        try:
            for i in range(6):
                l = 60 + 37 * ((t + i) % 5)
                mpk, msk = keys(100 * t + i, l)
                ctx = gpu.Context()
                ctx.load_keys(mpk, msk)
                y = np.random.default_rng(i).integers(0, 17, (2, l)).astype(np.uint32)
                sk = gpu.keygen(y, msk)
                a, b = ctx.get_keys()
                want = np.stack([(y.astype(np.int64) @ msk[:, s].astype(np.int64)) % Q[s] for s in range(3)], axis=1)
                if not (np.array_equal(a, mpk) and np.array_equal(b, msk) and np.array_equal(sk % np.array(Q, np.uint32)[None, :, None], want)):
                    bad.append((t, i))
                ctx.close()
        except Exception as e:  # noqa: BLE001 -- reported by the test's own thread
            bad.append((t, repr(e)))

    threads = [threading.Thread(target=one, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not bad, bad


def test_results_do_not_depend_on_earlier_calls(gpu):
    """The same encryption after calls that leave other data in the kept blocks."""
    l = 40
    mpk, _ = keys(3, l)
    mpk = np.stack([mpk[:, s] % q for s, q in enumerate(Q)], axis=1).astype(np.uint32)
    x = np.arange(2 * l, dtype=np.uint32).reshape(2, l) % 5
    first = gpu.encrypt(x, mpk, h(b"c2"), h(b"c3"))
    for n in (1, 7, 30):
        gpu.gauss_sample([h(b"c%d" % t) for t in range(n)], list(range(n)), 1 + n % 3, 3)
        assert np.array_equal(gpu.encrypt(x, mpk, h(b"c2"), h(b"c3")), first)


# 84 / 85 slots: 85 and 86 polynomials of the public key, around the staged size
@pytest.mark.parametrize("pinned", [False, True])
@pytest.mark.parametrize("l", [84, 85, 120])
def test_encryption_beside_the_key_upload(gpu, po, l, pinned):
    """The public key is uploaded while the noise is sampled: calls in turn with
    different keys, each message the oracle's."""
    print(f"[gpu-copy] encrypt {l} slots, pinned {pinned}", flush=True)
    rng = np.random.default_rng(l)
    x = rng.integers(0, 5, (2, l)).astype(np.uint32)
    ks = []
    for k in range(2):
        mpk = np.stack([rng.integers(0, q, (l + 1, N), dtype=np.uint32) for q in Q], axis=1)
        if pinned:
            p = gpu.host_empty(mpk.shape)
            p[...] = mpk
            mpk = p
        ks.append(mpk)
    for i in range(4):
        c = gpu.encrypt(x, ks[i % 2], h(b"e2%d" % i), h(b"e3%d" % i), 7)
        for b in range(2):
            assert np.array_equal(c[b], po.encrypt(x[b], ks[i % 2], h(b"e2%d" % i), h(b"e3%d" % i), 7 + b)), (i, b)


def test_threads_encrypting_at_once(gpu):
    rng = np.random.default_rng(2)
    ls = [90, 150, 20, 120]
    mpks = [np.stack([rng.integers(0, q, (l + 1, N), dtype=np.uint32) for q in Q], axis=1) for l in ls]
    xs = [rng.integers(0, 5, (1, l)).astype(np.uint32) for l in ls]
    want = [gpu.encrypt(x, m, h(b"t2%d" % t), h(b"t3")) for t, (x, m) in enumerate(zip(xs, mpks))]
    bad = []

    def one(t):
        try:
            for _ in range(5):
                if not np.array_equal(gpu.encrypt(xs[t], mpks[t], h(b"t2%d" % t), h(b"t3")), want[t]):
                    bad.append(t)
        except Exception as e:  # noqa: BLE001 -- reported by the test's own thread
            bad.append((t, repr(e)))

    threads = [threading.Thread(target=one, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not bad, bad
