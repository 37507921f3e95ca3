"""Threads that load keys, make functional keys and encrypt at once, in sizes
that share the copy threads, the runtime's copies and the kept blocks: every one
of them ends, having done all of its passes with the words a single thread
gets."""
import hashlib
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 4096
Q = (16760833, 2147352577, 2130706433)
PASSES = 5


def h(t: bytes) -> bytes:
    return hashlib.sha256(t).digest()


def one_pass(gpu, l, mpk, msk, x, y, t):
    ctx = gpu.Context()
    ctx.load_keys(mpk, msk)
    out = [gpu.keygen(y, msk), gpu.encrypt(x, mpk, h(b"te2%d" % t), h(b"te3")), *ctx.get_keys()]
    ctx.close()
    return out


def test_every_thread_ends(gpu):
    rng = np.random.default_rng(6)
    work = []
    for t, l in enumerate([96, 130, 24, 171]):
        mpk, msk = (np.stack([rng.integers(0, q, (n, N), dtype=np.uint32) for q in Q], axis=1) for n in (l + 1, l))
        work.append((l, mpk, msk, rng.integers(0, 5, (1, l)).astype(np.uint32),
                     rng.integers(0, 17, (2, l)).astype(np.uint32), t))
    want = [one_pass(gpu, *w) for w in work]
    done, bad = [0] * len(work), []

    def run(t):
        try:
            for _ in range(PASSES):
                got = one_pass(gpu, *work[t])
                if not all(np.array_equal(a, b) for a, b in zip(got, want[t])):
                    bad.append(t)
                done[t] += 1
        except Exception as e:  # noqa: BLE001 -- reported by the test's own thread
            bad.append((t, repr(e)))

    threads = [threading.Thread(target=run, args=(t,), daemon=True) for t in range(len(work))]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not any(t.is_alive() for t in threads), done
    assert not bad, bad
    assert done == [PASSES] * len(work)
