"""Requests of two models and two row lengths queued together, in turn, from
pinned and pageable memory, with c0 below and past the staged size (128 KiB):
each returns the bits that predict gives on the same stored rows."""
import hashlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def h(t: bytes) -> bytes:
    return hashlib.sha256(t).digest()


def model(gpu, rng, S, dim):
    sv = np.zeros((S, 785), np.uint32)
    for v in range(S):
        sv[v, rng.choice(np.arange(dim), size=6, replace=False)] = rng.integers(1, 17, 6)
    return gpu.SvmModel(2, [S // 2, S - S // 2], [1, 2], rng.normal(0, 1, (1, S)), rng.normal(0, 10, 1), sv)


@pytest.mark.parametrize("pinned", [(False, False), (True, True), (True, False), (False, True)])
def test_interleaved_requests(gpu, pinned):
    print(f"[gpu-serve-upload] pinned cl, c0: {pinned}", flush=True)
    rng = np.random.default_rng(5)
    keys = gpu.Context()
    keys.setup(h(b"uA"), h(b"uS"), h(b"uE"), 124)
    mpk, msk = keys.get_keys()
    models = [model(gpu, rng, 30, 50), model(gpu, rng, 17, 50)]
    pools = {}
    for l in (60, 124):
        c = gpu.Context()
        c.load_keys(mpk, msk)
        c.rows_reserve(100, l)
        c.encrypt_rows(rng.integers(0, 5, (100, l)).astype(np.uint32), h(b"u2%d" % l), h(b"u3%d" % l))
        refs = []
        for m in models:
            c.set_model(m)
            refs.append(c.predict(0, 100, want_kvalues=True)[:2])
        out = []
        for a, p in zip(c.export_rows(0, 100), pinned):
            b = gpu.host_empty(a.shape) if p else np.empty_like(a)
            b[...] = a
            out.append(b)
        pools[l] = (out[0], out[1], refs)
    srv = gpu.Server(keys, max_batch_rows=256)
    ids = [srv.add_model(m) for m in models]
    srv.start()
    try:
        # 100 rows of 124 slots: 145 KiB of c0
        reqs = [(i % 2, 124 if (i // 2) % 3 else 60, (7 * i) % 30, n)
                for i, n in enumerate([1, 2, 64, 3, 1, 33, 70, 5, 31, 32, 1, 1, 17, 64, 8, 2])]
        reqs += [(0, 124, 0, 100), (1, 60, 0, 100), (1, 124, 1, 90), (0, 60, 99, 1)]
        tickets = [srv.submit(ids[k], pools[l][0][r0:r0 + n], pools[l][1][r0:r0 + n], want_kvalues=True)
                   for k, l, r0, n in reqs]
        for t, (k, l, r0, n) in zip(tickets, reqs):
            lab, kv = srv.wait(t)[:2]
            rl, rk = pools[l][2][k]
            assert np.array_equal(lab, rl[r0:r0 + n]) and np.array_equal(kv, rk[r0:r0 + n]), (k, l, r0, n)
    finally:
        srv.close()
