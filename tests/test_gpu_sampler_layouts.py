"""The candidate pass with T0 and T2 in LDS (CUFE_AES_REP=3; the default layout
holds all four tables, 1 and 2 hold T0), where the sampler's other tests run the
default and T0 alone: samples, first samples and encrypted rows, also when a
lowered scan limit makes many chunks ask for all their blocks, and with every
candidate from whole words."""
import hashlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

VARIANTS = [{"CUFE_AES_REP": "3"}, {"CUFE_AES_REP": "3", "CUFE_GAUSS_SCAN": "8"},
            {"CUFE_AES_REP": "3", "CUFE_GAUSS_SCAN": "8", "CUFE_GAUSS_WHOLE": "1"}]


def h(t: bytes) -> bytes:
    return hashlib.sha256(t).digest()


@pytest.fixture(params=VARIANTS, ids=lambda v: "-".join(v.values()))
def variant(request, monkeypatch):
    print(f"[gpu-sampler] {request.param}", flush=True)
    return lambda: [monkeypatch.setenv(k, v) for k, v in request.param.items()]


@pytest.mark.parametrize("which", [1, 2, 3])
def test_samples(gpu, po, variant, which):
    keys = [h(b"lay%d-%d" % (which, t)) for t in range(3)]
    variant()
    full = gpu.gauss_sample(keys, [5, 6, 7], which, 2)
    first = gpu.gauss_sample_first(keys, [5, 6, 7], which, 2)
    for t in range(3):
        assert np.array_equal(full[t], po.gauss_calls(keys[t], 5 + t, which, 2)), t
    assert np.array_equal(first, full[:, :, :, 0])


def test_rows(gpu, variant):
    l, R = 40, 24
    ctx = gpu.Context()
    ctx.setup(h(b"lay-A"), h(b"lay-S"), h(b"lay-E"), l)
    x = np.random.default_rng(4).integers(0, 5, (R, l)).astype(np.uint32)
    got = []
    for _ in range(2):
        ctx.rows_reserve(R, l)
        ctx.encrypt_rows(x, h(b"lay2"), h(b"lay3"), nonce0=9)
        got.append(ctx.export_rows(0, R))
        variant()
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
    ctx.close()


@pytest.mark.parametrize("which,k", [(2, 304214978), (3, 608429953)])
@pytest.mark.parametrize("limit", ["14", "8"])
def test_uniform_words_past_the_tenth(gpu, po, monkeypatch, which, k, limit):
    """Three rejected uniform words among a chunk's first ten (7e-5 of chunks)
    send its last candidates past the words that every chunk leaves: streams that
    have such chunks, beside chains of rejections within the ten, against the
    oracle."""
    bound = k * ((1 << 32) // k)
    n = 900 if which == 2 else 1250  # chunks below any call's length
    keys, nonces = [], []
    for t in range(1000):
        key = h(b"far%d-%d" % (which, t))
        words = np.frombuffer(gpu.aes256ctr(key, t, 0, 24 * n), np.uint32).reshape(n, 96)
        if ((words[:, 50:60] >= bound).sum(axis=1) >= 3).any():
            keys.append(key)
            nonces.append(t)
        if len(keys) == 6:
            break
    print(f"[gpu-sampler] S{which}: streams {nonces}", flush=True)
    assert len(keys) == 6
    monkeypatch.setenv("CUFE_GAUSS_SCAN", limit)
    full = gpu.gauss_sample(keys, nonces, which, 1)
    first = gpu.gauss_sample_first(keys, nonces, which, 1)
    for t, key in enumerate(keys):
        assert np.array_equal(full[t], po.gauss_calls(key, nonces[t], which, 1)), nonces[t]
    assert np.array_equal(first, full[:, :, :, 0])
