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
