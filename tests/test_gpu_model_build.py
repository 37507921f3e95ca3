"""A model's key columns at the edges of what their build distinguishes: sparse
lists made on the device (empty vectors, full ones, more vectors than one pass
of the prefix sum), the last key slot used or not, two and three key digits,
the fp64 operand made when a kernel first reads it, and a model that is
refused leaving the one before it in place.  Key values equal the oracle's
decryption or the other form of the contraction."""
import hashlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LK, R, P = 30, 5, 50241


def h(t: bytes) -> bytes:
    return hashlib.sha256(t).digest()


@pytest.fixture(scope="module")
def keyed(gpu):
    ctx = gpu.Context()
    ctx.setup(h(b"mb-a"), h(b"mb-s"), h(b"mb-e"), LK)
    rng = np.random.default_rng(3)
    x = rng.integers(0, 5, (R, LK)).astype(np.uint32)
    ctx.rows_reserve(R, LK)
    ctx.encrypt_rows(x, h(b"mb2"), h(b"mb3"), nonce0=0)
    yield ctx, x
    ctx.close()


def model(gpu, sv):
    S = len(sv)
    return gpu.SvmModel(2, [S // 2, S - S // 2], [1, -1], np.ones((1, S)), [0.5], sv)


def vectors(rng, S, width, density, top):
    return (rng.integers(1, top + 1, (S, width)) * (rng.random((S, width)) < density)).astype(np.uint32)


@pytest.mark.parametrize("S,width,density,top", [(1, 29, 1.0, 1), (33, 16, 0.3, 16), (130, 17, 0.0, 1), (1025, 20, 0.2, 3),
                                                 (40, 30, 0.7, 4), (20, 29, 1.0, 3000), (9, 12, 1.0, 60000)])
def test_key_values_equal_oracle(gpu, po, keyed, monkeypatch, S, width, density, top):
    print(f"[gpu-model] {S} x {width} density {density} top {top}", flush=True)
    ctx, x = keyed
    rng = np.random.default_rng(S + width)
    sv = vectors(rng, S, width, density, top)
    ctx.set_model(model(gpu, sv))
    labels, kv, _ = ctx.predict(0, R, want_kvalues=True)
    _, msk = ctx.get_keys()
    cl, c0 = ctx.export_rows(0, R)
    sk = ctx.model_keys()
    for v in sorted({0, S // 2, S - 1}):
        y = np.zeros(LK, np.uint32)
        y[:width] = sv[v]
        assert np.array_equal(sk[v], po.keygen(y, msk)), v
    y = np.zeros((S, LK), np.uint32)
    y[:, :width] = sv
    ip = (x.astype(np.int64) @ y.astype(np.int64).T) % P
    assert np.array_equal(kv.astype(np.int64) % P, ip)
    if width < LK:  # with the last slot in use the fold does not end on zero slots
        pick = sorted({0, S // 2, S - 1})
        assert np.array_equal(kv[:, pick], po.kvalues_coef0(cl, c0, y[pick], sk[pick]))
    for form in ("limbs", "sgpr", "lds"):
        monkeypatch.setenv("CUFE_CONTRACT", form)
        lab, k2, _ = ctx.predict(0, R, want_kvalues=True)
        assert np.array_equal(k2, kv) and np.array_equal(lab, labels), form
    assert not np.any(kv[:, ~sv.any(axis=1)] % P)


def test_refused_model_leaves_the_one_before(gpu, keyed):
    ctx, x = keyed
    rng = np.random.default_rng(9)
    sv = vectors(rng, 12, 20, 0.5, 4)
    m = model(gpu, sv)
    ctx.set_model(m)
    before = ctx.predict(0, R, want_kvalues=True)[:2]
    bad = vectors(rng, 8, 20, 0.5, 4)
    wide = np.zeros((8, 785), np.uint32)
    wide[:, :20] = bad
    wide[5, 40] = 1
    with pytest.raises(gpu.CufeError, match="SV 5 has feature 40"):
        ctx.set_model(model(gpu, wide))
    ctx.model = m
    after = ctx.predict(0, R, want_kvalues=True)[:2]
    assert np.array_equal(before[0], after[0]) and np.array_equal(before[1], after[1])
