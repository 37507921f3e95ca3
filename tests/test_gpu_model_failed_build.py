"""A model build that fails after the model before it was let go of leaves none:
every call that reads the model refuses, and the next build works.  The failure
is the host's own refusal of an error bound widened past 2^62, which comes after
the functional keys and before the contraction's digits."""
import hashlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LK, R = 24, 5


def h(t: bytes) -> bytes:
    return hashlib.sha256(t).digest()


def model(gpu, seed, S):
    rng = np.random.default_rng(seed)
    return gpu.SvmModel(2, [S // 2, S - S // 2], [1, -1], np.ones((1, S)), [0.5],
                        rng.integers(0, 4, (S, 20)).astype(np.uint32))


@pytest.mark.parametrize("first", [None, 12, 300])
def test_failed_build_leaves_no_model(gpu, monkeypatch, first):
    ctx = gpu.Context()
    ctx.setup(h(b"fb-a"), h(b"fb-s"), h(b"fb-e"), LK)
    ctx.rows_reserve(R, LK)
    ctx.encrypt_rows(np.random.default_rng(1).integers(0, 5, (R, LK)).astype(np.uint32), h(b"fb2"), h(b"fb3"))
    m = model(gpu, 7, 40)
    ctx.set_model(m)
    want = ctx.predict(0, R, want_kvalues=True)[:2]
    if first:
        ctx.set_model(model(gpu, 8, first))
    monkeypatch.setenv("CUFE_FRAC_WIDEN", "63")
    with pytest.raises(gpu.CufeError, match="widening"):
        ctx.set_model(m)
    monkeypatch.delenv("CUFE_FRAC_WIDEN")
    print(f"[gpu-model] after a failed build, {first}", flush=True)
    assert ctx.contract_digits() == -1
    for call in (lambda: ctx.predict(0, R, want_kvalues=True), ctx.model_keys):
        with pytest.raises(gpu.CufeError, match="no model"):
            call()
    ctx.set_model(m)
    got = ctx.predict(0, R, want_kvalues=True)[:2]
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
    ctx.close()
