"""Coefficient 0 of the compact row encryption at the edges of its 16-row x
32-slot tiles: word for word the oracle's ciphertexts, with keys longer than
the rows."""
import hashlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LK = 70


def h(t: bytes) -> bytes:
    return hashlib.sha256(t).digest()


@pytest.fixture(scope="module")
def keyed(gpu):
    ctx = gpu.Context()
    ctx.setup(h(b"ec-a"), h(b"ec-s"), h(b"ec-e"), LK)
    yield ctx
    ctx.close()


@pytest.mark.parametrize("rows,l", [(1, 1), (1, 70), (15, 31), (16, 32), (17, 33), (33, 64), (40, 5)])
def test_rows_equal_oracle(gpu, po, keyed, rows, l):
    print(f"[gpu-coef0] {rows} rows x {l} slots", flush=True)
    rng = np.random.default_rng(rows * 100 + l)
    x = rng.integers(0, 5, (rows, l)).astype(np.uint32)
    keyed.rows_reserve(rows, l)
    keyed.encrypt_rows(x, h(b"ec2"), h(b"ec3"), nonce0=7)
    cl, c0 = keyed.export_rows(0, rows)
    mpk, _ = keyed.get_keys()
    mpk_l = np.ascontiguousarray(np.concatenate([mpk[:l], mpk[LK:LK + 1]]))
    for r in sorted({0, rows // 2, min(16, rows - 1), rows - 1}):
        want = po.encrypt(x[r], mpk_l, h(b"ec2"), h(b"ec3"), 7 + r)
        assert np.array_equal(c0[r], want[:l, :, 0]), r
        assert np.array_equal(cl[r], want[l]), r
