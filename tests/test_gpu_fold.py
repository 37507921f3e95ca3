"""Key generation and the sum part of decryption over every form of the fold:
few and many sparse vectors, dense ones, entries of 16 bits and more, sums
that are a multiple of a modulus (where mod_prime's q representative decides),
and residues equal to q.  Word for word the oracle's sequential fold."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 4096
Q = (16760833, 2147352577, 2130706433)


def residues(rng, n):
    return np.stack([rng.integers(0, q, (n, N), dtype=np.uint32) for q in Q], axis=1)


# 31 / 32 vectors: few / many; 15 / 16 / 17 / 33 dense ones: below, at and past
# the dense form's group of 16
@pytest.mark.parametrize("nvec,l,density", [(1, 1, 1.0), (1, 123, 1.0), (3, 785, 0.02), (15, 40, 1.0), (16, 41, 1.0),
                                            (17, 39, 0.6), (33, 5, 1.0), (31, 60, 0.1), (32, 60, 0.1), (40, 16, 0.0)])
def test_keygen_equals_oracle(gpu, po, nvec, l, density):
    print(f"[gpu-fold] {nvec} x {l} density {density}", flush=True)
    rng = np.random.default_rng(nvec * 1000 + l)
    msk = residues(rng, l)
    y = (rng.integers(1, 17, (nvec, l)) * (rng.random((nvec, l)) < density)).astype(np.uint32)
    got = gpu.keygen(y, msk)
    for v in {0, nvec // 2, nvec - 1}:
        assert np.array_equal(got[v], po.keygen(y[v], msk)), v


@pytest.mark.parametrize("nvec", [2, 20, 34])
@pytest.mark.parametrize("wide", [False, True])
def test_zero_sums_and_q_equal_oracle(gpu, po, nvec, wide):
    """Columns of zeros, of q, and pairs v, q - v that cancel; with wide, entries
    past 16 bits, at and above the moduli."""
    print(f"[gpu-fold] zero sums, {nvec} vectors, wide {wide}", flush=True)
    rng = np.random.default_rng(nvec + wide)
    l = 12
    msk = residues(rng, l)
    for s, q in enumerate(Q):
        msk[1, s, :1024] = q - msk[0, s, :1024]  # y_0 = y_1 there: a sum of 0 mod q
        msk[:, s, 2048:2304] = q
        msk[:, s, 2304:2560] = 0
        msk[3:, s, :1024] = np.where(rng.random((l - 3, 1024)) < 0.5, np.uint32(0), np.uint32(q))
        msk[2, s, :1024] = 0
    y = rng.integers(1, 17, (nvec, l)).astype(np.uint32)
    y[:, 1] = y[:, 0]
    if wide:
        y[:, 4] = rng.choice([65535, 65536, Q[0], Q[0] + 1, 2 * Q[0], Q[1], Q[2], 4294967295], nvec)
    y[1, 5:] = 0  # trailing zero slots canonicalise
    got = gpu.keygen(y, msk)
    c = np.concatenate([msk, residues(rng, 1)])
    d = gpu.decrypt(c, y, got)
    for v in {0, 1, nvec - 1}:
        assert np.array_equal(got[v], po.keygen(y[v], msk)), v
        assert np.array_equal(d[v], po.decrypt(c, y[v], got[v])), v
