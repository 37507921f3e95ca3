"""Key generation and decryption of every parameter set where the fold's forms
differ: slots around the deal to four waves, y of 16 bits and more, sums that are
a multiple of a modulus, residues equal to q, and more slots than one 64-bit sum
holds.  Word for word the oracle's sequential fold."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def residues(rng, ps, n):
    return np.stack([rng.integers(0, q, (n, ps.N), dtype=np.uint32) for q in ps.q], axis=1)


@pytest.mark.parametrize("pid", [0, 1, 2])
@pytest.mark.parametrize("nvec,l", [(1, 1), (1, 3), (2, 4), (3, 5), (5, 33)])
def test_keygen_and_decrypt_equal_oracle(gpu, po, pid, nvec, l):
    print(f"[gpu-pset-fold] set {pid}, {nvec} x {l}", flush=True)
    ps = gpu.PSet(pid)
    rng = np.random.default_rng(100 * pid + 10 * nvec + l)
    msk = residues(rng, ps, l + 1)
    for s, q in enumerate(ps.q):
        h = ps.N // 4
        msk[:, s, h:h + 64] = q
        msk[:, s, h + 64:h + 128] = 0
        if l > 2:  # y_0 = y_1: sums of 0 mod q, behind 0 or q
            msk[1, s, :h] = q - msk[0, s, :h]
            msk[2:l, s, :h] = np.where(rng.random((l - 2, h)) < 0.5, np.uint32(0), np.uint32(q))
    y = rng.integers(0, 17, (nvec, l)).astype(np.uint32)
    y[:, 0] = rng.choice([1, 65535, 65536, ps.q[0], ps.q[1] + 1, 4294967295], nvec)
    if l > 2:
        y[:, 1] = y[:, 0]
        y[0, 2:] = 0
    sk = ps.keygen(y, msk[:l])
    d = ps.decrypt(msk, y, sk)
    for v in range(nvec):
        assert np.array_equal(sk[v], po.ps_keygen(pid, y[v], msk[:l])), v
        assert np.array_equal(d[v], po.ps_decrypt(pid, msk, y[v], sk[v])), v


def test_more_slots_than_one_sum_holds(gpu, po):
    ps, l = gpu.PSet(0), 65540
    msk = np.empty((l, ps.nmod, ps.N), np.uint32)
    for s, q in enumerate(ps.q):
        msk[:, s] = q - 1
        msk[::7, s] = 4294967295
    y = np.full((1, l), ps.q[0] - 1, np.uint32)
    print(f"[gpu-pset-fold] set 0, {l} slots", flush=True)
    got = ps.keygen(y, msk)
    want = po.ps_keygen(0, y[0], msk)
    assert np.array_equal(got[0], want)
