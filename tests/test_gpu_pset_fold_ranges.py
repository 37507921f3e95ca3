"""Key generation for more vectors than one launch's threads allow (2^32: 32,768
vectors of the largest set, 256 threads for 64 of a key's 32,768 words): the fold
is launched over ranges of vectors, and each key is the one its vector gives
alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pid,nvec", [(2, 32769), (2, 16385)])
def test_keys_of_many_vectors(gpu, po, pid, nvec):
    print(f"[gpu-pset-fold] set {pid}, {nvec} vectors of one slot", flush=True)
    ps = gpu.PSet(pid)
    rng = np.random.default_rng(nvec)
    msk = np.stack([rng.integers(0, q, (1, ps.N), dtype=np.uint32) for q in ps.q], axis=1)
    pick = rng.integers(0, 8, nvec)
    y = np.array([0, 1, 2, 16, 65535, 65536, ps.q[0], 4294967295], np.uint32)
    want = np.stack([po.ps_keygen(pid, v[None], msk) for v in y])
    sk = ps.keygen(y[pick][:, None], msk)
    for v in sorted({*range(0, nvec, 61), *range(16382, 16385), *range(nvec - 3, nvec)}):
        assert np.array_equal(sk[v], want[pick[v]]), v
