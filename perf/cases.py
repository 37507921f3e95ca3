"""Timed cases of the library: what a program built on it calls, at the sizes it calls it.

Every case is one pass through public entry points of `cufe_amd`, host data in and host data
out, as the C ABI takes it.  The listed cases are the sizes of this repository's tests, of its
benchmark and of the reference's drop-in functions; `draw` spreads the same calls over their
whole range.  Inputs follow the benchmark: sparse binary rows of 123 features (14 ones) in 124
slots, linear SVMs over such vectors with integer coefficients, message entries 0..4, key
entries 0..16.
"""
from __future__ import annotations

import hashlib
import math
import random

import numpy as np

import cufe_amd as cf

N, L, P = cf.N, cf.L, cf.P
POLY_BYTES = 3 * N * 4  # one polynomial of the reference set


def listed():
    return [
        # One functional key for one vector: what a key authority answers a single request
        # with.  The smallest call; launch and transfer latency.
        {"name": "keygen_one_l123", "kind": "keygen", "l": 123, "keys": 1},
        # Functional keys of a block of dense vectors at the reference's key length.
        {"name": "keygen_128_l785", "kind": "keygen", "l": 785, "keys": 128},
        # One ciphertext decrypted under one key, every coefficient, and the rounded result.
        {"name": "decrypt_one_l123", "kind": "decrypt", "l": 123, "keys": 1},
        # The reference's encryption drop-in on one message at its key length: public key
        # in, whole ciphertext out.
        {"name": "encrypt_one_l785", "kind": "encrypt", "l": 785, "messages": 1},
        # The reference's plain prediction of one row: key generation, full decryption and
        # vote for every support vector.
        {"name": "svm_plain_100", "kind": "svm_plain", "svs": 100},
        # The whole scheme (setup, encrypt, keygen, decrypt, rounding) at the largest
        # parameter set, N = 8192 and four limbs.
        {"name": "scheme_n8192_l63", "kind": "scheme", "pset": 2, "l": 63},
        # A client that encrypts a block of rows and takes the compact ciphertexts out.
        {"name": "rows_export_67", "kind": "rows_export", "rows": 67, "slots": 124},
        # Rows encrypted into the resident store and predicted: the encrypted-prediction
        # pipeline from plaintext rows to labels, whole.
        {"name": "rows_predict_2048", "kind": "rows_predict", "rows": 2048, "slots": 124, "svs": 100},
        # A new model over rows in the store: functional keys made, then one block predicted.
        {"name": "model_2000", "kind": "model", "rows": 32, "slots": 124, "svs": 2000},
        # The benchmark's batched prediction over a resident store: labels of every row, and
        # the decrypted inner products of a block of rows.
        {"name": "predict_16384x2000", "kind": "predict", "rows": 16384, "slots": 124, "svs": 2000, "block": 256},
        # Requests of 1..64 rows queued on the server at once, two models.
        {"name": "serve_24", "kind": "serve", "requests": 24, "slots": 124, "svs": 2000, "svs2": 600},
        # Messages of uneven lengths encrypted as one batch and taken out.
        {"name": "encbatch_24", "kind": "encbatch", "messages": 24, "lmax": 128, "graph": True},
    ]


def _logint(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng: random.Random):
    kind = rng.choice(["keygen", "decrypt", "encrypt", "svm_plain", "scheme", "rows_export", "rows_predict", "model",
                       "predict", "predict", "serve", "encbatch"])
    if kind == "keygen":
        return {"kind": kind, "l": _logint(rng, 4, L), "keys": _logint(rng, 1, 128)}
    if kind == "decrypt":
        return {"kind": kind, "l": _logint(rng, 4, L), "keys": _logint(rng, 1, 64)}
    if kind == "encrypt":
        messages = _logint(rng, 1, 6)
        return {"kind": kind, "l": _logint(rng, 4, L // messages), "messages": messages}
    if kind == "svm_plain":
        return {"kind": kind, "svs": _logint(rng, 2, 200)}
    if kind == "scheme":
        return {"kind": kind, "pset": rng.choice([0, 1, 2]), "l": _logint(rng, 4, 100)}
    if kind == "rows_export":
        return {"kind": kind, "rows": _logint(rng, 1, 256), "slots": _logint(rng, 16, 300)}
    if kind == "rows_predict":
        slots = _logint(rng, 16, 400)
        return {"kind": kind, "rows": _logint(rng, 32, 2048 * 100 // slots), "slots": slots, "svs": _logint(rng, 2, 600)}
    if kind == "model":
        return {"kind": kind, "rows": _logint(rng, 1, 64), "slots": rng.choice([16, 124, 333]),
                "svs": _logint(rng, 2, 2000)}
    if kind == "predict":
        return {"kind": kind, "rows": _logint(rng, 1, 16384), "slots": 124, "svs": _logint(rng, 2, 2000),
                "block": _logint(rng, 1, 256)}
    if kind == "serve":
        return {"kind": kind, "requests": _logint(rng, 1, 24), "slots": 124, "svs": _logint(rng, 64, 2000),
                "svs2": _logint(rng, 2, 600)}
    return {"kind": kind, "messages": _logint(rng, 1, 24), "lmax": _logint(rng, 16, 128), "graph": rng.random() < 0.5}


# ---- inputs ------------------------------------------------------------------------------
def _key(case, seed, what):
    return hashlib.sha256(f"{case['kind']}-{seed}-{what}".encode()).digest()


def _rng(seed):
    return np.random.default_rng(seed)


def _sparse_rows(rng, n, slots, ones=14):
    """Binary rows: slot 0 empty, up to 14 ones among the others."""
    k = min(ones, slots - 1)
    x = np.zeros((n, slots), np.uint32)
    pick = np.argsort(rng.random((n, slots - 1)), axis=1)[:, :k]
    np.put_along_axis(x, 1 + pick, 1, axis=1)
    return x


def _model(rng, svs, slots, bias=False):
    n1 = (svs + 1) // 2
    coef = rng.choice(np.concatenate([np.arange(-16, 0), np.arange(1, 17)]), svs).astype(np.float64)[None, :]
    sv = _sparse_rows(rng, svs, slots)
    if bias:
        sv[:, 0] = 1
    return cf.SvmModel(2, [n1, svs - n1], [1, -1], coef, [0.5], sv)


def _small_secret(rng, l):
    """Secret polynomials as setup leaves them: rounded Gaussians of S1's width, as residues."""
    s = np.rint(rng.normal(0.0, 225.0, (l, 1, N))).astype(np.int64)
    q = np.array(cf.Q, np.int64)[None, :, None]
    return s, (s % q).astype(np.uint32)


def _residues(rng, shape):
    """Uniform residues [..][3][N], as ciphertext coefficients are."""
    out = np.empty(shape + (3, N), np.uint32)
    for s, q in enumerate(cf.Q):
        out[..., s, :] = rng.integers(0, q, shape + (N,), dtype=np.uint32)
    return out


def _keygen_inputs(case, seed):
    rng = _rng(seed)
    _, msk = _small_secret(rng, case["l"])
    y = rng.integers(0, 17, (case["keys"], case["l"])).astype(np.uint32)
    return y, msk


def _decrypt_inputs(case, seed):
    rng = _rng(seed)
    s, _ = _small_secret(rng, case["l"])
    y = rng.integers(0, 17, (case["keys"], case["l"])).astype(np.uint32)
    sk = np.einsum("kl,ln->kn", y.astype(np.int64), s[:, 0, :])
    q = np.array(cf.Q, np.int64)[None, :, None]
    return _residues(rng, (case["l"] + 1,)), y, (sk[:, None, :] % q).astype(np.uint32), sk


def _context(case, seed):
    ctx = cf.Context()
    ctx.setup(_key(case, seed, "a"), _key(case, seed, "s"), _key(case, seed, "e"), L)
    return ctx


class _Served:
    """A started server over its context, two models and the requests at hand (rows in pinned
    memory, as the benchmark's clients keep them)."""

    def __init__(self, case, seed):
        rng = _rng(seed)
        self.ctx = _context(case, seed)
        pool = 256
        self.ctx.rows_reserve(pool, case["slots"])
        self.ctx.encrypt_rows(_sparse_rows(rng, pool, case["slots"]), _key(case, seed, "2"), _key(case, seed, "3"))
        cl, c0 = self.ctx.export_rows(0, pool)
        self.cl, self.c0 = cf.host_empty(cl.shape), cf.host_empty(c0.shape)
        self.cl[...], self.c0[...] = cl, c0
        self.server = cf.Server(self.ctx, max_batch_rows=4096)
        self.ids = [self.server.add_model(_model(rng, case[k], case["slots"])) for k in ("svs", "svs2")]
        self.server.start()
        self.requests = []
        for i, n in enumerate(_request_rows(case)):
            r0 = int(rng.integers(0, pool - n + 1))
            self.requests.append((self.ids[i % 2], self.cl[r0:r0 + n], self.c0[r0:r0 + n]))


def _request_rows(case):
    """Rows of each request: 1..64, the same for every seed (one amount of work a case)."""
    return [1 + (37 * i + 30) % 64 for i in range(case["requests"])]


def prepare(case, seed):
    kind, rng = case["kind"], _rng(seed)
    st = {"kind": kind, "case": case}
    if kind == "keygen":
        st["y"], st["msk"] = _keygen_inputs(case, seed)
    elif kind == "decrypt":
        st["c"], st["y"], st["sk"], _ = _decrypt_inputs(case, seed)
    elif kind == "encrypt":
        st["mpk"] = _residues(rng, (case["l"] + 1,))  # a public key's words are uniform
        st["m"] = rng.integers(0, 5, (case["messages"], case["l"])).astype(np.uint32)
        st["seeds"] = _key(case, seed, "2"), _key(case, seed, "3")
    elif kind == "svm_plain":
        x, st["model"] = _svm_plain_inputs(case, seed)
        a = cf.sample_polya(_key(case, seed, "a"))
        mpk, st["msk"] = cf.setup(a, _key(case, seed, "s"), _key(case, seed, "e"), L)
        st["c"] = cf.encrypt(x, mpk, _key(case, seed, "2"), _key(case, seed, "3"))[0]
    elif kind == "scheme":
        st["ps"] = cf.PSet(case["pset"])
        st["x"] = rng.integers(0, 5, (1, case["l"])).astype(np.uint32)
        st["y"] = rng.integers(0, 17, (1, case["l"])).astype(np.uint32)
        st["seeds"] = [_key(case, seed, w) for w in "ase23"]
    elif kind in ("rows_export", "rows_predict"):
        st["ctx"] = _context(case, seed)
        st["x"] = _sparse_rows(rng, case["rows"], case["slots"])
        st["seeds"] = _key(case, seed, "2"), _key(case, seed, "3")
        if kind == "rows_predict":
            st["ctx"].set_model(_model(rng, case["svs"], case["slots"]))
    elif kind in ("model", "predict"):
        ctx = st["ctx"] = _context(case, seed)
        ctx.rows_reserve(case["rows"], case["slots"])
        ctx.encrypt_rows(_sparse_rows(rng, case["rows"], case["slots"]), _key(case, seed, "2"), _key(case, seed, "3"))
        st["model"] = _model(rng, case["svs"], case["slots"])
        if kind == "predict":
            ctx.set_model(st["model"])
    elif kind == "serve":
        st["served"] = _Served(case, seed)
    elif kind == "encbatch":
        st["ctx"] = _context(case, seed)
        lens = _enc_lens(case, seed)
        st["batch"] = cf.EncBatch(st["ctx"], lens)
        st["x"] = rng.integers(0, 5, int(lens.sum())).astype(np.uint32)
        st["seeds"] = _key(case, seed, "2"), _key(case, seed, "3")
    return st


def _enc_lens(case, seed):
    """Message lengths of the batch: the longest one given, the others spread below it (the
    same for every seed, so that cases of one name are one amount of work)."""
    n, top = case["messages"], case["lmax"]
    return np.array([max(1, top * (n - b) // n) for b in range(n)], np.int32)


def _svm_plain_inputs(case, seed):
    rng = _rng(seed)
    x = np.zeros((1, L), np.uint32)
    x[0, :124] = _sparse_rows(rng, 1, 124)[0]
    x[0, 0] = 1  # a bias feature in the row and in every support vector: no inner product is 0
    return x, _model(rng, case["svs"], 124, bias=True)


# ---- one pass ----------------------------------------------------------------------------
def run(st):
    kind, case = st["kind"], st["case"]
    if kind == "keygen":
        return cf.keygen(st["y"], st["msk"])
    if kind == "decrypt":
        d = cf.decrypt(st["c"], st["y"], st["sk"])
        return d, cf.crt_round(d)
    if kind == "encrypt":
        return cf.encrypt(st["m"], st["mpk"], *st["seeds"])
    if kind == "svm_plain":
        label, kv = cf.svm_predict_plain(st["model"], st["c"], st["msk"])
        return label, kv
    if kind == "scheme":
        ps, (sa, ss, se, s2, s3) = st["ps"], st["seeds"]
        mpk, msk = ps.setup(ps.sample_polya(sa), ss, se, case["l"])
        c = ps.encrypt(st["x"], mpk, s2, s3)
        sk = ps.keygen(st["y"], msk)
        d = ps.decrypt(c[0], st["y"], sk)
        return mpk, msk, c, sk, d, ps.crt_round(d, coef=-1)
    if kind in ("rows_export", "rows_predict"):
        ctx = st["ctx"]
        ctx.rows_reserve(case["rows"], case["slots"])
        ctx.encrypt_rows(st["x"], *st["seeds"])
        if kind == "rows_export":
            return ctx.export_rows(0, case["rows"])
        return ctx.predict(0, case["rows"], want_kvalues=True)[:2]
    if kind == "model":
        st["ctx"].set_model(st["model"])
        return st["ctx"].predict(0, case["rows"], want_kvalues=True)[:2]
    if kind == "predict":
        labels = st["ctx"].predict(0, case["rows"])[0]
        block = st["ctx"].predict(0, min(case["rows"], case["block"]), want_kvalues=True)
        return labels, block[0], block[1]
    if kind == "serve":
        srv = st["served"].server
        tickets = [srv.submit(m, cl, c0, want_kvalues=True) for m, cl, c0 in st["served"].requests]
        return [srv.wait(t)[:2] for t in tickets]
    batch = st["batch"]
    batch.run(st["x"], *st["seeds"], use_graph=case["graph"])
    return batch.export(0, case["messages"])


# ---- 64-bit values -----------------------------------------------------------------------
def exact(case, seed):
    """Where the output is a number that plain arithmetic gives: keys and decryptions modulo
    the primes, the rounded result, inner products and the vote.  Ciphertexts, sampled keys
    and served key values are determined by the sampler's keystream alone (a zero inner
    product decrypts to 0 or p by its noise): None."""
    q = np.array(cf.Q, np.int64)
    if case["kind"] == "keygen":
        y, msk = _keygen_inputs(case, seed)
        out = np.empty((y.shape[0], 3, N), np.int64)
        for s in range(3):
            m = msk[:, s].astype(np.int64)
            m[m > q[s] // 2] -= q[s]
            out[:, s] = (y.astype(np.int64) @ m) % q[s]
        return out
    if case["kind"] == "decrypt":
        c, y, _, sk = _decrypt_inputs(case, seed)
        if y.shape[0] > 4:
            return None
        d = np.empty((y.shape[0], 3, N), np.int64)
        for s in range(3):
            fold = (y.astype(np.int64) @ c[:-1, s].astype(np.int64)) % q[s]
            for v in range(y.shape[0]):
                d[v, s] = (fold[v] - _negacyclic(c[-1, s], sk[v] % q[s], int(q[s]))) % q[s]
        return d, np.array([_round(d[v, :, 0]) for v in range(y.shape[0])], np.int64)
    if case["kind"] == "svm_plain":
        x, m = _svm_plain_inputs(case, seed)
        kv = m.sv.astype(np.float64) @ x[0].astype(np.float64)
        return float(m.label[0] if float(m.sv_coef[0] @ kv) - m.rho[0] > 0 else m.label[1]), kv
    return None


def _negacyclic(a, b, q):
    """a * b mod (X^N + 1, q) as one product of big integers (96 bits a coefficient)."""
    w = 12
    ia = int.from_bytes(b"".join(int(v).to_bytes(w, "little") for v in a), "little")
    ib = int.from_bytes(b"".join(int(v).to_bytes(w, "little") for v in b), "little")
    raw = (ia * ib).to_bytes(2 * N * w, "little")
    c = [int.from_bytes(raw[w * i:w * i + w], "little") for i in range(2 * N)]
    return np.array([(c[i] - c[i + N]) % q for i in range(N)], np.int64)


def _round(res):
    """round(p x / Q) of the x with these residues."""
    Q = cf.Q[0] * cf.Q[1] * cf.Q[2]
    x = sum(int(r) * (Q // p) * pow(Q // p, -1, p) for r, p in zip(res, cf.Q)) % Q
    return (2 * P * x + Q) // (2 * Q)


# ---- what a pass cannot do without ---------------------------------------------------------
_CHUNKS = {1: 752, 2: 952, 3: 1324}  # 8-candidate chunks per 4096 samples of S1, S2, S3


def _gauss(calls, which, n=N):
    """Operations of sampled polynomials: 13 AES blocks a chunk (14 rounds of 16 table words)
    and about 100 operations a candidate."""
    return calls * _CHUNKS[which] * n / 4096 * (13 * 14 * 16 * 2 + 8 * 100)


def _ntt(limbs, n=N):
    return limbs * n / 2 * math.log2(n) * 6


def work(case):
    k = case["kind"]
    if k == "keygen":
        return {"bytes": (case["l"] + case["keys"]) * POLY_BYTES, "flops": 2 * case["keys"] * case["l"] * 3 * N}
    if k == "decrypt":
        n = case["keys"]
        return {"bytes": (case["l"] + 1 + 2 * n) * POLY_BYTES,
                "flops": 2 * n * case["l"] * 3 * N + _ntt(3 * (1 + 2 * n)) + n * 6 * N}
    if k == "encrypt":
        polys = case["messages"] * (case["l"] + 1)
        return {"bytes": (case["l"] + 1 + polys) * POLY_BYTES,
                "flops": _gauss(polys - case["messages"], 3) + _gauss(2 * case["messages"], 2) + _ntt(3 * polys)}
    if k == "svm_plain":
        n = case["svs"]
        return {"bytes": (2 * L + 1) * POLY_BYTES, "flops": 2 * n * 15 * 3 * N * 2 + _ntt(3 * (1 + 2 * n))}
    if k == "scheme":
        n, m = {0: (2048, 2), 1: (4096, 3), 2: (8192, 4)}[case["pset"]]
        polys = case["l"] + 1
        return {"bytes": (3 * polys + 2) * n * m * 4,
                "flops": _gauss(2 * case["l"], 1, n) + _gauss(case["l"], 3, n) + _gauss(2, 2, n) +
                         _ntt(m * (4 * polys + 3), n)}
    if k in ("rows_export", "rows_predict"):
        r, l = case["rows"], case["slots"]
        w = {"bytes": r * (l * 4 + POLY_BYTES + 12 * l), "flops": r * (_gauss(l, 3) + _gauss(2, 2) + 2 * 3 * N * l)}
        if k == "rows_predict":
            w["flops"] += 2.0 * 3 * r * case["svs"] * (N + l)
            w["bytes"] = r * (l * 4 + case["svs"] * 4 + 8) + case["svs"] * N * 2
        return w
    if k == "model":
        r, s, l = case["rows"], case["svs"], case["slots"]
        return {"bytes": (L + r) * POLY_BYTES + s * (l * 4 + 8) + r * s * 4,
                "flops": 2.0 * 14 * s * 3 * N + 2.0 * 3 * r * s * (N + l)}
    if k == "predict":
        r, s, l = case["rows"], case["svs"], case["slots"]
        return {"bytes": r * (POLY_BYTES + 12 * l + 8) + s * 2 * (N + l) + min(r, case["block"]) * s * 4,
                "flops": 2.0 * 3 * r * s * (N + l)}
    if k == "serve":
        r, s = sum(_request_rows(case)), (case["svs"] + case["svs2"]) // 2
        return {"bytes": r * (POLY_BYTES + 12 * case["slots"] + 8 + 4 * s),
                "flops": 2.0 * 3 * r * s * (N + case["slots"])}
    lens = _enc_lens(case, 0)
    slots, n = int(lens.sum()), case["messages"]
    return {"bytes": (slots + n) * POLY_BYTES + (int(lens.max()) + 1) * POLY_BYTES,
            "flops": _gauss(slots, 3) + _gauss(2 * n, 2) + _ntt(3 * (slots + 2 * n))}
