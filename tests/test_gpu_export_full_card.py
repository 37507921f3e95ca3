"""Rows taken out of the store with next to no device memory left: the export
needs none of its own, and its words are those of the same rows exported one
at a time before."""
import ctypes as C
import hashlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROWS = 4096  # their canonical words are 201 MB
LEFT = 160 << 20


def h(t: bytes) -> bytes:
    return hashlib.sha256(t).digest()


def test_export_without_room_for_its_words(gpu):
    hip = C.CDLL("libamdhip64.so")
    hip.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
    hip.hipFree.argtypes = [C.c_void_p]

    def free():
        f, t = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value

    ctx = gpu.Context()
    ctx.setup(h(b"xf-a"), h(b"xf-s"), h(b"xf-e"), 2)
    ctx.rows_reserve(ROWS, 2)
    rng = np.random.default_rng(5)
    ctx.encrypt_rows(rng.integers(0, 5, (ROWS, 2)).astype(np.uint32), h(b"xf2"), h(b"xf3"))
    want = {r: ctx.export_rows(r, 1) for r in (0, 1, 2047, ROWS - 1)}
    # a reservation past the card is refused, and gives back what the library keeps
    other = gpu.Context()
    other.setup(h(b"xf-a"), h(b"xf-s"), h(b"xf-e"), 2)
    with pytest.raises(gpu.CufeError, match="hipMalloc"):
        other.rows_reserve(6_000_000, 2)
    other.close()
    filler = []
    try:
        step = 64 << 30
        while step >= 16 << 20:
            p = C.c_void_p()
            if free() > LEFT + step and hip.hipMalloc(C.byref(p), step) == 0:
                filler.append(p)
            else:
                step //= 2
        print(f"[gpu-export] {free() >> 20} MiB left", flush=True)
        if free() >= ROWS * 3 * 4096 * 4:
            pytest.skip("the driver gave out less than the card's free memory")
        cl, c0 = ctx.export_rows(0, ROWS)
    finally:
        for p in filler:
            hip.hipFree(p)
    for r, (a, b) in want.items():
        assert np.array_equal(cl[r], a[0]) and np.array_equal(c0[r], b[0]), r
    again = ctx.export_rows(0, ROWS)
    assert np.array_equal(again[0], cl) and np.array_equal(again[1], c0)
    ctx.close()
