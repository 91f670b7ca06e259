"""The preprocess backward's chunk lists: every chunk's slice, filled by all
its primitives, stays inside the list buffers (host arithmetic only)."""
import ctypes as C
import os

import pytest

from tinygs_amd import _lib

SIZES = [1, 63, 64, 65, 255, 256, 257, 1023, 1024, 1025, 1100, 2047, 2049, 4097, 131071, 131073, 262144, 262145, 262209, 524288,
         524289, 525000, 1_000_003]


def _fn(name):
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built")
    f = getattr(_lib.load(), name)
    f.argtypes, f.restype = [C.c_int64], C.c_int64
    return f


@pytest.mark.parametrize("n", SIZES)
def test_chunk_lists_hold_every_chunk(n):
    chunks = _fn("_ZN3tgs9pb_chunksEl")(n)
    entries = _fn("_ZN3tgs15pb_list_entriesEl")(n)
    chunk = entries // chunks
    assert chunks * chunk == entries and chunk % 256 == 0
    # chunk c takes the 64-primitive units c, c + chunks, ...; its list starts at c * chunk
    units = (n + 63) // 64
    assert chunks * (chunk // 64) >= units
    for c in {0, chunks // 2, chunks - 1}:
        mine = range(c, units, chunks)
        held = sum(min(64, n - 64 * u) for u in mine)
        assert len(mine) <= chunk // 64
        assert c * chunk + held <= entries


@pytest.mark.parametrize("n", [1, 100_000, 262_144, 262_145, 330_000, 524_288, 524_289, 1_000_003, 1 << 20])
def test_chunks_are_resident_at_once(n):
    """Up to 2^20 primitives every chunk's workgroup has a place on the chip (256 CUs of four workgroups each), in as
    few rounds of 256 primitives as that takes."""
    chunks = _fn("_ZN3tgs9pb_chunksEl")(n)
    rounds = _fn("_ZN3tgs15pb_list_entriesEl")(n) // chunks // 256
    assert chunks <= 1024
    assert rounds == 1 or (n + 128 * rounds - 1) // (128 * rounds) > 1024
