"""CPU-only: the workspace that a grouped trellis call asks for holds what the call lays out in it."""
import ctypes as C

import pytest

from glq_amd import _lib

ALIGN = 256


def _align(v):
    return (v + ALIGN - 1) // ALIGN * ALIGN


def _slots(shards, k):
    """K slots of the small-batch launch over the 64-row strips of all layers."""
    rows = sum((m + 63) // 64 * 64 for m in shards)
    S, ks = C.c_int(0), C.c_int(0)
    _lib.load().glqh_trellis_mma_plan(C.c_int64(rows), C.c_int64(k), C.byref(S), C.byref(ks))
    assert S.value * ks.value * 32 >= k
    return ks.value


@pytest.mark.parametrize("B", [5, 8, 16])
@pytest.mark.parametrize("n", [1, 2, 3, 4])
def test_workspace_of_5_to_16_tokens_holds_the_groups_slots(n, B):
    """Widths 64..8192, equal shards and a tall one beside narrow ones (grouped-query q/k/v), rows at the edges of the
    64-row strips: x_rht per layer and every layer's [slot][token][row] sums."""
    lib = _lib.load()
    short = []
    for k in list(range(64, 3200, 64)) + list(range(3200, 8193, 448)):
        for m in (32, 64, 96, 512, 1024, 1536, 2304, 2560, 3072, 3648, 4096, 4608, 5248, 5376, 8192, 11008):
            for rest in {m, max(32, m // 4 // 32 * 32), m + 32}:
                shards = [m] + [rest] * (n - 1)
                need = n * _align(2 * B * k) + _align(4 * _slots(shards, k) * B * sum(shards))
                got = lib.glqh_fused_linear_trellis_group_workspace_bytes(B, k, sum(shards), n)
                if got < need:
                    short.append((k, shards, got, need))
    assert not short, (len(short), short[:4])


@pytest.mark.parametrize("entry,m,k,B,slots", [
    ("trellis_gemv", 2048, 11008, 600, 8), ("trellis_gemv", 2048, 11008, 1139, 5), ("trellis_gemv", 2048, 2048, 1600, 4),
    ("trellis_gemv", 2048, 2048, 2000, 2), ("trellis_gemv", 2048, 2048, 3100, 2), ("trellis_gemv", 2048, 2048, 4000, 1),
    ("trellis_gemv", 800, 16384, 600, 18), ("trellis_gemv", 512, 14336, 1024, 16), ("e8_matmul", 3264, 1792, 1347, 1),
    ("e8_matmul", 2048, 4096, 2000, 2), ("e8_matmul", 2048, 11008, 1139, 3)])
def test_slots_of_many_tokens(entry, m, k, B, slots):
    """K slots on either side of the line between those of 512- and of 256-token tiles: the order of a prompt's sums, and
    whether they are rounded to fp16 (up to 16 slots), hang on their number.  (256 CUs)"""
    got = getattr(_lib.load(), f"glqh_{entry}_workspace_bytes")(m, k, B)
    assert got == _align(4 * slots * B * m) + (B + 511) // 512 * 512 * k * 2
