"""The tiles that the blocks of calls with unstacked adapters read and store, walked on the CPU as the kernels do: every tile
that is read is one of the weight's, and every tile is stored once, wherever on 16 columns a side of the adapters begins."""
import ctypes

import pytest

from kiln_amd import _lib
from tests.test_gpu_adapter_sides import Side

CUS = 256
SMALL, MID = 1, 2


def _blocks(L, m, n, k, sides, n_adapters):
    """((kernel, tiles of a block, K slices, own rank tiles), [(first tile, end of its own tiles) of every column block])"""
    s = (Side * len(sides))(*(Side(16, 16, rank, first, rows) for rank, first, rows in sides))
    out = (ctypes.c_int * (4 + 2 * (n // 16)))()
    count = L.kiln_w4a16_debug_adapter_blocks(m, n, k, CUS, s, len(sides), 0, n_adapters, out, len(out))
    assert count >= 0
    return tuple(out[:4]), [(out[4 + 2 * i], out[5 + 2 * i]) for i in range(count)]


def _walk(plan, blocks, tiles):
    """What the kernels read and store of those blocks: tile by tile, or pair by pair on the mid-M kernel."""
    step = 2 if plan[0] == MID else 1
    stored = []
    for first, end in blocks:
        for p in range(0, plan[1], step):
            read = first + min(p, end - step - first)
            assert 0 <= read <= tiles - step, (first, end, p)
            if first + p < end:
                assert read == first + p, (first, end, p)
                stored += range(first + p, first + p + step)
    assert sorted(stored) == list(range(tiles))


def _splits(n):
    """Two and three sides of n columns that begin on a multiple of 16: even and odd tiles, one and several tiles wide."""
    t = n // 16
    two = [(b,) for b in sorted({1, 2, 3, 5, 17, 32, 33, t - 3, t - 1})]
    three = [(1, 2), (3, 16), (3, 17), (17, 18), (16, 33), (t - 2, t - 1)]
    return [tuple(16 * b for b in s) for s in two + three if s[-1] < t]


@pytest.mark.parametrize("n,k", [(1024, 1024), (768, 2560), (2560, 4096), (5120, 1536)])
@pytest.mark.parametrize("rank", [8, 16])
def test_automatic_plans(n, k, rank):
    L, own = _lib.load(), 0
    for borders in _splits(n):
        ends = borders + (n,)
        sides = [(rank, first, end - first) for first, end in zip((0,) + borders, ends)]
        for m in (1, 7, 16, 17, 20, 32, 33, 50, 64, 100):
            for n_adapters in (len(sides), 6):
                plan, blocks = _blocks(L, m, n, k, sides, n_adapters)
                if blocks:
                    _walk(plan, blocks, n // 16)
                    own += plan[3] > 0
    assert own > 0


@pytest.mark.parametrize("tiles", [2, 3, 5])
def test_blocks_of_up_to_16_rows_end_with_sides_from_five_adapters_on(tiles):
    L, n, k = _lib.load_tuning(), 1024, 1024
    for borders in _splits(n):
        sides = [(8, first, end - first) for first, end in zip((0,) + borders, borders + (n,))]
        for n_adapters in (len(sides), 4, 5, 8):
            L.kiln_w4a16_debug_gmp(tiles, 4, 1)
            L.kiln_w4a16_debug_lora_fold(3)
            plan, blocks = _blocks(L, 7, n, k, sides, n_adapters)
            assert plan == (SMALL, tiles, 1, (8 * len(sides) + 15) // 16 if n_adapters <= 4 else 1)
            _walk(plan, blocks, n // 16)
            ends = {0, n // 16} | ({b // 16 for b in borders} if n_adapters > 4 else set())
            assert {end for _, end in blocks} | {0} == ends
            assert n_adapters > 4 or len(blocks) == -(-n // (16 * tiles))


def _own(m, k, n, rank):
    plan, _ = _blocks(_lib.load(), m, n, k, [(rank, 0, n)], 1)
    return plan[3] > 0


@pytest.mark.parametrize("m,k,n,rank,own", [
    # short launches, the fewer ranks the shorter
    (1, 1024, 4096, 8, 1), (16, 1024, 4096, 8, 1), (1, 2560, 2560, 8, 1), (1, 2048, 2048, 32, 1), (1, 2560, 4096, 8, 1), (11, 1536, 8192, 8, 1),
    # 8 and 16 ranks whose projection in the first blocks ends before the launch would anyway
    (1, 1536, 16384, 8, 0), (1, 1536, 16384, 16, 0), (1, 4096, 3584, 8, 0), (8, 2560, 7936, 8, 0),
    # K slices, which few blocks have
    (1, 4096, 1024, 8, 1), (8, 8192, 2048, 8, 1),
    # blocks of all of K that fill the chip, against wider ones, and others
    (1, 4096, 4096, 8, 0), (11, 4096, 4096, 8, 0), (1, 5120, 4096, 8, 0), (8, 5120, 4096, 8, 0), (1, 6144, 4096, 8, 0), (1, 2048, 8192, 8, 0),
    (1, 4096, 8192, 8, 0), (1, 2560, 8192, 8, 0), (4, 2048, 8192, 8, 1), (4, 5504, 7936, 16, 1), (1, 5504, 7936, 24, 1), (1, 5504, 8192, 24, 1),
    # launches that fill the chip in one round: no border, no second round
    (1, 11008, 4096, 8, 1), (16, 11008, 4096, 8, 1), (16, 12032, 4096, 16, 1), (1, 1024, 8192, 16, 1), (1, 2048, 8192, 16, 1),
    # several rounds: wide blocks, or against many slices
    (8, 6656, 16128, 8, 0), (8, 15104, 7936, 8, 0), (16, 8192, 19712, 8, 1), (1, 9216, 15616, 8, 1),
    # the first way in three and four slices
    (1, 12288, 4096, 8, 0), (8, 14336, 4096, 8, 0),
    # from 17 rows on
    (24, 4096, 4096, 8, 1), (24, 1024, 8192, 16, 1), (50, 2560, 8192, 16, 1), (64, 1536, 16384, 8, 1), (32, 3072, 16384, 16, 0),
])
def test_where_blocks_project_by_themselves(m, k, n, rank, own):
    assert _own(m, k, n, rank) == bool(own)


@pytest.mark.parametrize("pairs", [1, 2, 3])
def test_plans_of_every_width_from_17_rows_on(pairs):
    L, n, k = _lib.load_tuning(), 1024, 1024
    taken = 0
    for borders in _splits(n):
        sides = [(8, first, end - first) for first, end in zip((0,) + borders, borders + (n,))]
        for ks in (1, 2):
            for m in (17, 33, 64):
                L.kiln_w4a16_debug_mid(1, pairs, ks)
                L.kiln_w4a16_debug_lora_fold(3)
                plan, blocks = _blocks(L, m, n, k, sides, len(sides))
                if plan[3] > 0:
                    assert plan[:2] == (MID, 2 * pairs) and len(blocks) == -(-n // (32 * pairs))
                    _walk(plan, blocks, n // 16)
                    taken += 1
    assert taken >= 15
