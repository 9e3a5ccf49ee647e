"""Calls whose blocks project x onto their adapters by themselves, every instance, against the product in
64 bits and the projection in a launch of its own; and where adapters are taken that way."""
import ctypes

import pytest
import torch

from kiln_amd import _lib, lora, marlin_gemm
from tests.test_gpu_adapter_sides import Side, _all_adapters, _packed


def _instances():
    """(tiles per block, wavefronts, groups of a slice, K slices, ranks): groups per wavefront even and uneven, one wavefront
    for several tiles, one and two rank tiles, ranks that fill a load of four rows or a tile and those that do not."""
    cases = []
    for tiles in range(1, 7):
        for waves, gs, ks in ((1, 1, 1), (3, 3, 2), (8, 20, 1), (12, 12, 1), (12, 24, 3), (10, 20, 1), (7, 20, 1), (8, 32, 1), (10, 50, 1)):
            gpw = -(-gs // waves)
            if gpw > (6 if tiles <= 2 else 3) or tiles * gpw > 16:
                continue
            for r in (4, 12) if (tiles + gs) % 2 else (20, 28):
                own, slots = (r + 15) // 16, min(gpw, 2)
                if waves <= min(16, (160 * 1024 - 128) // ((slots + own) * 4096)):
                    cases.append((tiles, waves, gs, ks, r))
    return cases


def _reference(x, w, sets):
    """(result, low-rank term) in 64 bits; sets: (StackedLora or None, first column) of each projection"""
    base = x.double() @ marlin_gemm.dequant_f32(w.b_packed, w.scales, w.groupsize).double()
    low = torch.zeros_like(base)
    for s, first in sets:
        col = 0
        for r, scale in zip(s.ranks, s.scales) if s is not None else ():
            low[:, first:first + s.b_cat.shape[0]] += scale * (x.double() @ s.a_cat[col:col + r].double().t()) @ s.b_cat[:, col:col + r].double().t()
            col += r
    return base + low, low


def _assert_close(y, want, low):
    # the result rounded once to bf16 and T once per slice of K, half an ulp each: 2^-8 of a row of either at most
    assert bool(((y.double() - want).norm(dim=1) <= 2.0 ** -8 * (want.norm(dim=1) + low.norm(dim=1))).all())


@pytest.mark.gpu
@pytest.mark.parametrize("tiles,waves,gs,ks,r", _instances())
def test_every_instance(tiles, waves, gs, ks, r):
    L, k, n = _lib.load_tuning(), gs * ks * 128, 512
    gen = torch.Generator(device="cuda").manual_seed(tiles * k + r)
    w = _packed(gen, k, n, 128 if gs % 2 == 0 else -1)
    # several adapters with scales of their own, zero among them
    ad, = _all_adapters(gen, k, (n,), ((r,) if r == 4 else (r - 9, 1, 8),))
    ad = lora.StackedLora(ad.a_cat, ad.b_cat, ad.ranks, ad.scales[:-1] + (0.0,) if r > 4 else ad.scales)
    for m in (1, 4, 5, 8, 11, 16):
        x = torch.randn(m, k, device="cuda", generator=gen).bfloat16()
        L.kiln_w4a16_debug_gmp(tiles, waves, ks)
        L.kiln_w4a16_debug_lora_fold(3)
        assert L.kiln_w4a16_takes_rank(m, n, k, r, -1) == 1
        got = marlin_gemm.marlin_w4a16_gemm_lora(x, w.b_packed, w.scales, w.groupsize, ad.a_cat, ad.b_cat, ad.ranks, ad.scales)
        L.kiln_w4a16_debug_gmp(0, 0, 0)
        L.kiln_w4a16_debug_lora_fold(0)
        other = marlin_gemm.marlin_w4a16_gemm_lora(x, w.b_packed, w.scales, w.groupsize, ad.a_cat, ad.b_cat, ad.ranks, ad.scales)
        want, low = _reference(x, w, [(ad, 0)])
        _assert_close(got, want, low)
        _assert_close(other, want, low)


def _mid_instances():
    """(pairs of tiles per block, groups of a slice, K slices, ranks) of the kernel of 17 rows on: one to four groups to a
    wavefront, dealt evenly and not, slices that meet, one and two rank tiles."""
    cases = []
    for pairs in (1, 2, 3):
        for gs, ks in ((4, 1), (6, 3), (8, 2), (11, 1), (20, 1), (23, 1), (8, 4)):
            for r in (4, 16, 20, 32):
                waves = min(gs, 8 if r <= 16 else 6)
                gpw = -(-gs // waves)
                if gpw > 4 or (pairs == 3 and gpw > 3) or (ks > 1 and waves < 8 and r > 16 and gs > 6):
                    continue
                cases.append((pairs, gs, ks, r))
    return cases


@pytest.mark.gpu
@pytest.mark.parametrize("pairs,gs,ks,r", _mid_instances())
def test_every_instance_from_17_rows_on(pairs, gs, ks, r):
    L, k, n = _lib.load_tuning(), gs * ks * 128, 768
    gen = torch.Generator(device="cuda").manual_seed(pairs * k + r)
    w = _packed(gen, k, n, 128 if gs % 2 == 0 else -1)
    ad, = _all_adapters(gen, k, (n,), ((r,) if r <= 16 else (r - 9, 1, 8),))
    taken = 0
    for m in (17, 32, 33, 64, 65, 100, 130):
        x = torch.randn(m, k, device="cuda", generator=gen).bfloat16()
        L.kiln_w4a16_debug_mid(1, pairs, ks)
        L.kiln_w4a16_debug_lora_fold(3)
        # (a rank that is a multiple of 8 is taken either way: the one below it, on the same plan, says whether blocks project it)
        own = L.kiln_w4a16_takes_rank(m, n, k, r if r % 8 else r - 4, -1)
        assert own == 0 or pairs < 3 or m <= 32  # three pairs and two row blocks: no registers for T
        taken += own
        got = marlin_gemm.marlin_w4a16_gemm_lora(x, w.b_packed, w.scales, w.groupsize, ad.a_cat, ad.b_cat, ad.ranks, ad.scales)
        _assert_close(got, *_reference(x, w, [(ad, 0)]))
    assert taken >= (7 if pairs == 1 and ks == 1 else 2)


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 7, 16])
@pytest.mark.parametrize("k,widths,ranks", [
    (512, (256, 512, 256), (None, (8, 8), (8, 8, 8))),         # columns of no side; blocks of one side's ranks
    (1024, (1280, 256, 256), ((16, 16), (8,), (8, 8))),        # a side of two rank tiles
    (4608, (256, 768, 256), ((8, 8), (8, 8), (8, 8))),         # K slices
    (640, (256, 256, 256), ((8,), (16,), (8,))),               # up to four adapters: every block has all of them
])
def test_more_than_four_adapters_side_by_side(k, widths, ranks, m):
    L, n = _lib.load_tuning(), sum(widths)
    gen = torch.Generator(device="cuda").manual_seed(k + m)
    w = _packed(gen, k, n, 128)
    adapters = _all_adapters(gen, k, widths, ranks)
    x = torch.randn(m, k, device="cuda", generator=gen).bfloat16()
    x[-1, 3] = float("inf")  # one row's infinity stays in its row
    firsts = [sum(widths[:i]) for i in range(len(widths))]
    own = [(a, f) for a, f in zip(adapters, firsts) if a is not None]
    sides = (Side * len(own))(*(Side(a.a_cat.data_ptr(), a.b_cat.data_ptr(), a.a_cat.shape[0], f, a.b_cat.shape[0]) for a, f in own))
    each, scales = sum((a.ranks for a, _ in own), ()), sum((a.scales for a, _ in own), ())
    stream = torch.cuda.current_stream().cuda_stream
    want, low = _reference(x[:-1], w, list(zip(adapters, firsts)))
    for plan in ((0, 0, 0), (5, 4, 1), (3, 4, 1)) if k < 4608 else ((0, 0, 0), (5, 9, 2), (3, 6, 2)):
        L.kiln_w4a16_debug_gmp(*plan)
        L.kiln_w4a16_debug_lora_fold(3)
        # the blocks' own way: of one side's ranks and ending with it from five adapters on, of all ranks else
        info, many = (ctypes.c_int * 4)(), len(each) > 4
        blocks = L.kiln_w4a16_debug_adapter_blocks(m, n, k, 256, sides, len(own), 0, len(each), info, 4)
        most = max(a.a_cat.shape[0] for a, _ in own) if many else sum(each)
        assert info[0] == 1 and info[3] == (most + 15) // 16 and (many or blocks == -(-n // (16 * info[1])))
        ws = marlin_gemm._workspace(x.device, stream, L.kiln_w4a16_workspace_bytes(m, n, k))
        out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
        assert L.kiln_w4a16_gemm_adapter_sides(x.data_ptr(), w.b_packed.data_ptr(), out.data_ptr(), w.scales.data_ptr(), m, n, k, ws.data_ptr(), 128,
                                               x.device.index, stream, sides, len(own), 0, len(each), (ctypes.c_int * len(each))(*each),
                                               (ctypes.c_float * len(each))(*scales)) == _lib.OK
        _assert_close(out[:-1], want, low)
        assert not bool(out[-1].isfinite().any())


# (k, K slices, columns, (rank, first column, columns) of each side): sides that begin inside a block of one to three pairs of
# tiles, on an odd tile, inside a tile, behind columns of no side
SIDES_ANYWHERE = [
    (1024, 1, 1024, ((8, 0, 272), (8, 272, 752))),
    (1024, 2, 1024, ((8, 0, 48), (16, 48, 208), (8, 256, 768))),
    (2048, 2, 1024, ((16, 0, 528), (16, 528, 496))),
    (640, 1, 768, ((8, 16, 16), (8, 48, 400), (16, 496, 256))),
    (1024, 1, 768, ((8, 0, 264), (8, 264, 100), (8, 381, 387))),
    (2048, 2, 1024, ((8, 0, 528), (8, 528, 496))),
    (2304, 3, 512, ((24, 0, 496), (8, 496, 16))),
]
# (rows, pairs of tiles per block, one of those): with two row blocks three pairs have no instance, and slices meet in blocks of
# eight wavefronts, which two rank tiles leave no room for
SIDES_ANYWHERE_CASES = [(m, pairs, i) for m in (17, 20, 33, 64, 100) for pairs in (1, 2, 3) for i, (_, ks, _, places) in enumerate(SIDES_ANYWHERE)
                        if m <= 32 or (pairs < 3 and (ks == 1 or sum(p[0] for p in places) <= 16))]


def _side_table(adapters, places):
    at = [(a.a_cat.data_ptr(), a.b_cat.data_ptr()) for a in adapters] if adapters else [(16, 16)] * len(places)
    return (Side * len(places))(*(Side(*ab, r, first, rows) for ab, (r, first, rows) in zip(at, places)))


def _assert_own(L, m, n, k, ks, pairs, places):
    L.kiln_w4a16_debug_mid(1, pairs, ks)
    L.kiln_w4a16_debug_lora_fold(3)
    plan = (ctypes.c_int * 4)()
    blocks = L.kiln_w4a16_debug_adapter_blocks(m, n, k, 256, _side_table(None, places), len(places), 0, len(places), plan, 4)
    assert (blocks, *plan) == (-(-n // (32 * pairs)), 2, 2 * pairs, ks, (sum(r for r, _, _ in places) + 15) // 16)


def test_sides_that_begin_anywhere_are_projected_by_every_block():
    L = _lib.load_tuning()
    for m, pairs, i in SIDES_ANYWHERE_CASES:
        k, ks, n, places = SIDES_ANYWHERE[i]
        _assert_own(L, m, n, k, ks, pairs, places)


@pytest.mark.gpu
@pytest.mark.parametrize("m,pairs,i", SIDES_ANYWHERE_CASES)
def test_sides_that_begin_anywhere_from_17_rows_on(m, pairs, i):
    L, (k, ks, n, places) = _lib.load_tuning(), SIDES_ANYWHERE[i]
    gen = torch.Generator(device="cuda").manual_seed(k + n + m)
    w = _packed(gen, k, n, 128 if pairs == 2 else -1)
    adapters = [_all_adapters(gen, k, (rows,), ((r,),))[0] for r, _, rows in places]
    adapters = [lora.StackedLora(a.a_cat, a.b_cat, a.ranks, (0.5 + 0.25 * i,)) for i, a in enumerate(adapters)]
    firsts = [first for _, first, _ in places]
    x = torch.randn(m, k, device="cuda", generator=gen).bfloat16()
    sides = _side_table(adapters, places)
    ranks, scales = sum((a.ranks for a in adapters), ()), sum((a.scales for a in adapters), ())
    a_cat, b_cat, col = torch.cat([a.a_cat for a in adapters]).contiguous(), torch.zeros(n, sum(ranks), dtype=torch.bfloat16, device="cuda"), 0
    for a, (r, first, rows) in zip(adapters, places):
        b_cat[first:first + rows, col:col + r] = a.b_cat
        col += r
    _assert_own(L, m, n, k, ks, pairs, places)
    stream = torch.cuda.current_stream().cuda_stream
    ws = marlin_gemm._workspace(x.device, stream, L.kiln_w4a16_workspace_bytes(m, n, k))
    # rows behind the last that must stay as they are: a block that stored past its columns would reach them
    out = torch.full((m + 1, n), float("nan"), dtype=torch.bfloat16, device="cuda")
    assert L.kiln_w4a16_gemm_adapter_sides(x.data_ptr(), w.b_packed.data_ptr(), out.data_ptr(), w.scales.data_ptr(), m, n, k, ws.data_ptr(), w.groupsize,
                                           x.device.index, stream, sides, len(places), 0, len(ranks), (ctypes.c_int * len(ranks))(*ranks),
                                           (ctypes.c_float * len(ranks))(*scales)) == _lib.OK
    want = marlin_gemm.marlin_w4a16_gemm_lora(x, w.b_packed, w.scales, w.groupsize, a_cat, b_cat, ranks, scales)
    assert bool(out[m].isnan().all()) and torch.equal(out[:m].view(torch.int16), want.view(torch.int16))
    _assert_close(out[:m], *_reference(x, w, list(zip(adapters, firsts))))


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 7, 16])
@pytest.mark.parametrize("tiles", [1, 3, 5])
@pytest.mark.parametrize("i", [i for i, (_, _, _, places) in enumerate(SIDES_ANYWHERE) if sum(p[0] for p in places) <= 32])
def test_up_to_four_adapters_that_begin_anywhere_give_the_stacked_sets_bits(i, tiles, m):
    L, (k, ks, n, places) = _lib.load_tuning(), SIDES_ANYWHERE[i]
    gen = torch.Generator(device="cuda").manual_seed(k + n + m)
    w = _packed(gen, k, n, 128)
    adapters = [_all_adapters(gen, k, (rows,), ((r,),))[0] for r, _, rows in places]
    adapters = [lora.StackedLora(a.a_cat, a.b_cat, a.ranks, (0.5 + 0.25 * i,)) for i, a in enumerate(adapters)]
    x = torch.randn(m, k, device="cuda", generator=gen).bfloat16()
    ranks, scales = sum((a.ranks for a in adapters), ()), sum((a.scales for a in adapters), ())
    a_cat, b_cat, col = torch.cat([a.a_cat for a in adapters]).contiguous(), torch.zeros(n, sum(ranks), dtype=torch.bfloat16, device="cuda"), 0
    for a, (r, first, rows) in zip(adapters, places):
        b_cat[first:first + rows, col:col + r] = a.b_cat
        col += r
    sides = _side_table(adapters, places)
    L.kiln_w4a16_debug_gmp(tiles, 6, ks)
    L.kiln_w4a16_debug_lora_fold(3)
    plan = (ctypes.c_int * 4)()
    blocks = L.kiln_w4a16_debug_adapter_blocks(m, n, k, 256, sides, len(places), 0, len(places), plan, 4)
    assert (blocks, *plan) == (-(-n // (16 * tiles)), 1, tiles, ks, (sum(ranks) + 15) // 16)
    ws = marlin_gemm._workspace(x.device, torch.cuda.current_stream().cuda_stream, L.kiln_w4a16_workspace_bytes(m, n, k))
    out = torch.full((m + 1, n), float("nan"), dtype=torch.bfloat16, device="cuda")
    assert L.kiln_w4a16_gemm_adapter_sides(x.data_ptr(), w.b_packed.data_ptr(), out.data_ptr(), w.scales.data_ptr(), m, n, k, ws.data_ptr(), 128,
                                           x.device.index, torch.cuda.current_stream().cuda_stream, sides, len(places), 0, len(ranks),
                                           (ctypes.c_int * len(ranks))(*ranks), (ctypes.c_float * len(ranks))(*scales)) == _lib.OK
    want = marlin_gemm.marlin_w4a16_gemm_lora(x, w.b_packed, w.scales, 128, a_cat, b_cat, ranks, scales)
    assert bool(out[m].isnan().all()) and torch.equal(out[:m].view(torch.int16), want.view(torch.int16))
    _assert_close(out[:m], *_reference(x, w, [(a, first) for a, (_, first, _) in zip(adapters, places)]))


def test_ranks_that_are_taken_as_they_are():
    """Multiples of 8 always; of 4 where blocks project by themselves, up to 32 and on the kernels of few rows; nothing else."""
    takes = _lib.load().kiln_w4a16_takes_rank
    assert [r for r in range(0, 67) if takes(4, 2560, 2560, r, -1)] == sorted({4, 12, 20, 28} | set(range(8, 65, 8)))
    assert [m for m in (0, 1, 16, 17, 64, 256, 300) if takes(m, 2560, 2560, 12, -1)] == [1, 16, 17, 64]
    assert takes(4, 2560, 2500, 12, -1) == takes(4, 100, 2560, 12, -1) == 0  # no shape of the kernels
    # long launches of up to 16 rows take fewer of them as they are, or none
    assert [[r for r in (4, 12, 20, 28, 8) if takes(m, 27648, 5120, r, -1)] for m in (1, 8, 16)] == [[8]] * 3
    assert [[r for r in (4, 12, 20, 28) if takes(m, 2560, 9216, r, -1)] for m in (1, 16)] == [[4, 12], [4, 12, 20]]


def test_a_wavefront_without_groups_finishes_no_ranks():
    """1664 = 4 + 4 + 4 + 1 groups: one wavefront of the last slice has any, and two rank tiles are two wavefronts' to finish."""
    L = _lib.load_tuning()
    taken = {}
    for k in (1664, 1792, 2048):
        L.kiln_w4a16_debug_mid(1, 1, 4)
        L.kiln_w4a16_debug_lora_fold(3)
        taken[k] = [L.kiln_w4a16_takes_rank(m, 512, k, r, -1) for m in (17, 32) for r in (12, 20, 28)]
    L.kiln_w4a16_debug_mid(-1, 0, 0)
    L.kiln_w4a16_debug_lora_fold(-1)
    assert taken == {1664: [1, 0, 0] * 2, 1792: [1, 1, 1] * 2, 2048: [1, 1, 1] * 2}
