"""The matrix-core kernel's blocks whose wavefronts share K, each half of them taking half of the block's groups (launches of
at most one block per compute unit).  Checked against the product in 64 bits where the split can go wrong: an odd number of
groups (the second half begins with a group that is not its own), K slices whose last one is shorter, down to a single group,
ragged rows, both block heights and widths, row sums formed by the blocks and by the units without one, per-column scales,
groups whose scale is zero; row sums added at the changes of group; with adapters, in the SwiGLU writer and under capture."""
import ctypes

import pytest
import torch

from kiln_amd import _lib, marlin_gemm

pytestmark = pytest.mark.gpu
RANKS, SCALES = (16, 32), (0.5, 1.0)

SHAPES = [
    (1500, 768, 1536, 128),     # the shortest: six groups, three to a half
    (1500, 896, 1536, -1),      # seven
    (1100, 3968, 512, 128),     # six slices of six groups, the last of one
    (513, 2048, 2048, 128),     # three slices, the last of four groups; one row in the last row block
    (600, 11008, 2048, 128),    # slices of 29 and 28 groups
    (1300, 1536, 1536, 128),    # blocks of 128 columns
    (1300, 1664, 1536, -1),     # the same, 13 groups
    (777, 2688, 2560, 128),
    (777, 9216, 2560, 128),     # 128-row blocks, row sums from the units without a block
    (640, 11008, 4096, -1),     # the same, slices of 29 groups, the last of 28
    (1300, 4096, 4096, 128),    # 128-row blocks, whole tiles for two thirds of the units
    (3001, 3200, 2560, 128),    # row sums from a launch in front, added at the changes of group: 25 groups
    (1900, 4096, 4096, -1),     # the same, 32 groups
    (1024, 3072, 8192, 128),    # the same, a tile for every unit, 24 groups
    # tiles dealt to the dies one after the other (13, 14 and 25 row blocks)
    (777, 3584, 4608, 128),     # 64-row blocks, row sums from the blocks
    (850, 3584, 4608, -1),      # ... from a launch in front
    (3137, 3200, 2560, 128),    # 128-row blocks
]


def _operands(m, k, n, g):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    plan = (ctypes.c_int * 8)()
    assert _lib.load().kiln_w4a16_debug_gemm_plan(m, n, k, cus, plan) == 0 and (plan[0], plan[6], plan[7]) == (1, 0, 1)
    gen = torch.Generator(device="cuda").manual_seed(m + k + n)
    words = torch.randint(-2**31, 2**31, (k // 16, 2 * n), dtype=torch.int64, device="cuda", generator=gen).to(torch.int32)
    scales = (torch.rand(1 if g == -1 else k // g, n, device="cuda", generator=gen) * 0.018 + 0.002).half()
    if scales.shape[0] > 1:
        scales[scales.shape[0] // 2, ::7] = 0
    x = torch.randn(m, k, device="cuda", generator=gen)
    return words, scales, [x.to(torch.bfloat16), (x * 0.5 + 0.5).to(torch.bfloat16)]


@pytest.mark.parametrize("m,k,n,g", SHAPES)
def test_result_against_64_bits(m, k, n, g):
    words, scales, xs = _operands(m, k, n, g)
    w = marlin_gemm.dequant_f32(words, scales, g).double()
    eager = []
    for x in xs:
        y = marlin_gemm.marlin_w4a16_gemm(x, words, scales, g)
        assert torch.equal(marlin_gemm.marlin_w4a16_gemm(x, words, scales, g).view(torch.int16), y.view(torch.int16))
        widths = [marlin_gemm.marlin_w4a16_gemm(x, words, scales, g, thread_k=k, thread_n=t) for t in (128, 256)]
        assert torch.equal(widths[0].view(torch.int16), widths[1].view(torch.int16))
        want = x.double() @ w
        # one rounding to bf16 (half an ulp: 2^-9 of the value's power of two) and f32 sums of a 136-fold surplus, 2e-4 of
        # the result's norm, 1e-3 where the activations have a mean: together under 2^-8 of a row's norm
        err = (y.double() - want).norm(dim=1) / want.norm(dim=1)
        assert float(err.max()) <= 2.0 ** -8, float(err.max())
        eager.append(y)
    x, y = xs[0].clone(), torch.empty_like(eager[0])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y.copy_(marlin_gemm.marlin_w4a16_gemm(x, words, scales, g))
    for i in (1, 0, 1):
        x.copy_(xs[i])
        y.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y.view(torch.int16), eager[i].view(torch.int16)), i


@pytest.mark.parametrize("m,k,n,g", SHAPES)
def test_adapters_and_the_swiglu_writer(m, k, n, g):
    words, scales, xs = _operands(m, k, n, g)
    w = marlin_gemm.dequant_f32(words, scales, g).double()
    gen = torch.Generator(device="cuda").manual_seed(1)
    a = (torch.randn(sum(RANKS), k, device="cuda", generator=gen) * k ** -0.5).to(torch.bfloat16)
    b = (torch.randn(n, sum(RANKS), device="cuda", generator=gen) * 0.1).to(torch.bfloat16)
    zeros = torch.zeros_like(b)
    col = torch.tensor([s for r, s in zip(RANKS, SCALES) for _ in range(r)], dtype=torch.float64, device="cuda")
    for x in xs:
        plain = marlin_gemm.marlin_w4a16_gemm(x, words, scales, g)
        assert torch.equal(marlin_gemm.marlin_w4a16_gemm_lora(x, words, scales, g, a, zeros, RANKS, SCALES), plain)
        y = marlin_gemm.marlin_w4a16_gemm_lora(x, words, scales, g, a, b, RANKS, SCALES)
        t = ((x.double() @ a.double().t()) * col).to(torch.bfloat16)    # rounded once, as T is kept
        want = x.double() @ w + t.double() @ b.double().t()
        # the plain call's bound, which has room for T's ties (under 1e-4 of the norm)
        err = (y.double() - want).norm(dim=1) / want.norm(dim=1)
        assert float(err.max()) <= 2.0 ** -8, float(err.max())
        h = marlin_gemm.marlin_w4a16_gemm_swiglu(x, words, scales, g)
        assert torch.equal(marlin_gemm.marlin_w4a16_gemm_swiglu_lora(x, words, scales, g, a, zeros, RANKS, SCALES), h)
        # gate and up in turns of 8 columns; the bound of the two factors, each within 2^-8 less its rounding, and one rounding
        pairs = (x.double() @ w).view(m, n // 16, 2, 8)
        gate, up = pairs[:, :, 0].reshape(m, -1), pairs[:, :, 1].reshape(m, -1)
        want_h = torch.nn.functional.silu(gate) * up
        err = (h.double() - want_h).norm(dim=1) / want_h.norm(dim=1)
        assert float(err.max()) <= 2.0 ** -7, float(err.max())


@pytest.mark.parametrize("m,k,n,g", [(1005, 1024, 14336, 128), (883, 896, 18176, -1), (1371, 1024, 10496, 128)])
def test_words_of_a_folded_launch_outlast_both_halves(m, k, n, g):
    """Halves of at most four groups with row sums from the launch's first blocks: no barrier of the block lies between the
    last half's look at the words and the end of the main loop, so the block counts itself as done (and the last one zeroes
    the words) only where the halves meet.  Such short halves come from a caller's count of compute units."""
    sms = 1024
    L, plan = _lib.load(), (ctypes.c_int * 8)()
    assert L.kiln_w4a16_debug_gemm_plan(m, n, k, sms, plan) == 0 and (plan[0], plan[2], plan[5], plan[6], plan[7]) == (1, 64, 1, 0, 1)
    assert L.kiln_w4a16_debug_prefill_rowsum_producers(m, n, k, sms) > 0 and k // 128 <= 8
    gen = torch.Generator(device="cuda").manual_seed(m)
    words = torch.randint(-2**31, 2**31, (k // 16, 2 * n), dtype=torch.int64, device="cuda", generator=gen).to(torch.int32)
    scales = (torch.rand(1 if g == -1 else k // g, n, device="cuda", generator=gen) * 0.018 + 0.002).half()
    x = torch.randn(m, k, device="cuda", generator=gen).to(torch.bfloat16)
    ws = torch.zeros(L.kiln_w4a16_workspace_bytes_tuned(m, n, k, -1, -1, sms), dtype=torch.uint8, device="cuda")
    zeroed = L.kiln_w4a16_workspace_zeroed_bytes()
    want = x.double() @ marlin_gemm.dequant_f32(words, scales, g).double()
    first = None
    for _ in range(20):
        y = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
        assert L.kiln_marlin_w4a16_gemm(x.data_ptr(), words.data_ptr(), y.data_ptr(), scales.data_ptr(), m, n, k, ws.data_ptr(), g, 0,
                                        torch.cuda.current_stream().cuda_stream, -1, -1, sms, 16) == _lib.OK
        torch.cuda.synchronize()
        assert int(ws[:zeroed].max()) == 0      # words and counts as they were, and nobody gave up waiting
        err = (y.double() - want).norm(dim=1) / want.norm(dim=1)
        assert float(err.max()) <= 2.0 ** -8, float(err.max())     # the bound of the calls above
        first = y if first is None else first
        assert torch.equal(y.view(torch.int16), first.view(torch.int16))


@pytest.mark.parametrize("sms,m,k,n,rows,halves", [(64, 515, 1280, 2304, 128, 0), (64, 543, 2176, 1280, 64, 1), (128, 516, 1536, 1792, 64, 1),
                                                   (128, 769, 3072, 4352, 128, 1), (200, 771, 768, 3328, 64, 1),
                                                   (200, 1547, 1280, 3328, 128, 0)])
def test_tiles_dealt_to_the_dies_for_other_counts_of_units(sms, m, k, n, rows, halves):
    """Tiles that fit a caller's count of compute units, and that no rectangle of dies holds."""
    L, plan = _lib.load(), (ctypes.c_int * 8)()
    assert L.kiln_w4a16_debug_gemm_plan(m, n, k, sms, plan) == 0
    assert (plan[0], plan[2], plan[6], plan[7]) == (1, rows, 0, halves)
    gen = torch.Generator(device="cuda").manual_seed(m)
    words = torch.randint(-2**31, 2**31, (k // 16, 2 * n), dtype=torch.int64, device="cuda", generator=gen).to(torch.int32)
    scales = (torch.rand(k // 128, n, device="cuda", generator=gen) * 0.018 + 0.002).half()
    x = torch.randn(m, k, device="cuda", generator=gen).to(torch.bfloat16)
    ws = torch.zeros(L.kiln_w4a16_workspace_bytes_tuned(m, n, k, -1, -1, sms), dtype=torch.uint8, device="cuda")
    want = x.double() @ marlin_gemm.dequant_f32(words, scales, 128).double()
    y = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
    assert L.kiln_marlin_w4a16_gemm(x.data_ptr(), words.data_ptr(), y.data_ptr(), scales.data_ptr(), m, n, k, ws.data_ptr(), 128, 0,
                                    torch.cuda.current_stream().cuda_stream, -1, -1, sms, 16) == _lib.OK
    err = (y.double() - want).norm(dim=1) / want.norm(dim=1)
    assert float(err.max()) <= 2.0 ** -8, float(err.max())      # the bound of the calls above
    assert int(ws[:L.kiln_w4a16_workspace_zeroed_bytes()].max()) == 0


@pytest.mark.parametrize("m,k,n,g", [(777, 2688, 2560, 128), (1300, 1664, 1536, -1)])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
def test_what_is_not_finite_in_the_group_that_both_halves_read(m, k, n, g, value):
    """With an odd number of groups the second half reads the first's last group and multiplies what it got by 0: rows with an
    infinity or NaN there are not finite, as with one set of wavefronts (the surplus of the codes is inf - inf), and no other
    row is touched."""
    words, scales, xs = _operands(m, k, n, g)
    plan = (ctypes.c_int * 8)()
    _lib.load().kiln_w4a16_debug_gemm_plan(m, n, k, torch.cuda.get_device_properties(0).multi_processor_count, plan)
    groups = -(-(k // 128) // plan[5])     # of a block: the first slice's
    assert groups % 2 == 1
    clean = marlin_gemm.marlin_w4a16_gemm(xs[0], words, scales, g)
    x, hit = xs[0].clone(), torch.tensor([0, 63, 64, m - 1], device="cuda")
    x[hit, (groups // 2) * 128 + 77] = value
    y = marlin_gemm.marlin_w4a16_gemm(x, words, scales, g)
    assert not bool(torch.isfinite(y[hit]).any())
    others = torch.ones(m, dtype=torch.bool, device="cuda")
    others[hit] = False
    assert torch.equal(y[others].view(torch.int16), clean[others].view(torch.int16))
