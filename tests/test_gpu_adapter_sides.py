"""Calls whose projections keep adapters of their own, read where they lie by the launch: against the same call on the
stacked set -- in every bit where its projection runs in the launch too (up to four adapters, or more than 16 rows) -- and against the
product in 64 bits.  Tiles that cross from one projection to the next, columns without adapters, one side alone, five to
eight adapters, the widest stacked rank, K slices, replays of a captured call.  That the launch did read them where they
lie is shown, not assumed: the entry point for such calls, which refuses all others, gives the same bits."""
import ctypes

import pytest
import torch

from kiln_amd import _calls, _lib, layer_pack, lora, marlin_gemm
from kiln_amd.layer_pack import LayerProjections, PackKind
from kiln_amd.marlin_proj import MarlinPackedProj

QKV = (PackKind.QProj, PackKind.KProj, PackKind.VProj)


class Side(ctypes.Structure):
    _fields_ = [("lora_a", ctypes.c_void_p), ("lora_b", ctypes.c_void_p), ("rank", ctypes.c_int), ("first_row", ctypes.c_int), ("rows", ctypes.c_int)]


def _sides(*sides):
    return (Side * len(sides))(*(Side(16, 16, *s) for s in sides))


def _takes(m, n, k, sides, swiglu=0, n_adapters=2):
    return _lib.load().kiln_w4a16_takes_adapter_sides(m, n, k, sides, len(sides), swiglu, n_adapters, -1)


def test_what_is_taken():
    qkv = _sides((16, 0, 8192), (16, 8192, 1024), (16, 9216, 1024))
    assert [_takes(m, 10240, 2560, qkv, 0, 6) for m in (0, 1, 16, 17, 128, 2048)] == [0, 1, 1, 1, 1, 0]
    assert _takes(4, 10240, 2560, qkv, 0, 8) == 1 and _takes(4, 10240, 2560, qkv, 0, 9) == 0
    assert _takes(4, 10240, 2560, _sides((16, 0, 8192), (12, 8192, 1024))) == 0           # not whole units of eight
    assert _takes(4, 10240, 2560, _sides((40, 0, 8192), (32, 8192, 1024))) == 0           # more than 64 together
    assert _takes(4, 10240, 2560, _sides((16, 8192, 1024), (16, 0, 8192))) == 0           # out of order
    assert _takes(4, 10240, 2560, _sides((16, 0, 8192), (16, 8000, 1024))) == 0           # columns of two sides
    assert _takes(4, 10240, 2560, _sides((16, 0, 8192), (16, 9728, 1024))) == 0           # columns past the last
    assert _takes(4, 10240, 2560, _sides((8, 0, 2048), (8, 2048, 2048), (8, 4096, 2048), (8, 6144, 2048))) == 0
    gate_up = _sides((16, 0, 9216), (16, 8, 9216))
    assert _takes(4, 18432, 2560, gate_up, 1) == 1
    assert _takes(4, 18432, 2560, _sides((16, 8, 9216), (16, 0, 9216)), 1) == 0
    assert _takes(4, 18432, 2560, _sides((16, 0, 9216), (16, 4, 9216)), 1) == 0
    assert _takes(4, 18432, 2560, _sides((16, 0, 4608), (16, 8, 9216)), 1) == 0


def test_what_is_refused():
    L = _lib.load()
    ok, ranks, scales = _sides((16, 0, 512), (16, 512, 512)), (ctypes.c_int * 2)(16, 16), (ctypes.c_float * 2)(1, 1)

    def call(m=4, n=1024, k=512, sides=ok, count=2, swiglu=0, adapters=2, ranks=ranks, scales=scales):
        return L.kiln_w4a16_gemm_adapter_sides(16, 16, 16, 16, m, n, k, 16, 128, -1, None, sides, count, swiglu, adapters, ranks, scales)

    assert call(m=0) == _lib.OK
    assert call(m=-1) == call(n=1000) == call(k=500) == 1          # the problem's shape
    argument, shape = call(sides=None), call(count=4, sides=_sides(*[(8, 256 * i, 256) for i in range(4)]))
    assert argument == call(adapters=0) == call(ranks=(ctypes.c_int * 2)(16, 8)) == call(ranks=None) == call(count=0) != _lib.OK
    assert shape == call(m=2048) == call(sides=_sides((16, 0, 512), (12, 512, 512)), ranks=(ctypes.c_int * 2)(16, 12)) != _lib.OK
    assert argument != shape
    assert call(sides=(Side * 2)(Side(8, 16, 16, 0, 512), Side(16, 16, 16, 512, 512))) == argument  # off 16 bytes


def _adapters(gen, k, n, ranks, first_scale=0):
    if ranks is None:
        return None
    return lora.stack_adapters([lora.LoraProjectionWeights(torch.randn(r, k, device="cuda", generator=gen).mul(k ** -0.5).bfloat16(),
                                                           torch.randn(n, r, device="cuda", generator=gen).mul(0.1).bfloat16()) for r in ranks],
                               tuple(0.5 + 0.25 * (first_scale + i) for i in range(len(ranks))))


def _all_adapters(gen, k, widths, ranks):
    """Every projection's, no two adapters of one scale."""
    made, count = [], 0
    for n, r in zip(widths, ranks):
        made.append(_adapters(gen, k, n, r, count))
        count += len(r or ())
    return made


def _packed(gen, k, n, g):
    words = torch.randint(-2**31, 2**31, (k // 16, 2 * n), dtype=torch.int64, device="cuda", generator=gen).to(torch.int32)
    return MarlinPackedProj(words, (torch.rand(1 if g == -1 else k // g, n, device="cuda", generator=gen) * 0.018 + 0.002).half(), g, k, n)


def _where_they_lie(x, fused, adapters, firsts, swiglu):
    """The call through the entry point that takes unstacked adapters only: the result, or None where it refuses."""
    own = [(a, first) for a, first in zip(adapters, firsts) if a is not None]
    sides = (Side * len(own))(*(Side(a.a_cat.data_ptr(), a.b_cat.data_ptr(), a.a_cat.shape[0], first, a.b_cat.shape[0]) for a, first in own))
    ranks, scales = sum((a.ranks for a, _ in own), ()), sum((a.scales for a, _ in own), ())
    (m, k), n = x.shape, fused.n
    L, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    ws = marlin_gemm._workspace(x.device, stream, L.kiln_w4a16_workspace_bytes(m, n, k))
    out = torch.full((m, n // 2 if swiglu else n), float("nan"), dtype=torch.bfloat16, device=x.device)
    takes = L.kiln_w4a16_takes_adapter_sides(m, n, k, sides, len(own), swiglu, len(ranks), x.device.index)
    st = L.kiln_w4a16_gemm_adapter_sides(x.data_ptr(), fused.b_packed.data_ptr(), out.data_ptr(), fused.scales.data_ptr(), m, n, k,
                                         ws.data_ptr(), fused.groupsize, x.device.index, stream, sides, len(own), swiglu, len(ranks),
                                         (ctypes.c_int * len(ranks))(*ranks), (ctypes.c_float * len(ranks))(*scales))
    assert st == (_lib.OK if takes else _lib.ERR_KERN_SHAPE)
    return out if takes else None


# (k, columns of each projection, ranks of each one's adapters, groupsize, rows up to which the launch reads them itself)
SIDE_BY_SIDE = [
    (2560, (8192, 1024, 1024), ((8, 8), (8, 8), (8, 8)), 128, 100),         # six adapters; blocks of three tiles cross at 8192
    (2560, (8192, 1024, 1024), ((8, 8, 8), (8, 8), (8, 8, 8)), 128, 100),   # eight, rank 64 together
    (2560, (8192, 1024, 1024), ((8, 8), None, (16,)), -1, 100),
    (2560, (8192, 4096), ((24,), (32, 8)), 128, 64),                        # rank 64 together
    (2560, (1024, 512), ((8,), (16, 8, 8, 16)), 128, 100),                  # five adapters
    (9216, (1280, 1280), ((8,), (8,)), 128, 64),                            # K slices
    (1024, (256, 256), ((8,), (16, 8, 8, 16)), -1, 100),
    (512, (256, 256, 512), (None, (8,), None), 128, 100),
    (128, (256, 256), ((8,), (8,)), 128, 16),                               # one group
]
# (k, columns of gate and of up, ranks of each one's adapters, groupsize, rows as above)
GATE_AND_UP = [
    (2560, 9216, ((8, 8), (8, 8)), 128, 128),
    (2560, 9216, (None, (16,)), 128, 128),
    (1024, 2816, ((8, 8, 8), (16, 24)), 128, 128),                          # five adapters, rank 64 together
    (1024, 2816, ((32,), None), -1, 128),
    (1024, 256, ((16, 8), (40,)), 128, 128),
    (256, 256, ((8,), (8,)), 128, 16),
]
SIDE_ROWS = [1, 4, 9, 16, 17, 33, 64, 100]  # (from 17 on the mid-M kernel: one and two row blocks, two runs)
GATE_ROWS = [1, 5, 16, 24, 50, 128]


def test_the_cases_below_are_taken():
    def ask(m, k, widths, ranks, swiglu):
        sides, first = [], 0
        for i, (n, r) in enumerate(zip(widths, ranks)):
            if r is not None:
                sides.append((sum(r), 8 * i if swiglu else first, n))
            first += n
        return _takes(m, first, k, _sides(*sides), swiglu, sum(len(r or ()) for r in ranks))

    for k, widths, ranks, _, most in SIDE_BY_SIDE:
        assert [m for m in SIDE_ROWS if ask(m, k, widths, ranks, 0)] == [m for m in SIDE_ROWS if m <= most], (k, widths, ranks)
    for k, n, ranks, _, most in GATE_AND_UP:
        assert [m for m in GATE_ROWS if ask(m, k, (n, n), ranks, 1)] == [m for m in GATE_ROWS if m <= most], (k, n, ranks)


@pytest.mark.gpu
@pytest.mark.parametrize("m", SIDE_ROWS)
@pytest.mark.parametrize("k,widths,ranks,g,most", SIDE_BY_SIDE)
def test_side_by_side(m, k, widths, ranks, g, most):
    gen = torch.Generator(device="cuda").manual_seed(m * k + sum(widths))
    fused = _packed(gen, k, sum(widths), g)
    layer = LayerProjections({})
    kinds = QKV[:len(widths)]
    for kind, n in zip(kinds, widths):
        layer.packed[kind] = MarlinPackedProj(fused.b_packed, fused.scales, g, k, n)  # (only the width is read)
    layer.same_input_fused[kinds] = fused
    adapters = _all_adapters(gen, k, widths, ranks)
    loras = dict(zip(kinds, adapters))
    x = torch.randn(m, k, device="cuda", generator=gen).bfloat16()
    firsts = [sum(widths[:i]) for i in range(len(widths))]
    own = _where_they_lie(x, fused, adapters, firsts, 0)  # (leaves the workspace without which the extension takes no call)
    assert (own is not None) == (m <= most)
    got = _calls.linear_sides(x, fused.b_packed, fused.scales, g, False, tuple(adapters), widths, 1.0, True)
    assert got is not None
    got = torch.cat(got, dim=1)
    assert torch.equal(torch.cat(layer.forward_same_input(kinds, x, loras), dim=1).view(torch.int16), got.view(torch.int16))
    stacked = lora.fuse_column_blocks([loras[kind] for kind in kinds], widths)
    want = lora.proj_forward(x, fused, stacked)
    if own is not None:
        assert torch.equal(own.view(torch.int16), got.view(torch.int16))
    if own is None or len(stacked.ranks) <= 4 or m > 16:  # (there the stacked set is projected inside too)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    exact = x.double() @ marlin_gemm.dequant_f32(fused.b_packed, fused.scales, g).double()
    low, col = torch.zeros_like(exact), 0
    for r, s in zip(stacked.ranks, stacked.scales):
        low += s * (x.double() @ stacked.a_cat[col:col + r].double().t()) @ stacked.b_cat[:, col:col + r].double().t()
        col += r
    # the result rounded once to bf16 and T once per slice of K, half an ulp each: 2^-8 of a row of either at most
    bound = 2.0 ** -8 * ((exact + low).norm(dim=1) + low.norm(dim=1))
    for y in (got, want):
        assert bool(((y.double() - exact - low).norm(dim=1) <= bound).all())


@pytest.mark.gpu
@pytest.mark.parametrize("m", GATE_ROWS)
@pytest.mark.parametrize("k,inter,ranks,g,most", GATE_AND_UP)
def test_gate_and_up(m, k, inter, ranks, g, most):
    gen = torch.Generator(device="cuda").manual_seed(m * k + inter)
    fused = _packed(gen, k, 2 * inter, g)
    x = torch.randn(m, k, device="cuda", generator=gen).bfloat16()
    sides = _all_adapters(gen, k, (inter, inter), ranks)

    def call():
        return lora.swiglu_forward(x, fused, *sides)

    own = _where_they_lie(x, fused, sides, (0, 8), 1)
    assert (own is not None) == (m <= most)
    assert _calls.linear_sides(x, fused.b_packed, fused.scales, g, True, tuple(sides), (inter, inter), 1.0, False) is not None
    got = call()
    if own is not None:
        assert torch.equal(own.view(torch.int16), got.view(torch.int16))
    present = [s for s in sides if s is not None]
    b_cat = marlin_gemm.interleave_gate_up_lora_b(*(s.b_cat if s is not None else None for s in sides), inter)
    want = marlin_gemm.marlin_w4a16_gemm_swiglu_lora(x, fused.b_packed, fused.scales, g, torch.cat([s.a_cat for s in present]).contiguous(), b_cat,
                                                     sum((s.ranks for s in present), ()), sum((s.scales for s in present), ()))
    if own is None or sum(len(s.ranks) for s in present) <= 4 or m > 16:
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    w = marlin_gemm.dequant_f32(fused.b_packed, fused.scales, g).double().view(k, inter // 8, 2, 8)
    halves = []
    for i, side in enumerate(sides):
        y = x.double() @ w[:, :, i].reshape(k, inter)
        col = 0
        for r, s in zip(side.ranks, side.scales) if side is not None else ():
            y = y + s * (x.double() @ side.a_cat[col:col + r].double().t()) @ side.b_cat[:, col:col + r].double().t()
            col += r
        halves.append(y)
    want = torch.nn.functional.silu(halves[0]) * halves[1]
    # as above: H rounded once, T in bf16; silu and the product keep or shrink a relative error of the terms' size
    assert bool(((got.double() - want).norm(dim=1) <= 2.0 ** -7 * want.norm(dim=1)).all())
    # captured and replayed, with eager calls in between
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        out = call()
    for _ in range(4):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), got.view(torch.int16))
        assert torch.equal(call().view(torch.int16), got.view(torch.int16))
