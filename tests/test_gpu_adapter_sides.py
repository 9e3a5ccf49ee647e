"""Calls whose projections keep adapters of their own, read where they lie by the launch: against the same call on the
stacked set -- in every bit where its projection runs in the launch too (up to four adapters, or more than 16 rows) -- and against the
product in 64 bits.  Tiles that cross from one projection to the next, columns without adapters, one side alone, the
widest stacked rank, K slices, replays of a captured call."""
import ctypes

import pytest
import torch

from kiln_amd import _lib, layer_pack, lora, marlin_gemm
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


def _adapters(gen, k, n, ranks):
    if ranks is None:
        return None
    return lora.stack_adapters([lora.LoraProjectionWeights(torch.randn(r, k, device="cuda", generator=gen).mul(k ** -0.5).bfloat16(),
                                                           torch.randn(n, r, device="cuda", generator=gen).mul(0.1).bfloat16()) for r in ranks],
                               tuple(0.5 + 0.25 * i for i in range(len(ranks))))


def _packed(gen, k, n, g):
    words = torch.randint(-2**31, 2**31, (k // 16, 2 * n), dtype=torch.int64, device="cuda", generator=gen).to(torch.int32)
    return MarlinPackedProj(words, (torch.rand(1 if g == -1 else k // g, n, device="cuda", generator=gen) * 0.018 + 0.002).half(), g, k, n)


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 4, 9, 16, 17, 33, 64, 100])  # (from 17 on the mid-M kernel: one and two row blocks, two runs)
@pytest.mark.parametrize("k,widths,ranks,g", [
    (2560, (8192, 1024, 1024), ((8, 8), (8, 8), (8, 8)), 128),      # six adapters; blocks of three tiles cross at 8192
    (2560, (8192, 1024, 1024), ((8, 8), None, (16,)), -1),
    (2560, (8192, 4096), ((24,), (32, 8)), 128),                    # rank 64 together
    (9216, (1280, 1280), ((8,), (8,)), 128),                        # K slices
    (256, (256, 256, 512), (None, (8,), None), 128),
    (128, (256, 256), ((8,), (16, 8, 8, 16)), 128),                 # one group
])
def test_side_by_side(m, k, widths, ranks, g):
    gen = torch.Generator(device="cuda").manual_seed(m * k + sum(widths))
    fused = _packed(gen, k, sum(widths), g)
    layer = LayerProjections({})
    kinds = QKV[:len(widths)]
    for kind, n in zip(kinds, widths):
        layer.packed[kind] = MarlinPackedProj(fused.b_packed, fused.scales, g, k, n)  # (only the width is read)
    layer.same_input_fused[kinds] = fused
    loras = {kind: _adapters(gen, k, n, r) for kind, n, r in zip(kinds, widths, ranks)}
    x = torch.randn(m, k, device="cuda", generator=gen).bfloat16()
    got = torch.cat(layer.forward_same_input(kinds, x, loras), dim=1)
    stacked = lora.fuse_column_blocks([loras[kind] for kind in kinds], widths)
    want = lora.proj_forward(x, fused, stacked)
    if len(stacked.ranks) <= 4 or m > 16:  # (there the stacked set is projected inside too)
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
@pytest.mark.parametrize("m", [1, 5, 16, 24, 50, 128])
@pytest.mark.parametrize("k,inter,ranks,g", [
    (2560, 9216, ((8, 8), (8, 8)), 128),
    (2560, 9216, (None, (16,)), 128),
    (1024, 2816, ((32,), None), -1),
    (256, 256, ((16, 8), (40,)), 128),
])
def test_gate_and_up(m, k, inter, ranks, g):
    gen = torch.Generator(device="cuda").manual_seed(m * k + inter)
    fused = _packed(gen, k, 2 * inter, g)
    x = torch.randn(m, k, device="cuda", generator=gen).bfloat16()
    sides = [_adapters(gen, k, inter, r) for r in ranks]

    def call():
        return lora.swiglu_forward(x, fused, *sides)

    got = call()
    present = [s for s in sides if s is not None]
    b_cat = marlin_gemm.interleave_gate_up_lora_b(*(s.b_cat if s is not None else None for s in sides), inter)
    want = marlin_gemm.marlin_w4a16_gemm_swiglu_lora(x, fused.b_packed, fused.scales, g, torch.cat([s.a_cat for s in present]).contiguous(), b_cat,
                                                     sum((s.ranks for s in present), ()), sum((s.scales for s in present), ()))
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
