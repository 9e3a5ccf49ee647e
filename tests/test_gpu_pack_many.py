"""Several weights quantised and packed by one launch (`kiln_w4a16_quantize_and_pack_many_device`), gate and up into their
interleaved pack as well: the same bits as the weights one by one and as the copy that interleaves two packed projections."""
import ctypes

import pytest
import torch

from kiln_amd import _lib, layer_pack, marlin_gemm
from kiln_amd.layer_pack import LayerProjections, PackKind

pytestmark = pytest.mark.gpu
OK = _lib.OK


class Item(ctypes.Structure):
    _fields_ = [("weight", ctypes.c_void_p), ("k", ctypes.c_int), ("n", ctypes.c_int), ("groupsize", ctypes.c_int), ("side", ctypes.c_int),
                ("b", ctypes.c_void_p), ("s", ctypes.c_void_p), ("pair_b", ctypes.c_void_p), ("pair_s", ctypes.c_void_p)]


def _empty(k, n, g):
    return (torch.full((k // 16, 2 * n), -1, dtype=torch.int32, device="cuda"),
            torch.full((1 if g == -1 else k // 128, n), float("nan"), dtype=torch.float16, device="cuda"))


def _weight(k, n, seed, odd):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    w = torch.randn(k * n + 1, device="cuda", generator=gen).to(torch.bfloat16)[1 if odd else 0:][:k * n].view(k, n)   # odd: off the 16-byte grid
    if seed % 3 == 1:
        w[k // 2, ::5] = float("inf")
        w[0, 1::7] = float("nan")
    return w


# one weight, as many as one launch takes, and one and two more; both groupsizes in turn
@pytest.mark.parametrize("count,groupsizes", [(1, (128,)), (1, (-1,)), (7, (128, -1)), (16, (128,)), (17, (128,)), (18, (-1,)), (33, (128, 128, -1))])
def test_many_weights_equal_one_by_one(count, groupsizes):
    shapes = [(128, 256), (384, 512), (2560, 256), (128, 2560), (1280, 1024)]
    calls, made, keep = (Item * count)(), [], []
    for i in range(count):
        (k, n), g = shapes[i // 2 % len(shapes)], groupsizes[i // 2 % len(groupsizes)]     # neighbours are a gate and an up
        w = _weight(k, n, i, odd=i % 4 == 3)
        b, s = _empty(k, n, g)
        if i % 2 == 0:
            pair = _empty(k, 2 * n, g)
        paired = i + 1 < count or i % 2 == 1
        calls[i] = Item(w.data_ptr(), k, n, g, i % 2, b.data_ptr(), s.data_ptr(), *((p.data_ptr() for p in pair) if paired else (None, None)))
        made.append((w, g, b, s, pair if paired else None))
        keep.append(pair)
    st = _lib.load().kiln_w4a16_quantize_and_pack_many_device(calls, count, 0, torch.cuda.current_stream().cuda_stream)
    assert st == OK, _lib.status_string(st)
    for i, (w, g, b, s, pair) in enumerate(made):
        b1, s1 = marlin_gemm.quantize_and_pack_device(w.clone(), g)
        assert torch.equal(b, b1) and torch.equal(s.view(torch.int16), s1.view(torch.int16)), i
        if pair and i % 2 == 1:
            b2, s2 = marlin_gemm.interleave_gate_up_device(made[i - 1][2], made[i - 1][3], b, s, g)
            assert torch.equal(pair[0], b2) and torch.equal(pair[1].view(torch.int16), s2.view(torch.int16)), i


def test_nothing_is_written_if_an_item_is_refused():
    w = _weight(256, 512, 0, odd=False)
    b, s = _empty(256, 512, 128)
    pair = _empty(256, 1024, 128)
    good = (w.data_ptr(), 256, 512, 128, 0, b.data_ptr(), s.data_ptr(), None, None)
    L = _lib.load()
    for bad in ((w.data_ptr(), 255, 512, 128, 0, b.data_ptr(), s.data_ptr(), None, None),
                (w.data_ptr(), 256, 128, 128, 0, b.data_ptr(), s.data_ptr(), None, None),
                (w.data_ptr(), 256, 512, 64, 0, b.data_ptr(), s.data_ptr(), None, None),
                (w.data_ptr(), 128 * 65536, 256, 128, 0, b.data_ptr(), s.data_ptr(), None, None),
                (None, 256, 512, 128, 0, b.data_ptr(), s.data_ptr(), None, None),
                (w.data_ptr(), 256, 512, 128, 0, b.data_ptr(), s.data_ptr(), pair[0].data_ptr(), None),
                (w.data_ptr(), 256, 512, 128, 2, b.data_ptr(), s.data_ptr(), pair[0].data_ptr(), pair[1].data_ptr())):
        calls = (Item * 2)(Item(*good), Item(*bad))
        assert L.kiln_w4a16_quantize_and_pack_many_device(calls, 2, 0, torch.cuda.current_stream().cuda_stream) != OK
    assert L.kiln_w4a16_quantize_and_pack_many_device(None, 0, 0, torch.cuda.current_stream().cuda_stream) == OK
    torch.cuda.synchronize()
    assert bool((b == -1).all()) and bool(s.isnan().all())


@pytest.mark.parametrize("groupsize", [128, -1])
@pytest.mark.parametrize("same_input", [False, True])
def test_layers_get_the_interleaved_pack_of_their_own_gate_and_up(groupsize, same_input):
    def layer(seed):
        shapes = {PackKind.QProj: (256, 512), PackKind.KProj: (256, 256), PackKind.VProj: (256, 256), PackKind.GateProj: (256, 768),
                  PackKind.UpProj: (256, 768), PackKind.DownProj: (768, 256), PackKind.InProjA: (256, 32)}
        return LayerProjections({kind: _weight(*shape, seed + i, odd=False) for i, (kind, shape) in enumerate(shapes.items())})
    layers = [layer(10), layer(20), LayerProjections({PackKind.GateProj: _weight(256, 512, 1, False)}), layer(30)]
    layers[3].weights_t[PackKind.UpProj] = _weight(256, 1024, 5, False)        # of another width: no pair
    stats = layer_pack.pack_layers(layers, groupsize=groupsize, fuse_gate_up=True, fuse_same_input_groups=same_input)
    assert stats["gate_up_fused"] == 2 and layers[2].gate_up_fused is None and layers[3].gate_up_fused is None
    for one in layers[:2]:
        gate, up, fused = one.packed[PackKind.GateProj], one.packed[PackKind.UpProj], one.gate_up_fused
        b, s = marlin_gemm.interleave_gate_up_device(gate.b_packed, gate.scales, up.b_packed, up.scales, groupsize)
        assert torch.equal(fused.b_packed, b) and torch.equal(fused.scales.view(torch.int16), s.view(torch.int16))
        assert (fused.k, fused.n, fused.groupsize) == (256, 1536, groupsize)
