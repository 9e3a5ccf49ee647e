"""The calls that go to the library without ctypes (`kiln_amd/_calls.py`) against the wrappers' checked route: the same
kernels run on the same operands, so the results are the same bits; the adapters' stacked set of a fused call (one
launch of `kiln_w4a16_stack_adapters`) against the torch operations that build it there."""
import pytest
import torch

from kiln_amd import _calls, layer_pack, lora, marlin_gemm, marlin_proj
from kiln_amd.layer_pack import LayerProjections, PackKind

pytestmark = pytest.mark.gpu
QKV = (PackKind.QProj, PackKind.KProj, PackKind.VProj)


def _layer(k=256, inter=512, g=128):
    shapes = {PackKind.QProj: 512, PackKind.KProj: 256, PackKind.VProj: 256, PackKind.GateProj: inter, PackKind.UpProj: inter}
    layer = LayerProjections({kind: (torch.randn(k, n, device="cuda") * 0.05).bfloat16() for kind, n in shapes.items()})
    layer_pack.pack_layers([layer], groupsize=g, fuse_gate_up=True, fuse_same_input_groups=True)
    return layer


def _adapters(k, n, ranks):
    if ranks is None:
        return None
    two = [lora.LoraProjectionWeights((torch.randn(r, k, device="cuda") * 0.05).bfloat16(), (torch.randn(n, r, device="cuda") * 0.1).bfloat16()) for r in ranks]
    return two[0] if len(two) == 1 else lora.stack_adapters(two, tuple(0.5 + i for i in range(len(two))))


@pytest.fixture
def both(monkeypatch):
    """(result of the direct call, which must have been taken; result of the checked route)"""
    def run(fn):
        fn()                                     # the workspace exists from here on
        taken = []
        for name in ("linear", "linear_lora", "linear_sides", "mlp"):
            real = getattr(_calls, name)
            monkeypatch.setattr(_calls, name, lambda *a, real=real: taken.append(real(*a)) or taken[-1])
        direct = fn()
        assert taken and taken[0] is not None
        for name in ("linear", "linear_lora", "linear_sides", "mlp"):
            monkeypatch.setattr(_calls, name, lambda *a: None)
        checked = fn()
        monkeypatch.undo()
        torch.cuda.synchronize()
        return direct, checked
    return run


@pytest.mark.parametrize("m", [1, 16, 17, 130])
@pytest.mark.parametrize("ranks", [(None, None, None), ((8,), None, (16, 8)), ((4,), (3, 2), None), ((16, 8), (16,), (24,)), (None, (7,), None)])
def test_projections_of_one_input(both, m, ranks):
    layer = _layer()
    x = torch.randn(m, 256, device="cuda").bfloat16()
    loras = {kind: _adapters(256, layer.packed[kind].n, r) for kind, r in zip(QKV, ranks)}
    direct, checked = both(lambda: layer.forward_same_input(QKV, x, loras, 0.75))
    # (the checked route pads no stacked rank here but in proj_forward: zeros either way, which add nothing)
    for a, b in zip(direct, checked):
        assert a.shape == b.shape and torch.equal(a, b)


@pytest.mark.parametrize("m", [1, 16, 130])
@pytest.mark.parametrize("ranks", [((8,), (8,)), ((16, 8), None), (None, (5,)), ((3,), (16, 16)), ((16, 16), (16, 16))])
def test_gate_and_up(both, m, ranks):
    layer = _layer(g=-1)
    x = torch.randn(1, m, 256, device="cuda").bfloat16()
    g, u = (_adapters(256, 512, r) for r in ranks)
    direct, checked = both(lambda: layer.swiglu(x, g, u, 0.75))
    assert direct.shape == (1, m, 512) and torch.equal(direct, checked)


@pytest.mark.parametrize("ranks", [(8,), (16, 32), (4, 8), (7,)])
def test_one_projection(both, ranks):
    w = marlin_proj.pack_from_bf16((torch.randn(384, 512, device="cuda") * 0.05).bfloat16(), 128)
    l = _adapters(384, 512, ranks)
    for x in (torch.randn(5, 384, device="cuda").bfloat16(), torch.randn(2, 33, 384, device="cuda").bfloat16()):
        for adapters in (None, l):
            direct, checked = both(lambda: lora.proj_forward(x, w, adapters, 0.5))
            assert direct.shape == (*x.shape[:-1], 512) and torch.equal(direct, checked)


def test_mlp_and_given_outputs(both):
    layer = _layer()
    gu = layer.gate_up_fused
    down = marlin_proj.pack_from_bf16((torch.randn(512, 256, device="cuda") * 0.05).bfloat16(), 128)
    x = torch.randn(40, 256, device="cuda").bfloat16()
    direct, checked = both(lambda: marlin_gemm.marlin_w4a16_mlp(x, gu.b_packed, gu.scales, down.b_packed, down.scales, 128))
    assert torch.equal(direct, checked)
    out = torch.empty(40, 1024, dtype=torch.bfloat16, device="cuda")
    direct, checked = both(lambda: marlin_gemm.marlin_w4a16_gemm(x, gu.b_packed, gu.scales, 128, out=out))
    assert direct is not None and direct.data_ptr() == out.data_ptr() == checked.data_ptr()


@pytest.mark.parametrize("make", [lambda x: x.float(), lambda x: x.t().contiguous().t(), lambda x: x.cpu(), lambda x: x[0]],
                         ids=["dtype", "strides", "cpu", "rank"])
def test_anything_else_goes_to_the_checked_route(make):
    w = marlin_proj.pack_from_bf16((torch.randn(256, 256, device="cuda") * 0.05).bfloat16(), 128)
    x = make(torch.randn(4, 256, device="cuda").bfloat16())
    assert _calls.linear(x, w.b_packed, w.scales, 128, None, False, 2) is None
