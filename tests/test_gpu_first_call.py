"""The first call on a stream, which finds no workspace, and calls on a strided x give the bits of every other call, also where
unstacked adapters, or a rank that is no multiple of 8, are projected elsewhere than their stacked and padded set."""
import pytest
import torch

from kiln_amd import lora, marlin_gemm
from kiln_amd.layer_pack import LayerProjections, PackKind
from kiln_amd.marlin_proj import MarlinPackedProj

QKV = (PackKind.QProj, PackKind.KProj, PackKind.VProj)


def _packed(gen, k, n):
    words = torch.randint(-2**31, 2**31, (k // 16, 2 * n), dtype=torch.int64, device="cuda", generator=gen).to(torch.int32)
    return MarlinPackedProj(words, (torch.rand(k // 128, n, device="cuda", generator=gen) * 0.018 + 0.002).half(), 128, k, n)


def _adapters(gen, k, n, ranks):
    return lora.stack_adapters([lora.LoraProjectionWeights(torch.randn(r, k, device="cuda", generator=gen).mul(k ** -0.5).bfloat16(),
                                                           torch.randn(n, r, device="cuda", generator=gen).mul(0.1).bfloat16()) for r in ranks],
                               tuple(0.5 + 0.25 * i for i in range(len(ranks))))


def _calls_of(gen, k):
    """name -> a call on x, of the kinds whose adapters are read as they lie"""
    widths = (2048, 512, 512)
    layer, fused, wide = LayerProjections({}), _packed(gen, k, sum(widths)), _packed(gen, k, 2 * 2816)
    for kind, n in zip(QKV, widths):
        layer.packed[kind] = MarlinPackedProj(fused.b_packed, fused.scales, 128, k, n)  # (only the width is read)
    layer.same_input_fused[QKV] = fused
    six, two = ({kind: _adapters(gen, k, n, r) for kind, n in zip(QKV, widths)} for r in ((8, 8), (8,)))
    gate, up, twelve = _adapters(gen, k, 2816, (8, 4, 4)), _adapters(gen, k, 2816, (8, 4, 4)), _adapters(gen, k, sum(widths), (8, 4))
    return {
        "side by side, six adapters": lambda x: torch.cat(layer.forward_same_input(QKV, x, six), dim=-1),
        "side by side, three": lambda x: torch.cat(layer.forward_same_input(QKV, x, two), dim=-1),
        "gate and up, six": lambda x: lora.swiglu_forward(x, wide, gate, up),
        "rank 12": lambda x: lora.proj_forward(x, fused, twelve),
    }


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 5, 11, 16, 24, 50])
@pytest.mark.parametrize("k", [1024, 2560])
def test_the_first_call_of_a_stream_and_a_strided_x_give_the_same_bits(k, m):
    gen = torch.Generator(device="cuda").manual_seed(k + m)
    for name, call in _calls_of(gen, k).items():
        x = torch.randn(m, k, device="cuda", generator=gen).bfloat16()
        strided = torch.empty(m, 2 * k, dtype=torch.bfloat16, device="cuda")[:, :k]
        strided.copy_(x)
        torch.cuda.synchronize()
        with torch.cuda.stream(torch.cuda.Stream()):
            marlin_gemm._workspaces.clear()
            first = call(x)
            assert len(marlin_gemm._workspaces) == 1
            others = [call(x), call(strided), call(x.unsqueeze(0))[0], call(x)]
        torch.cuda.synchronize()
        for y in others:
            assert torch.equal(first.view(torch.int16), y.view(torch.int16)), name
