"""The group size of a call is 128 or -1 as the caller's integer says, not as its lower 32 bits do: anything else is
refused by every entry point, and an integer beyond 64 bits leaves no exception behind in a call that goes on."""
import pytest
import torch

from kiln_amd import _calls, lora, marlin_gemm, marlin_proj
from kiln_amd.marlin_proj import MarlinPackedProj

NARROWS_TO_128 = 2 ** 32 + 128


@pytest.mark.parametrize("groupsize", [2 ** 70, -2 ** 70, NARROWS_TO_128])
def test_quantize_answers_none_and_raises_nothing(groupsize):
    assert _calls.quantize(((torch.zeros(128, 256, dtype=torch.bfloat16), groupsize),), ()) is None


@pytest.mark.gpu
@pytest.mark.parametrize("groupsize", [2 ** 70, NARROWS_TO_128, 2 ** 32 - 1, 64])
def test_every_gemm_entry_point_refuses(groupsize):
    x = torch.randn(4, 256, device="cuda").bfloat16()
    w = marlin_proj.pack_from_bf16((torch.randn(256, 512, device="cuda") * 0.05).bfloat16(), 128)
    down = marlin_proj.pack_from_bf16((torch.randn(256, 256, device="cuda") * 0.05).bfloat16(), 128)
    a, b = torch.zeros(8, 256, dtype=torch.bfloat16, device="cuda"), torch.zeros(512, 8, dtype=torch.bfloat16, device="cuda")
    one, half = lora.LoraProjectionWeights(a, b), lora.LoraProjectionWeights(a, b[:256].contiguous())

    def packed(g):
        return MarlinPackedProj(w.b_packed, w.scales, g, w.k, w.n)

    entries = [
        lambda g: marlin_gemm.marlin_w4a16_gemm(x, w.b_packed, w.scales, g),
        lambda g: marlin_gemm.marlin_w4a16_gemm_swiglu(x, w.b_packed, w.scales, g),
        lambda g: marlin_gemm.marlin_w4a16_mlp(x, w.b_packed, w.scales, down.b_packed, down.scales, g),
        lambda g: marlin_gemm.marlin_w4a16_gemm_lora(x, w.b_packed, w.scales, g, a, b, (8,), (1.0,)),
        lambda g: marlin_gemm.marlin_w4a16_gemm_swiglu_lora(x, w.b_packed, w.scales, g, a, b, (8,), (1.0,)),
        lambda g: marlin_proj.matmul_bf16(x, packed(g)),
        lambda g: lora.proj_forward(x, packed(g), one),
        lambda g: lora.swiglu_forward(x, packed(g), half),
    ]
    for call in entries:
        assert torch.isfinite(call(128)).all()
        with pytest.raises(marlin_gemm.MarlinGemmError, match="groupsize must be -1 or 128"):
            call(groupsize)


@pytest.mark.gpu
def test_packing_refuses_an_integer_beyond_64_bits():
    w = torch.randn(256, 512, device="cuda").bfloat16()
    with pytest.raises(marlin_proj.MarlinProjError, match="groupsize must be -1 or 128"):
        marlin_proj.pack_from_bf16(w, 2 ** 70)
    with pytest.raises(marlin_gemm.MarlinGemmError, match="groupsize"):
        marlin_gemm.quantize_and_pack_device(w, NARROWS_TO_128)
