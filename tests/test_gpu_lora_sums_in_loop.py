"""Calls with adapters whose product runs in several rounds of 128-row blocks add the row sums where a plain call does, at
the changes of group: with adapters of zeros they equal the plain call in every bit, whether the projection runs inside
the product's launch or in front of it, and the error against 64 bits is the plain call's."""
import ctypes

import pytest
import torch

from kiln_amd import _lib, marlin_gemm

pytestmark = pytest.mark.gpu
RANKS, SCALES = (16, 32), (0.5, 1.0)

# several rounds of 128-row blocks
SHAPES = [
    (2048, 2560, 18432, 128),   # whole rounds and a rest in K slices
    (1100, 2560, 18432, -1),    # a ragged last row block, one scale per column
    (777, 2560, 18432, 128),    # the product fills the chip's slots: the projection runs in front
    (4096, 9216, 2560, 128),    # 64 rows per block of the projection: in front as well
    (8191, 128, 28672, 128),    # one group: no look at the words under the main loop
    (4097, 256, 16384, 128),    # two: the look is asked for in the first
    (8191, 384, 8192, -1),
]


def _operands(m, k, n, g, zero_b):
    gen = torch.Generator(device="cuda").manual_seed(m + k + n)
    words = torch.randint(-2**31, 2**31, (k // 16, 2 * n), dtype=torch.int64, device="cuda", generator=gen).to(torch.int32)
    scales = (torch.rand(1 if g == -1 else k // g, n, device="cuda", generator=gen) * 0.018 + 0.002).half()
    x = torch.randn(m, k, device="cuda", generator=gen)
    xs = [x.to(torch.bfloat16), (x * 0.5 + 0.5).to(torch.bfloat16)]
    a = (torch.randn(sum(RANKS), k, device="cuda", generator=gen) * k ** -0.5).to(torch.bfloat16)
    b = torch.randn(n, sum(RANKS), device="cuda", generator=gen) * (0.0 if zero_b else 0.1)
    return words, scales, xs, a, b.abs().to(torch.bfloat16) if zero_b else b.to(torch.bfloat16)


def _several_rounds_of_128_rows(m, k, n):
    L, plan = _lib.load(), (ctypes.c_int * 8)()
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert L.kiln_w4a16_debug_gemm_plan(m, n, k, cus, plan) == 0 and (plan[0], plan[2], plan[3]) == (1, 128, 256)
    assert L.kiln_w4a16_debug_prefill_rowsum_producers(m, n, k, cus) == 0


@pytest.mark.parametrize("m,k,n,g", SHAPES)
def test_adapters_with_zero_b_equal_the_plain_call_bit_for_bit(m, k, n, g):
    _several_rounds_of_128_rows(m, k, n)
    words, scales, xs, a, b = _operands(m, k, n, g, zero_b=True)
    for x in xs:
        plain = marlin_gemm.marlin_w4a16_gemm(x, words, scales, g)
        with_adapters = marlin_gemm.marlin_w4a16_gemm_lora(x, words, scales, g, a, b, RANKS, SCALES)
        assert torch.equal(plain.view(torch.int16), with_adapters.view(torch.int16))
        plain = marlin_gemm.marlin_w4a16_gemm_swiglu(x, words, scales, g)
        with_adapters = marlin_gemm.marlin_w4a16_gemm_swiglu_lora(x, words, scales, g, a, b, RANKS, SCALES)
        assert torch.equal(plain.view(torch.int16), with_adapters.view(torch.int16))


@pytest.mark.parametrize("m,k,n,g", SHAPES)
def test_projection_inside_and_in_front_agree_and_meet_64_bits(m, k, n, g):
    L = _lib.load_tuning()
    words, scales, xs, a, b = _operands(m, k, n, g, zero_b=False)
    z = L.kiln_w4a16_workspace_zeroed_bytes()
    size = L.kiln_w4a16_workspace_bytes(m, n, k)
    ws = torch.full((size + 256,), 0xA5, dtype=torch.uint8, device="cuda")
    ws[:z].zero_()
    ranks, lora_scales = (ctypes.c_int * 2)(*RANKS), (ctypes.c_float * 2)(*SCALES)

    def call(x):
        out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
        rc = L.kiln_w4a16_gemm_lora(x.data_ptr(), words.data_ptr(), out.data_ptr(), scales.data_ptr(), m, n, k, ws.data_ptr(), g,
                                    torch.cuda.current_device(), torch.cuda.current_stream().cuda_stream, a.data_ptr(),
                                    b.data_ptr(), sum(RANKS), len(RANKS), ranks, lora_scales)
        assert rc == _lib.OK, _lib.status_string(rc)
        torch.cuda.synchronize()
        assert int(ws[:z].count_nonzero()) == 0 and bool((ws[size:] == 0xA5).all())
        return out

    try:
        L.kiln_w4a16_debug_lora_fold(0)
        in_front = [call(x) for x in xs]
        L.kiln_w4a16_debug_lora_fold(-1)
        for i in range(8):                      # alternating activations: every launch sees its own T
            assert torch.equal(call(xs[i % 2]).view(torch.int16), in_front[i % 2].view(torch.int16)), i
    finally:
        L.kiln_w4a16_debug_lora_fold(-1)
    w = marlin_gemm.dequant_f32(words, scales, g).double()
    col = torch.tensor([s for r, s in zip(RANKS, SCALES) for _ in range(r)], dtype=torch.float64, device="cuda")
    for x, y in zip(xs, in_front):
        t = ((x.double() @ a.double().t()) * col).to(torch.bfloat16)    # rounded once, as T is kept
        want = x.double() @ w + t.double() @ b.double().t()
        # the plain call's bound (5e-4 of the norm beyond the rounding to bf16), and T: f32 sums that round the other way
        # at a tie, one in some 2^13 of its values by half an ulp (2^-9), under 1e-4 of the norm of a delta smaller than the result
        off = (y.double() - want.to(torch.bfloat16).double()).norm() / want.norm()
        assert float(off) <= 6e-4, float(off)
