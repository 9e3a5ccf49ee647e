"""The matrix-core kernel's 128-row blocks in launches of several rounds add the row sums at every change of group
(a multiply-add in place of the change of scale's multiplication) instead of in a contraction behind the main loop.
Checked against the product in 64 bits where that can go wrong: one group (no change at all), two and three (every
change is the first or the last), ragged rows, K slices, per-column scales, groups whose scale is zero, and
activations with a mean, which make the surplus far larger than the result."""
import ctypes

import pytest
import torch

from kiln_amd import _lib, marlin_gemm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n,g", [
    (8192, 128, 28672, 128),
    (4097, 256, 16384, 128),
    (8191, 384, 8192, -1),
    (2048, 2560, 18432, 128),
    (777, 2560, 18432, -1),
    (8191, 512, 8192, 128),
    (4000, 9216, 2560, 128),
])
def test_result_against_64_bits(m, k, n, g):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    L, plan = _lib.load_tuning(), (ctypes.c_int * 8)()
    assert L.kiln_w4a16_debug_prefill_rowsum_producers(m, n, k, cus) == 0  # the sums come from a launch in front
    assert L.kiln_w4a16_debug_gemm_plan(m, n, k, cus, plan) == 0 and (plan[0], plan[2], plan[3]) == (1, 128, 256)
    gen = torch.Generator(device="cuda").manual_seed(m + k + n)
    words = torch.randint(-2**31, 2**31, (k // 16, 2 * n), dtype=torch.int64, device="cuda", generator=gen).to(torch.int32)
    scales = (torch.rand(1 if g == -1 else k // g, n, device="cuda", generator=gen) * 0.018 + 0.002).half()
    if scales.shape[0] > 1:
        scales[scales.shape[0] // 2, ::7] = 0
    x = torch.randn(m, k, device="cuda", generator=gen).to(torch.bfloat16)
    w = marlin_gemm.dequant_f32(words, scales, g).double()
    for xt in (x, (x.float() * 0.5 + 0.5).to(torch.bfloat16)):
        y = marlin_gemm.marlin_w4a16_gemm(xt, words, scales, g)
        again = marlin_gemm.marlin_w4a16_gemm(xt, words, scales, g)
        assert torch.equal(y, again)
        want = xt.double() @ w
        # one rounding to bf16 (half an ulp: 2^-9 of the value's power of two) and f32 sums of 136-fold surplus,
        # whose error is 1e-4 to 2e-4 of the result's norm on these inputs: together under 2^-8 of a row's norm
        err = (y.double() - want).norm(dim=1) / want.norm(dim=1)
        assert float(err.max()) <= 2.0 ** -8, float(err.max())
        # and no more than the rounding alone but for ties it decides the other way
        off = (y.double() - want.to(torch.bfloat16).double()).norm() / want.norm()
        assert float(off) <= 5e-4, float(off)
