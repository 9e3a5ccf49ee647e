"""Overrides on shapes whose automatic call adds the row sums at the changes of group: one that leaves the plan as it is
gives the automatic call's bits, and blocks of 128 and of 256 columns agree in every bit."""
import ctypes

import pytest
import torch

from kiln_amd import _lib, marlin_gemm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n,g", [
    (2048, 2560, 18432, 128),    # a rest in K slices, whole tiles with thread_k = k
    (8192, 2560, 18432, 128),    # whole tiles only
    (1100, 2560, 18432, -1),
    (8191, 128, 28672, 128),     # one group
    (4097, 256, 16384, 128),
    (4000, 9216, 2560, 128),
])
def test_unchanged_plans_and_block_widths(m, k, n, g):
    L, plan = _lib.load(), (ctypes.c_int * 8)()
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert L.kiln_w4a16_debug_gemm_plan(m, n, k, cus, plan) == 0 and (plan[0], plan[2], plan[3]) == (1, 128, 256)
    assert L.kiln_w4a16_debug_prefill_rowsum_producers(m, n, k, cus) == 0
    gen = torch.Generator(device="cuda").manual_seed(m + k + n)
    words = torch.randint(-2**31, 2**31, (k // 16, 2 * n), dtype=torch.int64, device="cuda", generator=gen).to(torch.int32)
    scales = (torch.rand(1 if g == -1 else k // g, n, device="cuda", generator=gen) * 0.018 + 0.002).half()
    x = (torch.randn(m, k, device="cuda", generator=gen) * 0.5 + 0.25).to(torch.bfloat16)

    def call(**overrides):
        return marlin_gemm.marlin_w4a16_gemm(x, words, scales, g, **overrides).view(torch.int16)

    automatic = call()
    assert torch.equal(call(thread_n=256), automatic)
    assert torch.equal(call(thread_k=128), automatic)         # asks for more slices than there are: none are added
    whole = call(thread_k=k, thread_n=256)
    assert torch.equal(call(thread_k=k, thread_n=128), whole)
    if plan[5] == 1 or plan[4] * 256 == n:                    # no K slices to begin with
        assert torch.equal(whole, automatic)
    # the bound of two bf16 roundings of sums in another order
    want = x.double() @ marlin_gemm.dequant_f32(words, scales, g).double()
    off = (whole.view(torch.bfloat16).double() - want.to(torch.bfloat16).double()).norm() / want.norm()
    assert float(off) <= 5e-4, float(off)
