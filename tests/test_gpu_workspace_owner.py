"""`marlin_gemm._workspaces` is the only owner of the wrappers' workspaces: the direct calls (`_calls`) use the entry that
is there at the time of the call, and an entry that is dropped is freed."""
import pytest
import torch

from kiln_amd import _calls, _lib, marlin_gemm

pytestmark = pytest.mark.gpu
M, K, N = 1024, 2560, 18432       # row sums in the workspace behind its zeroed prefix


def _operands():
    gen = torch.Generator(device="cuda").manual_seed(3)
    words = torch.randint(-2**31, 2**31, (K // 16, 2 * N), dtype=torch.int64, device="cuda", generator=gen).to(torch.int32)
    scales = (torch.rand(K // 128, N, device="cuda", generator=gen) * 0.01 + 0.002).half()
    return torch.randn(M, K, device="cuda", generator=gen).bfloat16(), words, scales


def test_a_dropped_workspace_is_freed_and_not_used_again():
    x, words, scales = _operands()
    stream = torch.cuda.Stream()
    key = (torch.cuda.current_device(), stream.cuda_stream)
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        first = marlin_gemm.marlin_w4a16_gemm(x, words, scales, 128)
        assert _calls.linear(x, words, scales, 128, None, False, 2) is not None
        stream.synchronize()
        size = marlin_gemm._workspaces[key].numel()
        before = torch.cuda.memory_allocated()
        del marlin_gemm._workspaces[key]
        assert torch.cuda.memory_allocated() <= before - size
        assert _calls.linear(x, words, scales, 128, None, False, 2) is None
        again = marlin_gemm.marlin_w4a16_gemm(x, words, scales, 128)
        assert key in marlin_gemm._workspaces and torch.equal(first, again)
        stream.synchronize()


def test_direct_calls_use_the_workspace_that_the_health_check_sees():
    x, words, scales = _operands()
    stream = torch.cuda.Stream()
    key, prefix = (torch.cuda.current_device(), stream.cuda_stream), _lib.load().kiln_w4a16_workspace_zeroed_bytes()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        want = marlin_gemm.marlin_w4a16_gemm(x, words, scales, 128)
        mine = torch.full((marlin_gemm._workspaces[key].numel() + 4096,), 0xA5, dtype=torch.uint8, device="cuda")
        mine[:prefix].zero_()
        marlin_gemm._workspaces[key] = mine
        y = _calls.linear(x, words, scales, 128, None, False, 2)
        stream.synchronize()
        assert torch.equal(y, want) and bool((mine[prefix:-4096] != 0xA5).any()) and bool((mine[-4096:] == 0xA5).all())
        # a tensor that is no workspace is left to the checked route
        marlin_gemm._workspaces[key] = mine[::2]
        assert _calls.linear(x, words, scales, 128, None, False, 2) is None
        marlin_gemm._workspaces[key] = mine
        assert marlin_gemm.workspace_wait_status() == 0
        del marlin_gemm._workspaces[key]
