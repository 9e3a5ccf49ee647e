"""The projection of a call with adapters in the units a product leaves whose blocks' wavefronts share K (one block per compute
unit): its blocks of eight wavefronts take 64 rows and whole groups of K.  Where it can go wrong: a last tile of one row, ranks
of every padded width, one K slice and several that meet, a single group to a slice, several shares of one block in turns, row
sums on the way (128-row blocks), per-column scales, the SwiGLU writer.  Against 64 bits, against the plain call (adapters of
zeros), against the projection in a launch in front, and under capture."""
import ctypes

import pytest
import torch

from kiln_amd import _lib, marlin_gemm

pytestmark = pytest.mark.gpu

# rows, K, N, groupsize, ranks; blocks of the projection, tiles of 64 rows
SHAPES = [
    (300, 1024, 8192, 128, (16, 32), 24, 5),      # 8 groups: slices of two groups, five to a tile
    (321, 1024, 8192, 128, (5,), 24, 6),          # one row in the last tile; a rank that is no multiple of 16
    (648, 1920, 3840, -1, (8, 4), 56, 11),
    (603, 2560, 3072, 128, (16, 32), 16, 10),     # one K slice
    (761, 7808, 2560, 128, (32, 32), 16, 12),     # ... of 61 groups; the widest rank
    (1199, 2176, 3072, 128, (16,), 16, 19),       # two tiles to a block, one after the other
    (1200, 2176, 3072, -1, (16, 32, 8), 16, 19),
    (1203, 7296, 2304, -1, (16, 32), 40, 19),     # 128-row blocks: the row sums on the way, two slices
    (706, 6400, 8192, 128, (8, 16), 64, 12),
    (577, 11008, 3072, 128, (4, 4), 16, 10),      # 86 groups to a share, more than there is room for row sums: none are formed
]


def _operands(m, k, n, g, ranks):
    gen = torch.Generator(device="cuda").manual_seed(m + k + n)
    words = torch.randint(-2**31, 2**31, (k // 16, 2 * n), dtype=torch.int64, device="cuda", generator=gen).to(torch.int32)
    scales = (torch.rand(1 if g == -1 else k // g, n, device="cuda", generator=gen) * 0.018 + 0.002).half()
    x = torch.randn(m, k, device="cuda", generator=gen)
    a = (torch.randn(sum(ranks), k, device="cuda", generator=gen) * k ** -0.5).to(torch.bfloat16)
    b = (torch.randn(n, sum(ranks), device="cuda", generator=gen) * 0.1).to(torch.bfloat16)
    return words, scales, [x.to(torch.bfloat16), (x * 0.5 + 0.5).to(torch.bfloat16)], a, b


def _is_inside(m, k, n, blocks, tiles):
    L, plan, cus = _lib.load(), (ctypes.c_int * 8)(), torch.cuda.get_device_properties(0).multi_processor_count
    assert L.kiln_w4a16_debug_gemm_plan(m, n, k, cus, plan) == 0 and (plan[0], plan[7]) == (1, 1)
    assert L.kiln_w4a16_debug_prefill_projection_blocks(m, n, k, cus) == blocks and -(-m // 64) == tiles


@pytest.mark.parametrize("m,k,n,g,ranks,blocks,tiles", SHAPES)
def test_result_against_64_bits(m, k, n, g, ranks, blocks, tiles):
    _is_inside(m, k, n, blocks, tiles)
    words, scales, xs, a, b = _operands(m, k, n, g, ranks)
    w = marlin_gemm.dequant_f32(words, scales, g).double()
    factors = [0.5 + 0.25 * i for i in range(len(ranks))]
    col = torch.tensor([s for r, s in zip(ranks, factors) for _ in range(r)], dtype=torch.float64, device="cuda")
    eager = []
    for x in xs:
        plain = marlin_gemm.marlin_w4a16_gemm(x, words, scales, g)
        assert torch.equal(marlin_gemm.marlin_w4a16_gemm_lora(x, words, scales, g, a, torch.zeros_like(b), ranks, factors), plain)
        y = marlin_gemm.marlin_w4a16_gemm_lora(x, words, scales, g, a, b, ranks, factors)
        t = ((x.double() @ a.double().t()) * col).to(torch.bfloat16)    # rounded once, as T is kept
        product = x.double() @ w
        want = product + t.double() @ b.double().t()
        # one rounding to bf16 (2^-9 of a value's power of two) and f32 sums of a 136-fold surplus, T's ties under 1e-4 of the norm
        err = (y.double() - want).norm(dim=1) / want.norm(dim=1)
        assert float(err.max()) <= 2.0 ** -8, float(err.max())
        h = marlin_gemm.marlin_w4a16_gemm_swiglu_lora(x, words, scales, g, a, b, ranks, factors)
        pairs = want.view(m, n // 16, 2, 8)
        want_h = torch.nn.functional.silu(pairs[:, :, 0].reshape(m, -1)) * pairs[:, :, 1].reshape(m, -1)
        # two factors within 2^-8 less its rounding, and one rounding
        err = (h.double() - want_h).norm(dim=1) / want_h.norm(dim=1)
        assert float(err.max()) <= 2.0 ** -7, float(err.max())
        eager.append(y)
    x, y = xs[0].clone(), torch.empty_like(eager[0])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y.copy_(marlin_gemm.marlin_w4a16_gemm_lora(x, words, scales, g, a, b, ranks, factors))
    for i in (1, 0, 1):
        x.copy_(xs[i])
        y.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y.view(torch.int16), eager[i].view(torch.int16)), i


@pytest.mark.parametrize("m,k,n,g,ranks,blocks,tiles", SHAPES)
def test_inside_and_in_front_agree_in_every_bit(m, k, n, g, ranks, blocks, tiles):
    """... and every call leaves the zeroed prefix of the workspace zero, the sticky word included."""
    L = _lib.load_tuning()
    words, scales, xs, a, b = _operands(m, k, n, g, ranks)
    zeroed = L.kiln_w4a16_workspace_zeroed_bytes()
    ws = torch.full((L.kiln_w4a16_workspace_bytes(m, n, k),), 0xA5, dtype=torch.uint8, device="cuda")
    ws[:zeroed].zero_()
    ranks_c, factors = (ctypes.c_int * len(ranks))(*ranks), (ctypes.c_float * len(ranks))(*[0.5] * len(ranks))

    def call(x):
        out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
        rc = L.kiln_w4a16_gemm_lora(x.data_ptr(), words.data_ptr(), out.data_ptr(), scales.data_ptr(), m, n, k, ws.data_ptr(), g,
                                    torch.cuda.current_device(), torch.cuda.current_stream().cuda_stream, a.data_ptr(),
                                    b.data_ptr(), sum(ranks), len(ranks), ranks_c, factors)
        assert rc == _lib.OK, _lib.status_string(rc)
        torch.cuda.synchronize()
        assert int(ws[:zeroed].max()) == 0
        return out.view(torch.int16)

    try:
        L.kiln_w4a16_debug_lora_fold(0)
        in_front = [call(x) for x in xs]
        L.kiln_w4a16_debug_lora_fold(-1)
        for i in range(10):
            assert torch.equal(call(xs[i % 2]), in_front[i % 2]), i
    finally:
        L.kiln_w4a16_debug_lora_fold(-1)
