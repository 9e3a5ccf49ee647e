"""An MLP whose gate+up launch writes the row sums of H in f32 for a down launch that adds them at its changes of group:
bit-equal to the two entry points, both against 64 bits, and the sums themselves.  The writer's blocks as whole tiles and
in K slices, the other form of the sums beside it."""
import ctypes

import pytest
import torch

from kiln_amd import _lib, marlin_gemm

pytestmark = pytest.mark.gpu


def _plan(m, k, n):
    L, plan = _lib.load(), (ctypes.c_int * 8)()
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert L.kiln_w4a16_debug_gemm_plan(m, n, k, cus, plan) == 0
    several = (plan[0], plan[2], plan[3]) == (1, 128, 256) and L.kiln_w4a16_debug_prefill_rowsum_producers(m, n, k, cus) == 0
    return several, several and plan[4] * 256 < n and plan[5] > 1


@pytest.mark.parametrize("m,hidden,inter,n_down,g,writer_sliced,plain", [
    (4096, 2560, 9216, 2560, 128, False, True),    # whole tiles write, a down launch of several rounds reads
    (2048, 2560, 9216, 5120, 128, True, True),     # the last round of the writer in two K slices
    (2300, 2560, 4096, 8192, -1, True, True),      # three, ragged rows, one scale per column
    (2048, 2560, 9216, 2560, 128, True, False),    # a down launch of one round: the other form
])
def test_sums_of_h(m, hidden, inter, n_down, g, writer_sliced, plain):
    assert _plan(m, hidden, 2 * inter) == (True, writer_sliced)
    assert _plan(m, inter, n_down)[0] == plain
    L = _lib.load()
    gen = torch.Generator(device="cuda").manual_seed(m + inter)

    def weight(k, n):
        words = torch.randint(-2**31, 2**31, (k // 16, 2 * n), dtype=torch.int64, device="cuda", generator=gen).to(torch.int32)
        return words, (torch.rand(1 if g == -1 else k // g, n, device="cuda", generator=gen) * 0.01 + 0.002).half()

    (b_gu, s_gu), (bd, sd) = weight(hidden, 2 * inter), weight(inter, n_down)
    x = (torch.randn(m, hidden, device="cuda", generator=gen) * 0.5 + 0.25).to(torch.bfloat16)
    z, size = L.kiln_w4a16_workspace_zeroed_bytes(), L.kiln_w4a16_mlp_workspace_bytes(m, hidden, inter, n_down)
    ws = torch.full((size + 256,), 0xA5, dtype=torch.uint8, device="cuda")
    ws[:z].zero_()
    y = torch.empty(m, n_down, dtype=torch.bfloat16, device="cuda")
    for _ in range(2):
        rc = L.kiln_w4a16_mlp(x.data_ptr(), b_gu.data_ptr(), s_gu.data_ptr(), bd.data_ptr(), sd.data_ptr(), y.data_ptr(), m, hidden, inter,
                              n_down, ws.data_ptr(), g, torch.cuda.current_device(), torch.cuda.current_stream().cuda_stream)
        assert rc == _lib.OK, _lib.status_string(rc)
    torch.cuda.synchronize()
    assert int(ws[:z].count_nonzero()) == 0 and bool((ws[size:] == 0xA5).all())
    h = marlin_gemm.marlin_w4a16_gemm_swiglu(x, b_gu, s_gu, g)
    assert torch.equal(y.view(torch.int16), marlin_gemm.marlin_w4a16_gemm(h, bd, sd, g).view(torch.int16))

    # the sums, behind H in the workspace: c = -136 * sum of H over a group, [group][row], in a quarter of the operand's room
    sums, groups = ws[size - m * (inter // 128) * 16:size], inter // 128
    if plain:
        got = sums[:groups * m * 4].clone().view(torch.float32).view(groups, m)
        want = -136.0 * h.double().view(m, groups, 128).sum(dim=2).t()
        # 128 f32 additions of values of at most max |H|: each partial sum rounds by half an ulp, 2^-24 of it
        bound = 136.0 * 128 * 2.0 ** -24 * h.double().abs().view(m, groups, 128).sum(dim=2).t() + 1e-30
        assert bool(((got.double() - want).abs() <= bound).all())
        assert bool((sums[groups * m * 4:] == 0xA5).all())
    else:
        assert bool((sums != 0xA5).any(dim=0))

    w = marlin_gemm.dequant_f32(b_gu, s_gu, g).double().view(hidden, inter // 8, 2, 8)
    gate, up = (x.double() @ w[:, :, side].reshape(hidden, inter) for side in (0, 1))
    want = torch.nn.functional.silu(gate) * up
    # one rounding to bf16 and f32 sums, as for the plain product; silu keeps or shrinks a relative error of this size
    err = (h.double() - want).norm(dim=1) / want.norm(dim=1)
    assert float(err.max()) <= 2.0 ** -8, float(err.max())
    want = h.double() @ marlin_gemm.dequant_f32(bd, sd, g).double()
    off = (y.double() - want.to(torch.bfloat16).double()).norm() / want.norm()
    assert float(off) <= (5e-4 if plain else 4e-3), float(off)    # (the other form keeps the contraction's error)
