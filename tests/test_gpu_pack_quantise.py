"""The device quantiser's one-read kernel where it can go wrong: quotients on and next to its rounding boundaries for every
fp16 mantissa a scale can have, a weight off the 16-byte grid, and packed projections laid side by side -- all
against the host quantiser, bit for bit."""
import numpy as np
import pytest
import torch

from kiln_amd import layer_pack, marlin_proj
from kiln_amd.layer_pack import LayerProjections, PackKind
from kiln_amd.marlin_gemm import pack

pytestmark = pytest.mark.gpu


def _same_as_host(w: torch.Tensor, groupsize: int):
    b, s = pack.quantize_and_pack_device(w, groupsize)
    b_host, s_host, _ = pack.quantize_and_pack(w.float().cpu().numpy(), *w.shape, groupsize, want_dequant=False)
    assert np.array_equal(s.cpu().numpy().view(np.uint16), np.asarray(s_host).view(np.uint16)), "scales differ"
    assert np.array_equal(b.cpu().numpy(), b_host), "packed words differ"


@pytest.mark.parametrize("groupsize", [128, -1])
@pytest.mark.parametrize("exponent", [-20, -9, 0, 9])
def test_every_scale_mantissa_and_weights_around_its_halves(groupsize, exponent):
    # column c's largest weight is (128 + c % 128) * 2^exponent (every bf16 mantissa); its other weights are the bf16
    # values nearest to the halves of its step, and their neighbours on either side
    n = 256
    top = (128.0 + np.arange(n) % 128) * 2.0 ** exponent
    scale = (2 * top / 15).astype(np.float32).astype(np.float16).astype(np.float64)
    halves = np.concatenate([np.arange(-7.5, 8.0, 1.0)] * 8)[:127]
    w = np.concatenate([top[None], halves[:, None] * scale[None]]).astype(np.float32)
    t = torch.from_numpy(w).bfloat16().view(torch.int16)
    t[1:] += torch.from_numpy((np.arange(127) // 16 % 3 - 1).astype(np.int16))[:, None]
    t = t.view(torch.bfloat16).cuda()
    t = torch.where(t.abs() > t[:1], t[:1].expand_as(t) * torch.sign(t), t)     # the first row stays the largest
    _same_as_host(t.contiguous(), groupsize)


@pytest.mark.parametrize("groupsize", [128, -1])
def test_weight_off_the_16_byte_grid(groupsize):
    k, n = 256, 256
    base = (torch.randn(k * n + 8, device="cuda") * 0.05).bfloat16()
    for off in (1, 4, 7):
        _same_as_host(base[off:off + k * n].view(k, n), groupsize)


@pytest.mark.parametrize("groupsize", [128, -1])
def test_side_by_side_packs_share_memory_and_hold_the_separate_packs_bits(groupsize):
    kinds = layer_pack.SAME_INPUT_GROUPS[0]
    ws = {kind: (torch.randn(384, n, device="cuda") * 0.05).bfloat16() for kind, n in zip(kinds, (512, 256, 768))}
    layer = LayerProjections(dict(ws))
    layer_pack.pack_layers([layer], groupsize=groupsize, fuse_same_input_groups=True)
    fused = layer.same_input_fused[kinds]
    assert fused.b_packed.data_ptr() == layer.packed[PackKind.QProj].b_packed.data_ptr()
    apart = [marlin_proj.pack_from_bf16(ws[k], groupsize) for k in kinds]
    for kind, p in zip(kinds, apart):
        assert torch.equal(layer.packed[kind].b_packed, p.b_packed) and torch.equal(layer.packed[kind].scales, p.scales)
    assert torch.equal(fused.b_packed.view(-1), torch.cat([p.b_packed.view(-1) for p in apart]))
    assert torch.equal(fused.scales.view(-1), torch.cat([p.scales.view(-1) for p in apart]))


def test_gptq_tensors_larger_than_the_pinned_stage(monkeypatch):
    monkeypatch.setattr(marlin_proj, "_STAGE_BYTES", 40 << 10)
    monkeypatch.setattr(marlin_proj, "_FIRST_PIECE_BYTES", 8 << 10)
    k, n = 384, 768
    q = torch.randint(-2**31, 2**31 - 1, (k // 8, n), dtype=torch.int32)
    s = torch.rand(k // 128, n).half()
    p = marlin_proj.pack_from_gptq(q, s, None, 128, "cuda")
    b, st = pack.repack_gptq(q.numpy(), s.numpy(), None, 128)
    assert np.array_equal(p.b_packed.cpu().numpy(), b) and np.array_equal(p.scales.cpu().numpy(), st)
    assert marlin_proj.matmul_bf16(torch.zeros(2, k, dtype=torch.bfloat16, device="cuda"), p).abs().max() == 0
