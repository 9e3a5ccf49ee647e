"""The weights that run side by side go to the quantiser ahead of the others where they are many: the same words and scales
as one weight at a time, on either side of the size from which they do, and with nothing else to pack."""
import pytest
import torch

from kiln_amd import marlin_proj


@pytest.mark.gpu
@pytest.mark.parametrize("groupsize", [128, -1])
@pytest.mark.parametrize("columns", [3840, 4096, 6912, 7168])  # of 2048 rows: below and from 14 Mi weights on
@pytest.mark.parametrize("others", [0, 1, 3])
def test_the_run_ahead_and_the_rest(columns, others, groupsize):
    gen = torch.Generator(device="cuda").manual_seed(columns + others)
    shapes = [(2048, columns - 512), (2048, 256), (2048, 256)] + [(512, 768), (1024, 512), (1024, 512)][:others]
    weights = [torch.randn(k, n, device="cuda", generator=gen).mul(k ** -0.5).bfloat16() for k, n in shapes]
    pairs = ((4, 5),) if others == 3 else ()
    for _ in range(2):
        packed, fused = marlin_proj.pack_on_device_with_pairs([(w, groupsize) for w in weights], ((0, 1, 2),), pairs)
        for w, p in zip(weights, packed):
            alone = marlin_proj.pack_from_bf16(w, groupsize)
            assert torch.equal(p.b_packed, alone.b_packed) and torch.equal(p.scales.view(torch.int16), alone.scales.view(torch.int16))
        first = packed[0].b_packed
        assert packed[1].b_packed.data_ptr() == first.data_ptr() + first.numel() * 4  # side by side in memory
        assert len(fused) == len(pairs)
