"""The host tensors a GPTQ loader holds: plain ones, `Parameter`s, subclasses of either with and without `requires_grad`, a
subclass that runs its operations itself.  All of them take the device's route."""
import numpy as np
import pytest
import torch

from kiln_amd import _calls, marlin_proj
from kiln_amd.marlin_gemm import pack

K, N, G = 256, 512, 128


class LoaderParameter(torch.nn.Parameter):
    pass


class LoaderTensor(torch.Tensor):
    pass


class Wrapped(torch.Tensor):
    """Holds a tensor and runs every operation on it."""

    @staticmethod
    def __new__(cls, held):
        w = torch.Tensor._make_wrapper_subclass(cls, held.shape, strides=held.stride(), dtype=held.dtype, device=held.device)
        w.held = held
        return w

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        out = func(*(a.held if isinstance(a, Wrapped) else a for a in args), **(kwargs or {}))
        first = args[0]
        return cls(out) if isinstance(first, Wrapped) and isinstance(out, torch.Tensor) else out


FORMS = {
    "tensor": lambda t: t,
    "parameter": lambda t: torch.nn.Parameter(t, requires_grad=t.is_floating_point()),
    "parameter subclass": lambda t: LoaderParameter(t, requires_grad=False),
    "parameter subclass with grad": lambda t: LoaderParameter(t, requires_grad=t.is_floating_point()),
    "tensor subclass": lambda t: t.as_subclass(LoaderTensor),
}


def _tensors(seed=0):
    gen = torch.Generator().manual_seed(seed)
    q = torch.randint(-2**31, 2**31, (K // 8, N), dtype=torch.int64, generator=gen).to(torch.int32)
    s = torch.rand(K // G, N, generator=gen).half()
    return q, s, torch.full((K // G, N // 8), 0x88888888 - 2**32, dtype=torch.int32)


def _takes(q, s, z):
    """Does the device's route take these?  (Where there is no device, it fails on that, behind its checks.)"""
    if torch.cuda.is_available():
        torch.cuda.init()
    try:
        return _calls.repack(q, s, z, K, N, G, 0, 1 << 20, 1 << 20) is not None
    except RuntimeError:
        assert not torch.cuda.is_available()
        return True


@pytest.mark.parametrize("form", FORMS)
def test_what_takes_the_devices_route(form):
    q, s, z = _tensors()
    as_form = FORMS[form]
    assert _takes(as_form(q), s, z) and _takes(q, as_form(s), z) and _takes(q, s, as_form(z)) and _takes(*map(as_form, (q, s, z)))
    assert not _takes(as_form(q), as_form(s.float()), z) and not _takes(as_form(q)[:-1], s, z) and not _takes(q.t().contiguous().t(), s, z)


def test_zero_points_that_cannot_be_read_in_place_are_the_host_routes():
    q, s, z = _tensors()
    assert _takes(Wrapped(q), Wrapped(s), z) and not _takes(q, s, Wrapped(z))
    # zeros that have no memory, words that stand for their negatives, memory that was given back
    assert not _takes(q, s, torch._efficientzerotensor(z.shape, dtype=torch.int32)) and not _takes(q, s, torch._neg_view(z))
    z.untyped_storage().resize_(0)
    assert not _takes(q, s, z)


@pytest.mark.gpu
@pytest.mark.parametrize("form", [*FORMS, "wrapped"])
@pytest.mark.parametrize("stage", [32 << 20, 16 << 10])   # in one piece, in several
def test_same_packs_from_every_form(form, stage, monkeypatch):
    monkeypatch.setattr(marlin_proj, "_STAGE_BYTES", stage)
    monkeypatch.setattr(marlin_proj, "_FIRST_PIECE_BYTES", min(stage, marlin_proj._FIRST_PIECE_BYTES))
    q, s, z = _tensors(1)
    as_form = FORMS.get(form, Wrapped)
    p = marlin_proj.pack_from_gptq(as_form(q), as_form(s), z if form == "wrapped" else as_form(z), G, "cuda")
    b, tiled = pack.repack_gptq(q.numpy(), s.numpy(), None, G)
    assert np.array_equal(p.b_packed.cpu().numpy(), b) and np.array_equal(p.scales.cpu().numpy().view(np.uint16), tiled.view(np.uint16))
    assert type(p.b_packed) is type(p.scales) is torch.Tensor and not p.scales.requires_grad


def test_a_forked_childs_call_is_refused(monkeypatch):
    """torch refuses a child that was forked after the parent used the GPU; the device given with its index or without."""
    monkeypatch.setattr(torch.cuda, "_is_in_bad_fork", lambda: True)
    for device in ("cuda", "cuda:0"):
        with pytest.raises(RuntimeError, match="forked subprocess"):
            marlin_proj.pack_from_gptq(*_tensors(), G, device)


def test_scales_with_a_gradient_on_the_host_route():
    """A shape the library has no pack for yields None, whatever form its tensors come in."""
    q = torch.zeros(4, 100, dtype=torch.int32)
    for as_form in FORMS.values():
        s = as_form(torch.ones(1, 100).half())
        assert marlin_proj.pack_from_gptq(as_form(q), s, None, -1, "cpu") is None
        assert marlin_proj.pack_from_gptq(as_form(q), s, None, -1, "cuda:0") is None
