"""The extension that calls the library without ctypes (`kiln_amd/lib/_torch_calls.so`, built from
csrc/torch/torch_calls.cpp): `linear`, `linear_lora`, `linear_sides`, `mlp`, `quantize`, `repack`.  Each takes the plain case -- contiguous CUDA
tensors of the right types, a workspace that is already there -- and returns None for anything else, upon
which the wrappers here take their checked route (same kernels, the reference's error texts).

Like the library itself it must be built: a missing file is an error, not a slower path.
"""
from __future__ import annotations

import ctypes
import importlib.util

import torch  # noqa: F401  (the extension links against its libraries)

from . import _lib

EXTENSION_PATH = _lib.LIB_PATH.with_name("_torch_calls.so")

# in the order bind() takes them
_FUNCTIONS = ("kiln_marlin_w4a16_gemm", "kiln_w4a16_gemm_lora", "kiln_w4a16_gemm_swiglu", "kiln_w4a16_gemm_swiglu_lora",
              "kiln_w4a16_mlp", "kiln_w4a16_workspace_bytes", "kiln_w4a16_mlp_workspace_bytes", "kiln_w4a16_stack_adapters",
              "kiln_w4a16_quantize_and_pack_many_device", "kiln_w4a16_takes_adapter_sides", "kiln_w4a16_gemm_adapter_sides",
              "kiln_w4a16_repack_gptq_device", "kiln_w4a16_takes_rank")


_ext = None
_adapter_types: tuple = ()
_workspaces: dict | None = None


def set_adapter_types(stacked: type, single: type) -> None:
    """The classes `linear_sides` takes adapters as (lora.StackedLora, lora.LoraProjectionWeights)."""
    global _adapter_types
    _adapter_types = (stacked, single)
    if _ext is not None:
        _ext.set_adapter_types(*_adapter_types)


def set_workspaces(workspaces: dict) -> None:
    """The dictionary `{(device index, stream handle): uint8 tensor}` the calls look their workspace up in."""
    global _workspaces
    _workspaces = workspaces
    if _ext is not None:
        _ext.set_workspaces(_workspaces)


def _bind(ext):
    return lambda L: ext.bind(*(ctypes.cast(getattr(L, name), ctypes.c_void_p).value for name in _FUNCTIONS))


def _import() -> None:
    """Load the extension and put its functions in the place of the stand-ins below."""
    global _ext
    if not EXTENSION_PATH.exists():
        raise _lib.LibraryMissing(
            f"kiln-marlin-gemm: {EXTENSION_PATH} is not built; run `python -m kiln_amd.build` (needs hipcc).")
    spec = importlib.util.spec_from_file_location("kiln_amd._torch_calls", EXTENSION_PATH)
    ext = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(ext)
    _ext = ext
    if _adapter_types:
        ext.set_adapter_types(*_adapter_types)
    if _workspaces is not None:
        ext.set_workspaces(_workspaces)
    _lib.on_active_library(_bind(ext))
    _lib.load()
    for name in _NAMES:
        globals()[name] = getattr(ext, name)


def _stand_in(name: str):
    # the first call loads the extension (not the import of this package: the build imports it too)
    def first_call(*args):
        _import()
        return globals()[name](*args)
    return first_call


_NAMES = ("linear", "linear_lora", "linear_sides", "mlp", "quantize", "repack")
linear, linear_lora, linear_sides, mlp, quantize, repack = map(_stand_in, _NAMES)
