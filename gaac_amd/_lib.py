"""gaac_amd/libgaac_hip.so (see include/gaac_hip.h): calls() has its entry points as functions that take tensors (gaac_amd/_binding.so), load()
is the library for ctypes.  There is no fallback: if one of the two is missing, or a call is made without a GPU, the call raises."""
from __future__ import annotations
import ctypes, os
import torch

_LIB_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "libgaac_hip.so")
_lib = None
_calls = None

c_int, c_long, c_float, c_void_p = ctypes.c_int, ctypes.c_long, ctypes.c_float, ctypes.c_void_p
P = c_void_p

_SIGNATURES = {
    "gaac_wait_words": [P, c_int, P],
    "gaac_exponent_hist": [P, c_long, c_int, P, P],
    "gaac_bases_from_hist": [P, c_int, P, P, P],
    "gaac_encode_tiles": [c_int, P, c_long, c_long, c_int, c_int, c_int, P, P, c_int, P, P, P, P, P, P, P],
    "gaac_compact": [P, P, P, P, P, c_int, c_int, P],
    "gaac_tile_scan": [P, c_int, c_int, P, P, P, P],
    "gaac_page_pack": [P, P, P, P, P, c_int, c_int, c_int, P, P, P, P],
    "gaac_page_finish": [P, P, P, c_int, c_int, c_int, P, P, P, P, P, c_long, P, P],
    "gaac_row_offsets": [P, c_int, c_int, c_int, P, P, P],
    "gaac_decode_tiles": [c_int, P, P, P, P, P, P, P, P, c_int, P, c_int, c_int, c_int, P, c_long, c_long, P],
    "gaac_cache_prefill": [P, P] + [c_long] * 4 + [c_int] * 7 + [P] * 27,
    "gaac_attn_split": [P] * 16 + [P, P, c_int, c_int, c_int, P, c_int, c_float, c_int, c_int, P, P, P, c_int, P, P, P, P],
    "gaac_attn_combine": [P, P, P, P, c_int, c_int, P],
    "gaac_cache_append": [P, c_int, c_int, P, P, P, P, c_int, c_int, c_int] + [P] * 18 + [P, P],
    "gaac_cache_check": [P, c_int, P, P, P, c_int, P, P],
    "gaac_paged_store": [P, P, c_long, c_long, P, c_int, P, c_int, P, P, P, P, P, P, P, P, P, P, c_int, P],
    "gaac_paged_free": [P, c_int, P, P, P],
    "gaac_paged_release": [P, c_int, P, P, P, c_int, P],
    "gaac_paged_decode": [P, c_int, P, P, P, c_int, P, P, c_long, P, P, P, P, c_int, P],
    "gaac_paged_attn": [P, c_int, P, P, P, c_int, P, c_int, P, c_int, c_int, c_int, c_float, c_int, P, P, P, P, c_int, P, P, P, P, P, P, c_int, P, P, P],
    "gaac_bf16_attn": [P, P, c_int, P, c_long, P, c_int, c_int, c_int, c_float, c_int, P, P, P, P, P, P],
    "gaac_attn_fused": [P] * 16 + [P, P, c_int, c_int, c_int, P, c_int, c_float, c_int, c_int, P, P, P, c_int, c_int, P, P, P, P, P, P],
    "gaac_attn_fused_static": [P] * 16 + [P, P, c_int, c_int, c_int, P, c_int, c_float, c_int, c_int, P, P, P, c_int, c_int, P, P],
    "gaac_static_init": [],
    "gaac_static_reset": [P],
    "gaac_static_flags": [P, P],
    "gaac_attn_launch": [P] * 16 + [P, P, c_int, c_int, c_int, P, c_int, c_float, c_int, c_int, P, P, P, c_int, P, P, P, P, P],
}


def lib_path() -> str:
    """The library file: gaac_amd/libgaac_hip.so, or the instrumented build named by GAAC_HIP_LIB (read when the library is loaded)."""
    return os.environ.get("GAAC_HIP_LIB") or _LIB_PATH


def load():
    """The loaded library (ctypes.CDLL).  Raises if it has not been built (python -m gaac_amd.build)."""
    global _lib
    if _lib is None:
        path = lib_path()
        if not os.path.exists(path):
            raise RuntimeError(f"{path} is missing: build it with `python -m gaac_amd.build` (hipcc, gfx950). "
                               "gaac_amd has no CPU or PyTorch fallback.")
        lib = ctypes.CDLL(path)
        lib.gaac_last_error.restype = ctypes.c_char_p
        lib.gaac_last_error.argtypes = []
        for name, args in _SIGNATURES.items():
            fn = getattr(lib, name)
            fn.restype = c_int
            fn.argtypes = args
        _lib = lib
    return _lib


def calls():
    """The entry points as functions, in the order of arguments of include/gaac_hip.h: tensors on the device, addresses or None for pointers,
    numbers, last the stream (its handle, or the function `stream`).  They raise RuntimeError with the library's message."""
    global _calls
    if _calls is None:
        load()
        try:
            from . import _binding
        except ImportError as e:
            raise RuntimeError(f"gaac_amd/_binding.so is missing or does not fit the installed torch ({e}): build it with `python -m gaac_amd.build`") from e
        _binding.bind(lib_path())
        _calls = _binding
    return _calls


def exported_symbols() -> list[str]:
    return ["gaac_last_error", *_SIGNATURES]


def ptr(t: torch.Tensor | None):
    if t is None:
        return None
    if not t.is_cuda:
        raise RuntimeError("gaac_amd kernels need device tensors (got a CPU tensor): there is no CPU path")
    return t.data_ptr()


def stream() -> int:
    """The current stream of the current device as a handle (torch.cuda.current_stream() builds a Stream object on the way: 3 us
    against 0.1, of the 5 us that a launch takes)."""
    return torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice())


def call(name: str, *args):
    getattr(_calls or calls(), name)(*args)
