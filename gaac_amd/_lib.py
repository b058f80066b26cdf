"""gaac_amd/libgaac_hip.so (see include/gaac_hip.h): calls() has its entry points as functions that take tensors (gaac_amd/_binding.so), load()
is the library for ctypes, which takes the calls where there is no binding for the installed torch.  There is no other fallback: if the library is
missing, or a call is made without a GPU, the call raises."""
from __future__ import annotations
import ctypes, os, warnings
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
    "gaac_prompt_store": [P, P] + [c_long] * 4 + [c_int] * 7 + [P] * 22 + [c_long] + [P] * 4 + [c_long, c_int, c_int, P, P],
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


class _CtypesCalls:
    """calls() through ctypes, for any torch: 14 us for an attention() where the binding takes 9.0, or 7.2 as a whole call (binding.cpp).  These are left to Python."""
    def attend(self, *args): return None
    token_append = prompt_store = page_encode = page_decode = attend
    def __getattr__(self, name):
        fn, n, error = getattr(load(), name), len(_SIGNATURES[name]), load().gaac_last_error
        def entry(*args):
            if len(args) != n: raise TypeError(f"{name} takes {n} arguments ({len(args)} given)")
            args = [ptr(a) if isinstance(a, torch.Tensor) else a() if callable(a) else a for a in args]
            try: rc = fn(*args)
            except ctypes.ArgumentError as e: raise TypeError(f"{name}: {e}") from None
            if rc != 0: raise RuntimeError(f"{name} failed ({rc}): {error().decode(errors='replace')}")
        setattr(self, name, entry)
        return entry


def calls():
    """The entry points as functions, in the order of arguments of include/gaac_hip.h: tensors on the device, addresses or None for pointers,
    numbers, last the stream (its handle, or the function `stream`).  They raise RuntimeError with the library's message.  The binding reads
    tensors by the layout of the torch that it was built with, and is left alone where another one is installed.  attend, token_append, prompt_store,
    page_encode and page_decode make a public call as a whole, or return None and leave it to Python."""
    global _calls
    if _calls is None:
        load()
        try:
            from . import _binding
            wrong = _binding.torch_version != torch.__version__ and f"is built for torch {_binding.torch_version}"
        except ImportError as e:
            wrong = f"cannot be loaded ({e})"
        if wrong:
            warnings.warn(f"gaac_amd/_binding.so {wrong}: calls go through ctypes and cost the host about twice the time; build it with `python -m gaac_amd.build`",
                          RuntimeWarning, stacklevel=2)
            _calls = _CtypesCalls()
        else:
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
