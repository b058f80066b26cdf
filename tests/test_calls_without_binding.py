"""The library's calls where gaac_amd/_binding.so is missing or was built for another torch: through ctypes, with the same errors."""
import sys

import pytest
import torch

from gaac_amd import _lib


@pytest.fixture(params=["missing", "built for another torch"])
def calls(request, monkeypatch):
    _lib.calls()
    from gaac_amd import _binding
    monkeypatch.setattr(_lib, "_calls", None)
    if request.param == "missing":
        monkeypatch.setitem(sys.modules, "gaac_amd._binding", None)
        monkeypatch.delattr("gaac_amd._binding")
    else: monkeypatch.setattr(_binding, "torch_version", "1.0")
    with pytest.warns(RuntimeWarning, match="calls go through ctypes"): calls = _lib.calls()
    assert calls is not _binding and _lib.calls() is calls
    return calls


def test_the_binding_is_for_this_torch():
    from gaac_amd import _binding
    assert _lib.calls() is _binding and _binding.torch_version == torch.__version__


def test_errors(calls):
    for name, args in _lib._SIGNATURES.items():
        with pytest.raises(TypeError, match=f"{name} takes {len(args)} arguments"): getattr(calls, name)(*[0] * (len(args) + 1))
        if name in ("gaac_static_init", "gaac_static_reset"): continue      # these go to the device
        zeros = [None if a is _lib.P else 0.0 if a is _lib.c_float else 0 for a in args]
        with pytest.raises(RuntimeError, match=name + r" failed \(-1\): .{8}"): _lib.call(name, *zeros)
    seen = []
    with pytest.raises(RuntimeError, match="no CPU path"): calls.gaac_exponent_hist(torch.zeros(16, 2, 128), 16, 2, None, lambda: seen.append(1))
    assert not seen      # the stream is asked for when the arguments before it are known to be usable
    with pytest.raises(TypeError): calls.gaac_exponent_hist(None, 1.5, 2, None, None)


@pytest.mark.gpu
def test_a_page(calls):
    from gpu_util import require_gpu
    dev = require_gpu()
    from gaac_amd import Codec, TileEncoder, attention
    gen = torch.Generator(device=dev).manual_seed(1)
    x = torch.randn(2, 333, 128, generator=gen, device=dev).to(torch.bfloat16)
    q = torch.randn(1, 8, 128, generator=gen, device=dev).to(torch.bfloat16)
    codec = Codec(2).calibrate(x)
    k, v = (TileEncoder(kind).encode(codec, x) for kind in "kv")
    assert torch.equal(Codec.decode(k), x) and torch.equal(Codec.decode(v), x)
    want = torch.nn.functional.scaled_dot_product_attention(q.float().view(2, 4, 128), x.float(), x.float()).view(1, 8, 128)
    assert (attention(q, k, v).float() - want).norm() < 8e-3 * want.norm()      # weights and output rounded to bf16, 2^-9 each
