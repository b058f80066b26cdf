"""The library's calls from Python (gaac_amd/_binding.so): conversion of arguments and errors, without a GPU."""
import pytest
import torch

from gaac_amd import _lib


def test_every_entry_point_is_there_and_counts_its_arguments():
    calls = _lib.calls()
    for name, args in _lib._SIGNATURES.items():
        with pytest.raises(TypeError, match=f"{name} takes {len(args)} arguments"): getattr(calls, name)(*[0] * (len(args) + 1))


def test_messages_of_the_library_are_raised():
    """Null pointers and zeros are refused ahead of any HIP call: the message that the entry point left arrives."""
    for name, args in _lib._SIGNATURES.items():
        if name in ("gaac_static_init", "gaac_static_reset"): continue      # these go to the device
        zeros = [None if a is _lib.P else 0.0 if a is _lib.c_float else 0 for a in args]
        with pytest.raises(RuntimeError, match=name + r" failed \(-1\): .{8}"): _lib.call(name, *zeros)


def test_arguments_that_are_refused():
    x, calls, seen = torch.zeros(16, 2, 128, dtype=torch.bfloat16), _lib.calls(), []
    def stream():
        seen.append(1)
        return 0
    with pytest.raises(RuntimeError, match="no CPU path"): calls.gaac_exponent_hist(x, 16, 2, None, stream)
    assert not seen      # the stream is asked for when the arguments before it are known to be usable
    with pytest.raises(RuntimeError, match="bad arguments"): calls.gaac_exponent_hist(None, 16, 2, None, stream)
    assert seen
    for bad in ("x", 1.5, [0]):
        with pytest.raises(TypeError): calls.gaac_exponent_hist(bad, 16, 2, None, None)
        with pytest.raises(TypeError): calls.gaac_exponent_hist(None, bad, 2, None, None)
    with pytest.raises(TypeError, match="function that returns an address"): calls.gaac_exponent_hist(None, 16, 2, None, lambda: None)
    with pytest.raises(ZeroDivisionError): calls.gaac_exponent_hist(None, 16, 2, None, lambda: 1 // 0)
    with pytest.raises(AttributeError, match="undefined symbol"): calls.bind("libc.so.6")
    calls.bind(_lib.lib_path())
