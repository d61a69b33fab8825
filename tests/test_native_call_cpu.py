"""Calls of the kernel library's functions through the extension module: the same values arrive as through ctypes (no GPU: functions
that answer from sizes, and argument checks that come ahead of a launch)."""
import ctypes
import gc
import threading
import time
import weakref

import numpy as np
import pytest

from vllm_distributed_amd.ops import native as N

pytestmark = pytest.mark.skipif(not N.is_available(), reason="libvda_ops.so is not built")


def test_values_are_those_of_ctypes():
    for args in ((1, 10, 32, 8, 128, 4000), (7, 2000, 28, 4, 128, 1 << 33)):
        assert N.value("vda_prefill_parts", *args) == N.lib().vda_prefill_parts(*args)
    for scale in (0.3, 0, 1, -1.0):                      # a float among integers; whole numbers in its place
        args = (43, 43, 128, 576, 16, 300, 1, scale, 4)
        assert N.value("vda_mla_splits", *args) == N.lib().vda_mla_splits(*args)


def _decode(**change):
    names = ("out q k v table lens starts alibi part lse S T Hq Hkv D block cols nsplit maxq qs os scale softcap window dtype fp8 ks vs "
             "sink chunk v_shift bias far").split()
    ok = dict(zip(names, [None] * 10 + [1, 1, 32, 8, 128, 16, 4, 1, 1, 4096, 4096, 0.1, 0.0, 0, 0, 0, 1.0, 1.0, None, 0, 0, None, 0]))
    n = len(N._SIGS["vda_paged_attention_decode"])
    return list(dict(ok, **change).values()) + [0] * (n - len(ok))


# the codes of checks on arguments that go into registers, onto the stack, and lie behind four floats
@pytest.mark.parametrize("change,code", [(dict(Hkv=5), -1), (dict(nsplit=0), -6), (dict(chunk=-1), -7), (dict(v_shift=4), -7),
                                         (dict(maxq=9), -4), (dict(bias=64, far=-1), -7)])
def test_a_status_names_the_function(change, code):
    args = _decode(**change)
    assert N.lib().vda_paged_attention_decode(*args) == code
    assert N.value("vda_paged_attention_decode", *args) == code
    with pytest.raises(RuntimeError, match=f"vda_paged_attention_decode failed with code {code}"):
        N.call("vda_paged_attention_decode", *args)


def test_other_kinds_of_arguments_go_through_ctypes():
    assert N.value("vda_scan_lane_channel", ctypes.c_int(30), 32, True) == N.lib().vda_scan_lane_channel(30, 32, 1)
    for bad in ("8", 2.5, np.float32(2)):
        with pytest.raises(ctypes.ArgumentError):
            N.value("vda_scan_lane_channel", bad, 32, 1)
    with pytest.raises(TypeError):
        N.value("vda_scan_lane_channel", 30)


def test_a_function_that_is_not_there():
    N.lib()
    with pytest.raises(RuntimeError, match="has no kernel vda_nothing"):
        N.call("vda_nothing", 1)


@pytest.mark.parametrize("argument", [7, ctypes.c_int(7)])          # straight from the object; through ctypes
def test_a_name_is_bound_again_while_its_function_runs(argument):
    """What a call uses lives until it has answered."""
    from vllm_distributed_amd.ops import _vda_call
    alive = []

    def body(x):
        _vda_call.bind("vda_test_again", target, "I", other)
        gc.collect()
        alive.append(bound() is not None)
        return x + 1

    kind = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_int)
    code = kind(body)                                              # (holds the code that is called; what is bound holds none)
    target = ctypes.cast(code, ctypes.c_void_p).value
    other, function = kind(target), kind(target)
    bound = weakref.ref(function)
    _vda_call.bind("vda_test_again", target, "I", function)
    del function
    assert _vda_call.value("vda_test_again", argument) == 8
    gc.collect()
    assert alive == [True] and bound() is None


def test_the_library_is_loaded_once(monkeypatch):
    """Threads whose first calls come together wait for one of them to load it and to bind its functions."""
    N.lib()
    loads, real, started = [], ctypes.CDLL, threading.Barrier(3)

    def load(path):
        loads.append(path)
        time.sleep(0.2)
        return real(path)

    monkeypatch.setattr(N.ctypes, "CDLL", load)
    monkeypatch.setattr(N, "_LIB", None)
    got = []

    def first():
        started.wait()
        got.append(N.lib())

    threads = [threading.Thread(target=first) for _ in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(loads) == 1 and len(got) == 3 and all(x is got[0] for x in got)
