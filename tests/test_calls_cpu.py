"""The native call module fills the C ABI's structures as the ctypes classes would: its entry
points are bound to Python callbacks, so every field that would reach the library is seen."""

import ctypes as C

import numpy as np
import pytest
import torch

from animaxs_amd import QKPrologue, QuantizedLinearWeightBuffers, _abi
from animaxs_amd import executors as E

ATT = C.CFUNCTYPE(C.c_int, C.c_void_p, C.POINTER(_abi.AttentionArgs))
LIN = C.CFUNCTYPE(C.c_int, C.c_void_p, _abi.Buffer, C.c_int64, C.POINTER(_abi.QWeight), _abi.Buffer, C.c_int64,
                  C.c_int64, C.c_int32)
MV = C.CFUNCTYPE(C.c_int, C.c_void_p, C.POINTER(_abi.QWeight), _abi.Buffer, C.c_int64, _abi.Buffer, C.c_int64)


def fields(s):
    return {n: fields(getattr(s, n)) if isinstance(getattr(s, n), C.Structure) else getattr(s, n)
            for n, _ in s._fields_ if not isinstance(getattr(s, n), C._Pointer)}


class Seen:
    def __init__(self):
        self.calls = []
        self.status = 0
        self.keep = [ATT(self.att(i)) for i in range(3)] + [LIN(self.lin(i)) for i in range(2)] + [MV(self.mv)]

    def att(self, which):
        def f(h, a):
            a = a.contents
            pro = fields(a.prologue.contents) if a.prologue else None
            L = [C.cast(a.key_lengths, C.POINTER(C.c_int32))[i] for i in range(a.batch)] \
                if a.key_lengths and not a.key_lengths_on_device else a.key_lengths
            self.calls.append(("att", which, h, fields(a), pro, L))
            return self.status
        return f

    def lin(self, which):
        def f(h, x, xo, w, y, yo, rows, family):
            self.calls.append(("lin", which, h, fields(x), xo, fields(w.contents), fields(y), yo, rows, family))
            return self.status
        return f

    def mv(self, h, w, x, xo, y, yo):
        self.calls.append(("mv", h, fields(w.contents), fields(x), xo, fields(y), yo))
        return self.status


@pytest.fixture
def seen():
    s = Seen()
    lib = _abi.load()
    _abi.calls.bind(tuple(C.cast(f, C.c_void_p).value for f in s.keep), E.as_buffer, QuantizedLinearWeightBuffers,
                    QKPrologue, E.lengths_address)
    yield s
    _abi._bind_calls(lib)


class Executor:
    _h = C.c_void_p(4096)
    _layout = staticmethod(E.AttentionExecutor._layout)
    _call = E.AttentionExecutor._call
    encode, encode_noalloc, execute = (E.AttentionExecutor.encode, E.AttentionExecutor.encode_noalloc,
                                       E.AttentionExecutor.execute)


ATT_ARGS = dict(query=(256, 64), key=_abi.Buffer(512, 128), value=(768, 32), output=(1024, 16), heads=2, query_count=3,
                key_count=np.int64(5), head_dim=64)


def test_attention_defaults_and_every_argument(seen):
    ex = Executor()
    ex.encode(**ATT_ARGS)
    kind, which, h, a, pro, L = seen.calls[-1]
    assert (which, h, pro, L) == (0, 4096, None, None)
    assert a["query"] == {"ptr": 256, "length": 64} and a["key"] == {"ptr": 512, "length": 128}
    assert (a["heads"], a["query_count"], a["key_count"], a["head_dim"]) == (2, 3, 5, 64)
    assert (a["key_value_heads"], a["causal"], a["layout"], a["token_stride"], a["batch"]) == (0, 0, -1, 0, 1)
    assert (a["scale"], a["kv_token_stride"], a["key_lengths_on_device"]) == (0.0, 0, 0)
    p = QKPrologue((2, 4), None, 1e-5, (8, 16), 7, True, False, (32, 64), 9)
    ex.encode_noalloc(**ATT_ARGS, query_offset=1, key_offset=2, value_offset=3, output_offset=4, key_value_heads=1,
                      causal=True, layout=("tokenMajor", 128), batch=2, key_lengths=[3, 4], scale=0.5, prologue=p,
                      kv_token_stride=64)
    kind, which, h, a, pro, L = seen.calls[-1]
    assert which == 1 and L == [3, 4] and pro == fields(p.to_c())
    assert [a[n + "_offset"] for n in ("query", "key", "value", "output")] == [1, 2, 3, 4]
    assert (a["key_value_heads"], a["causal"], a["layout"], a["token_stride"], a["batch"], a["scale"],
            a["kv_token_stride"]) == (1, 1, 1, 128, 2, 0.5, 64)
    ex.execute(**ATT_ARGS, key_lengths=4096, key_lengths_on_device=True, key_value_heads=None, layout=None, prologue=None,
               **{"".join(["ba", "tch"]): 4})
    kind, which, h, a, pro, L = seen.calls[-1]
    assert which == 2 and a["key_lengths"] == 4096 and a["key_lengths_on_device"] == 1 and a["batch"] == 4


def test_attention_refusals(seen):
    ex = Executor()
    with pytest.raises(TypeError, match="unexpected"):
        ex.encode(**ATT_ARGS, rows=3)
    with pytest.raises(TypeError, match="head_dim"):
        ex.encode(**{k: v for k, v in ATT_ARGS.items() if k != "head_dim"})
    with pytest.raises(TypeError, match="host tensor"):
        ex.encode(**{**ATT_ARGS, "query": torch.zeros(4)})
    with pytest.raises(TypeError):
        ex.encode(**{**ATT_ARGS, "query": "text"})
    with pytest.raises(ValueError):
        ex.encode(**ATT_ARGS, layout="rows")
    assert not seen.calls
    seen.status = _abi.E_INVALID_SHAPE
    with pytest.raises(_abi.AnimaError) as e:
        ex.encode(**ATT_ARGS)
    assert e.value.status == _abi.E_INVALID_SHAPE


def test_linear_and_matvec(seen):
    w = QuantizedLinearWeightBuffers(1, (16, 32), (48, 64), None, 3, 4, 5, 6, 7, 8)

    class Other(QuantizedLinearWeightBuffers):   # goes through its own to_c
        pass

    lin = E.LinearExecutor.__new__(E.LinearExecutor)
    lin._h = C.c_void_p(8192)
    try:
        for weight in (w, Other(**vars(w))):
            lin.encode((80, 96), weight, (112, 128), 9, input_offset=10, output_offset=12, family="mlpUp")
            assert seen.calls[-1] == ("lin", 0, 8192, {"ptr": 80, "length": 96}, 10, fields(w.to_c()),
                                      {"ptr": 112, "length": 128}, 12, 9, _abi.FAMILY_MLP_UP)
        lin.execute((80, 96), w, (112, 128), 9)
        assert seen.calls[-1][:3] == ("lin", 1, 8192)
    finally:
        lin._h = C.c_void_p()

    class Ctx:
        handle = C.c_void_p(64)
    E.LinearExecutor.encode_matvec(Ctx, w, (80, 96), (112, 128), 4, 8)
    assert seen.calls[-1] == ("mv", 64, fields(w.to_c()), {"ptr": 80, "length": 96}, 4, {"ptr": 112, "length": 128}, 8)


def test_the_module_carries_this_interpreters_tag():
    """An untagged module would load under any interpreter, whatever ABI it was compiled for."""
    import sysconfig
    from animaxs_amd import _calls, build
    assert _calls.__file__.endswith(sysconfig.get_config_var("EXT_SUFFIX"))
    assert not (build.PKG / "_calls.so").exists()
