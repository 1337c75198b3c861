"""The argument blocks' packer against field-by-field ctypes stores (CPU)."""
import ctypes

import pytest

from cuda_llm_ops_amd import _lib


@pytest.mark.parametrize("cls", [_lib.DecodeArgs, _lib.PagedDecodeArgs, _lib.PrefillArgs, _lib.BackwardArgs,
                                 _lib.SparsePrefillArgs])
@pytest.mark.parametrize("wide", [False, True])
def test_packed_block_equals_stores(cls, wide):
    """`wide`: values their C types cannot hold (stored as ctypes stores them)."""
    ref, values, n = cls(), [], 1
    for name, t in cls._fields_:
        if hasattr(t, "_length_"):
            v = [n + i + (1 << 40) for i in range(t._length_)]
            getattr(ref, name)[:] = v
            values += v
        else:
            v = 0.25 * n if t is ctypes.c_float else n
            if wide and t is ctypes.c_int32:
                v += 1 << 33
            if wide and t is ctypes.c_float:
                v = 1e300
            setattr(ref, name, v)
            values.append(v)
        n += 7
    got = _lib.ArgsPacker(cls)(*values)
    for name, t in cls._fields_:
        a, b = getattr(got, name), getattr(ref, name)
        assert (list(a) == list(b)) if hasattr(t, "_length_") else (a == b), name
