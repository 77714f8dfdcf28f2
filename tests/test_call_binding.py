"""The CPython binding of the per-call entry points: the same C functions as the ctypes binding,
argument counts and ranges checked, every status returned."""
import inspect

import pytest

from dynakv_amd import _lib
from dynakv_amd.kernels import (compressed_cache, cutoff, decode, fused, joint, layer, model_ops,
                                prefill, two_stage)


def test_same_functions_as_ctypes():
    lib, calls = _lib.load(), _lib.calls()
    for B, S in ((1, 1), (3, 777), (16, 8192)):
        assert (calls.dkv_splitk_workspace_floats(B, 32, 8, S, 128, 0)
                == lib.dkv_splitk_workspace_floats(B, 32, 8, S, 128, 0))
        assert (calls.dkv_joint_av_workspace_floats(B, 32, S, 1024)
                == lib.dkv_joint_av_workspace_floats(B, 32, S, 1024))
    # a status comes back as it is (checked before any device work), NULL as None
    assert calls.dkv_add_rmsnorm(None, 99, None, 0, None, 0, None, None, 0, 1, 8, 1e-5) \
        == _lib.DKV_E_UNSUPPORTED
    assert calls.dkv_gemv(None, _lib.DKV_BF16, None, 0, None, 0, None, 0, -1, 8, 8) == _lib.DKV_E_ARG
    assert calls.dkv_gemv(None, _lib.DKV_BF16, None, 0, None, 0, None, 0, 0, 8, 8) == _lib.DKV_OK


def test_arguments_are_checked():
    f = _lib.calls().dkv_splitk_workspace_floats
    with pytest.raises(TypeError):
        f(1, 2, 3)
    with pytest.raises(TypeError):
        f(1, 32, 8, 96.0, 128, 0)
    with pytest.raises(OverflowError):
        f(1, 32, 8, 1 << 40, 128, 0)
    with pytest.raises(TypeError):
        _lib.calls().dkv_add_rmsnorm("stream", 1, None, 0, None, 0, None, None, 0, 1, 8, 1e-5)


def test_every_wrapped_entry_point_is_bound():
    """Each ``lib.dkv_*`` the kernel wrappers call exists in the module and is declared."""
    import re
    names = set()
    for mod in (compressed_cache, cutoff, decode, fused, joint, layer, model_ops, prefill,
                two_stage):
        names |= set(re.findall(r"(?:lib|calls\(\))\.(dkv_\w+)", inspect.getsource(mod)))
    assert names
    for n in names:
        assert hasattr(_lib.calls(), n), n
        assert n in _lib.exported_symbols(), n
