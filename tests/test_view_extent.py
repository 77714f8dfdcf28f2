"""``_lib.view_extent`` (evaluated in Python) against the library's ``dkv_view_extent_elems``."""
import ctypes
import itertools

import torch

from dynakv_amd import _lib


def _library(t):
    n = max(t.dim(), 1)
    arr = ctypes.c_longlong * n
    return _lib.load().dkv_view_extent_elems(t.dim(), arr(*t.shape), arr(*t.stride()))


def test_view_extent_is_the_librarys():
    base = torch.zeros(4, 6, 10, 16)
    views = [base, base[1:, ::2], base[:, :, 3:7], base[2, 1, 4], base[0, 0, 0, 0],
             torch.zeros(0, 4, 128), torch.zeros(3, 0), base[:, :1].expand(4, 5, 10, 16)]
    views += [base.permute(p) for p in itertools.permutations(range(4))]
    views += [base.as_strided((2, 3), (a, b)) for a in (0, 1, 7) for b in (0, 1, 5)]
    for t in views:
        assert _lib.view_extent(t) == _library(t), (t.shape, t.stride())
