"""Without the call module (no C headers at build time, another interpreter, the library alone) the
wrappers run on the ctypes binding: the same functions, the same results."""
import shutil
import sysconfig

import pytest
import torch

from dynakv_amd import _lib, build
from dynakv_amd.kernels.compressed_cache import CustomDynamicCache
from dynakv_amd.kernels.cutoff import CutoffHead
from dynakv_amd.kernels.decode import grouped_decode_attention
from dynakv_amd.kernels.layer import DecodeLayerPlan


def test_library_alone(tmp_path, monkeypatch):
    shutil.copy(_lib.LIB_PATH, tmp_path)
    monkeypatch.setattr(_lib, "LIB_PATH", tmp_path / _lib.LIB_PATH.name)
    monkeypatch.setattr(_lib, "_calls", None)
    assert _lib.calls() is _lib.load()
    assert _lib.calls().dkv_splitk_workspace_floats(1, 32, 8, 96, 128, 0) > 0


def test_module_is_named_for_its_interpreter():
    assert build.CALL_PATH.name == _lib.CALL_NAME
    assert _lib.CALL_NAME.endswith(sysconfig.get_config_var("EXT_SUFFIX"))
    assert _lib.calls() is not _lib.load()  # built here


def test_build_without_headers(tmp_path, monkeypatch):
    """The module is left out, an earlier one with it; nothing raises."""
    stale = tmp_path / _lib.CALL_NAME
    stale.write_bytes(b"")
    monkeypatch.setattr(build, "CALL_PATH", stale)
    monkeypatch.setattr(build.sysconfig, "get_paths", lambda: {"include": str(tmp_path)})
    build._build_binding(verbose=False)
    assert not stale.exists()


@pytest.mark.gpu
def test_same_results(dev, monkeypatch):
    """A prompt, a decode append, attention and a layer step on either binding."""
    print("[gpu] ctypes binding", flush=True)
    B, G, Hq, S, D = 2, 2, 8, 90, 128
    g = torch.Generator().manual_seed(3)
    r = lambda *d: torch.randn(*d, generator=g).to(dev, torch.bfloat16)  # noqa: E731
    w, b, basis = r(G, D, D) * 0.05, r(G, D), r(G, D, 128) * 0.1
    x, q, c = r(B * G, S, D), r(B, Hq, 128), r(B, G * D)
    ln = torch.randint(1, D + 1, (B * G, S), generator=g, dtype=torch.int32).to(dev)

    def run():
        cache = CustomDynamicCache()
        cache.update_sp(x, ln, x, ln, D, 0, D)
        one = ln[:, :1].contiguous()
        fk, fv, lk, lv, ok, ov = cache.update_sp(x[:, :1], one, x[:, :1], one, D, 0, D)
        out = [grouped_decode_attention(q.clone(), fk, fv, lk, ok, lv, ov, basis, basis, theta=1e4,
                                        route=_lib.DKV_ROUTE_FUSED)]
        head = CutoffHead(w, b, w, b, groups=G)
        out += head.kv_process_fused(c.view(B, 1, -1), c.view(B, 1, -1))[:4]
        plan = DecodeLayerPlan(cache, 0, head, basis, basis, batch=B, heads=Hq, theta=1e4)
        out.append(plan.step(q.clone(), c, c, S + 1))
        return out + list(cache.get_origin_states(D, 0))

    fast = run()
    monkeypatch.setattr(_lib, "_calls", _lib.load())
    for a, e in zip(run(), fast):
        assert torch.equal(a, e)
