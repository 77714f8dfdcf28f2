"""A prompt's K and V slots hold buffers of their own: no tensor of one shares its storage with the
other's, so one slot's growth frees the buffers it replaces."""
import pytest
import torch

from dynakv_amd.kernels.compressed_cache import CustomDynamicCache


def _storages(slot):
    return {t.untyped_storage().data_ptr() for t in slot[:4]}


@pytest.mark.gpu
@pytest.mark.parametrize("B,S,W", [(8, 300, 128), (2, 64, 1024)])
def test_slots_do_not_share_storage(dev, B, S, W):
    print(f"[gpu] slot storage {(B, S, W)}", flush=True)
    x = torch.randn(B, S, W, device=dev).to(torch.bfloat16)
    kl = torch.full((B, S), W, dtype=torch.int32, device=dev)
    vl = torch.full((B, S), W // 2, dtype=torch.int32, device=dev)
    cache = CustomDynamicCache()
    cache.update_sp(x, kl, x, vl, W, 0, W)
    ck, cv = cache.key_cache_sp[0], cache.value_cache_sp[0]
    assert not _storages(ck) & _storages(cv)
    for slot, kept in ((ck, W), (cv, W // 2)):
        assert slot[0].untyped_storage().nbytes() == B * S * kept * 2
    # decode tokens past the prompt's capacity: the flats are replaced, each by one of its own
    one = [t[:, :1].contiguous() for t in (kl, vl)]
    cache.update_sp(x[:, :1], one[0], x[:, :1], one[1], W, 0, W)
    assert not _storages(ck) & _storages(cv)
    for slot in (ck, cv):
        assert slot[0].untyped_storage().nbytes() == slot[0].numel() * 2
