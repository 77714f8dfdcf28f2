"""Prompt packing and dense re-expansion at the edges of their 16-byte pieces: widths that are no
whole number of pieces, counts that end a row's buffer inside a piece, counts past 16 pieces, zero
counts, appends behind a prompt -- buffers, tables, pointers and expansion bit-exact."""
import numpy as np
import pytest
import torch

from dynakv_amd import _lib
from dynakv_amd.kernels.compressed_cache import CustomDynamicCache
from oracle.packing import PackedSlot

from test_gpu_cache import _cmp_slot, _rounded

# (rows, tokens, width, dtype)
CASES = [
    (1, 2, 1, torch.bfloat16),
    (3, 65, 7, torch.float16),
    (2, 33, 60, torch.bfloat16),
    (5, 64, 128, torch.bfloat16),
    (2, 130, 129, torch.float16),
    (3, 17, 300, torch.float32),
    (2, 40, 1024, torch.bfloat16),
]


@pytest.mark.gpu
@pytest.mark.parametrize("i", range(len(CASES)))
def test_pack_and_expand(dev, i):
    B, S, W, dtype = CASES[i]
    print(f"[gpu] pack edges {CASES[i]}", flush=True)
    rng = np.random.default_rng(1200 + i)
    cache, rk, rv = CustomDynamicCache(), PackedSlot(), PackedSlot()
    for part in (S, S + 3):
        x = [_rounded(rng.standard_normal((B, part, W)).astype(np.float32), dtype) for _ in range(2)]
        n = [rng.integers(0, W + 1, (B, part)).astype(np.int32) for _ in range(2)]
        n[0][:, -1], n[1][:, 0] = W, W  # a whole last token, a whole first one
        cache.update_sp(x[0].to(dev), torch.from_numpy(n[0]).to(dev), x[1].to(dev),
                        torch.from_numpy(n[1]).to(dev), W, 0, W)
        rk.append_prefill(x[0].float().numpy(), n[0], W)
        rv.append_prefill(x[1].float().numpy(), n[1], W)
        _cmp_slot(cache.key_cache_sp[0], rk, "K")
        _cmp_slot(cache.value_cache_sp[0], rv, "V")
        for got, ref in zip(cache.get_origin_states(W, 0), (rk, rv)):
            np.testing.assert_array_equal(got.float().cpu().numpy(),
                                          ref.decompress(W).astype(np.float32))


# (rows, tokens, width, dtype, state order): new slots of rows with very different totals
NEW = [
    (1, 2, 8, torch.bfloat16, "rows"),
    (3, 65, 7, torch.float16, "rows"),
    (4, 300, 128, torch.bfloat16, "tokens"),
    (2, 33, 60, torch.float32, "dims"),
    (9, 1030, 33, torch.bfloat16, "rows"),
]


@pytest.mark.gpu
@pytest.mark.parametrize("i", range(len(NEW)))
def test_new_slots_written_whole(dev, i):
    """A prompt onto slots that do not exist, in memory that held other values: the zeros past
    each row's last coefficient (rows without any among them) and the pointers are written."""
    B, S, W, dtype, order = NEW[i]
    print(f"[gpu] new slots {NEW[i]}", flush=True)
    rng = np.random.default_rng(1300 + i)
    perm = {"rows": (0, 1, 2), "tokens": (1, 0, 2), "dims": (0, 2, 1)}[order]  # memory order
    x = [_rounded(rng.standard_normal((B, S, W)).astype(np.float32), dtype) for _ in range(2)]
    n = [rng.integers(0, W + 1, (B, S)).astype(np.int32) for _ in range(2)]
    for k, t in enumerate(n):
        t[:, S // (2 + k):] //= np.arange(1, B + 1)[:, None] ** 2
        if B > 2:
            t[B - 2 + k] = 0
    n[0][0, 0], n[1][0, 1] = W, W
    inv = np.argsort(perm).tolist()
    g = [t.permute(perm).contiguous().to(dev).permute(inv) for t in x]
    dirty = [torch.full((m,), -1, dtype=torch.int16, device=dev)
             for m in (64, 256, 512, 2 * B * S * W, 4 * B * S * W)]
    del dirty
    cache, rk, rv = CustomDynamicCache(), PackedSlot(), PackedSlot()
    cache.update_sp(g[0], torch.from_numpy(n[0]).to(dev), g[1], torch.from_numpy(n[1]).to(dev),
                    W, 0, W)
    rk.append_prefill(x[0].float().numpy(), n[0], W)
    rv.append_prefill(x[1].float().numpy(), n[1], W)
    for slot, ref, what in ((cache.key_cache_sp[0], rk, "K"), (cache.value_cache_sp[0], rv, "V")):
        _cmp_slot(slot, ref, what)
        for b, end in enumerate(slot[3].tolist()):
            assert end == slot[5][b]
            assert not slot[0][b, end:].any()


@pytest.mark.gpu
def test_row_totals(dev):
    """Sums of raw and clipped counts, negative and oversized ones among them, strided tables."""
    print("[gpu] row totals", flush=True)
    rng = np.random.default_rng(5)
    for rows, n, md in ((1, 1, 8), (7, 257, 128), (3, 1000, 1024)):
        k, v = (torch.from_numpy(rng.integers(-3, md + 9, (n, rows)).astype(np.int32)).to(dev).t()
                for _ in range(2))
        out = torch.full((2, 2, rows), -1, dtype=torch.int64, device=dev)
        rc = _lib.calls().dkv_row_totals(_lib.stream_of(k), k.data_ptr(), k.stride(0), k.stride(1),
                                         v.data_ptr(), v.stride(0), v.stride(1), rows, n, md,
                                         out.data_ptr())
        assert rc == _lib.DKV_OK
        for s, t in enumerate((k, v)):
            assert torch.equal(out[0, s], t.sum(1))
            assert torch.equal(out[1, s], t.clamp(0, md).sum(1))
