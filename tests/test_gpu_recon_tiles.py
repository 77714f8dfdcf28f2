"""dkv_recon_kv with several 64-token tiles per workgroup (more than 512 tiles in all), at ragged
ends and position offsets, with the bounds of the single-tile cases against float64."""
import pytest
import torch

import test_gpu_recon as base

# (B, G, S, R, dtype, pos0, strided rows); tiles per workgroup 2, 2, 3, 5
TILED = [
    (16, 8, 257, 128, torch.bfloat16, 0, False),
    (1, 8, 2081, 128, torch.float16, 0, True),
    (24, 8, 193, 72, torch.float16, 21, False),
    (32, 8, 256, 128, torch.bfloat16, 5, False),
]


@pytest.mark.gpu
@pytest.mark.parametrize("i", range(len(TILED)))
def test_tiled_recon_matches_float64(dev, i, monkeypatch):
    monkeypatch.setitem(base.CASES, f"tiled_{i}", TILED[i])
    base.test_recon_kv_matches_float64(dev, f"tiled_{i}")


@pytest.mark.gpu
def test_unaligned_outputs(dev):
    """Output rows on 8-byte boundaries (8-byte stores) hold what 16-byte aligned ones do."""
    print("[gpu] recon_kv unaligned outputs", flush=True)
    from dynakv_amd import _lib
    from dynakv_amd.kernels.decode import rope_table
    G, S, R, dt = 2, 77, 128, torch.bfloat16
    ck, cv, kb, vb = (torch.from_numpy(a).to(device=dev, dtype=dt)
                      for a in base._inputs(1, G, S, R, dt, seed=3))
    k, v = base.recon_kv(ck, cv, kb, vb, batch=1, theta=base.THETA)
    ld = 132
    out = torch.zeros(2, G * S * ld + 4, dtype=dt, device=dev)
    st = _lib.stream_of(ck)
    rope, tiles = rope_table(dev, st, base.THETA, S)
    rc = _lib.load().dkv_recon_kv(
        st, _lib.dtype_code(dt), ck.data_ptr(), cv.data_ptr(), S * R, R, kb.data_ptr(),
        vb.data_ptr(), R * 128, 128, out[0, 4:].data_ptr(), out[1, 4:].data_ptr(), S * ld, ld, G, G,
        S, R, 0, rope.data_ptr(), tiles)
    assert rc == _lib.DKV_OK
    torch.cuda.synchronize()
    for got, want in ((out[0], k), (out[1], v)):
        rows = got[4:].view(G, S, ld)
        assert torch.equal(rows[..., :128], want.view(G, S, 128))
        assert not rows[..., 128:].any()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("R", [8, 40, 64, 128])
@pytest.mark.parametrize("transposed", [False, True])
def test_one_tile_equals_several(dev, R, dtype, transposed):
    """A call of several tiles per workgroup, and the same tokens in calls of up to 512 workgroups
    (one tile each, another kernel for rank-major bases): the same bits."""
    B, G, S = 16, 8, 257  # 16 x 8 rows x 5 tiles x K, V: 1280 workgroups of one tile
    print(f"[gpu] recon one tile against several R={R} {dtype} transposed={transposed}", flush=True)
    ck, cv, kb, vb = (torch.from_numpy(a).to(device=dev, dtype=dtype)
                      for a in base._inputs(B, G, S, R, dtype, seed=40 + R))
    if transposed:
        kb, vb = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (kb, vb))
    k, v = base.recon_kv(ck, cv, kb, vb, batch=B, theta=base.THETA)
    for b in range(0, B, 3):
        rows = slice(b * G, (b + 1) * G)
        for t0, t1 in ((0, 64), (64, 200), (192, 257)):
            kk, vv = base.recon_kv(ck[rows, t0:t1], cv[rows, t0:t1], kb, vb, batch=1,
                                   theta=base.THETA, pos0=t0)
            assert torch.equal(kk[0], k[b, :, t0:t1]) and torch.equal(vv[0], v[b, :, t0:t1])
