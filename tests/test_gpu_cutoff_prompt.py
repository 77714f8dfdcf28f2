"""The cutoff head at a prompt's row counts: the wave-per-tile kernel (D <= 128) and the tiled
logits kernels (D >= 256) at the edges of their tiles, against the oracle with the checks and
tolerances of the decode-size tests."""
import pytest
import torch

from dynakv_amd import _lib
from dynakv_amd.kernels import cutoff as CK

from test_gpu_cutoff import _check, _dev_rows, _inputs

# (G, D, M, dtype, low_rank, row padding): the smallest row counts of each kernel, one row past a
# 16-, 32- or 64-row tile, and a last tile of one row
CASES = [
    (8, 128, 321, torch.bfloat16, None, 0),
    (8, 128, 353, torch.float16, 37, 64),
    (4, 128, 656, torch.bfloat16, None, 0),
    (2, 64, 1281, torch.float16, None, 8),
    (1, 1024, 97, torch.bfloat16, None, 0),    # 32-row tiles
    (1, 1024, 129, torch.float16, 300, 64),
    (1, 1024, 641, torch.bfloat16, None, 0),   # 64-row tiles
    (2, 256, 385, torch.bfloat16, None, 8),
    (1, 512, 1345, torch.float16, None, 0),
    (2, 512, 161, torch.bfloat16, None, 0),
    (8, 128, 256, torch.float16, None, 0),     # 256 workgroups of the 8-wave kernel, then one
    (8, 128, 257, torch.float16, None, 0),     # row more
    (2, 64, 1025, torch.bfloat16, None, 8),
]


@pytest.mark.gpu
@pytest.mark.parametrize("i", range(len(CASES)))
def test_prompt_rows_against_oracle(dev, i):
    G, D, M, dtype, low_rank, pad = CASES[i]
    print(f"[gpu] cutoff prompt {CASES[i]}", flush=True)
    xk, Wk, bk = _inputs(G, D, M, dtype, 3.0, seed=8100 + i)
    xv, Wv, bv = _inputs(G, D, M, dtype, 3.0, seed=8200 + i)
    t = lambda a: torch.from_numpy(a).to(device=dev, dtype=dtype)  # noqa: E731
    head = CK.CutoffHead(t(Wk) if G > 1 else t(Wk[0]), t(bk), t(Wv) if G > 1 else t(Wv[0]), t(bv),
                         groups=G, low_rank=low_rank)
    k_out, v_out, len_k, len_v, _, _ = head.kv_process_fused(_dev_rows(xk, dtype, dev, pad),
                                                             _dev_rows(xv, dtype, dev, pad))
    torch.cuda.synchronize()
    ws = CK._WS_CACHE[(dev.index, torch.cuda.current_stream(dev).cuda_stream)]
    n = M * G * D * 2
    _check(f"prompt {i} K", k_out, len_k, xk, Wk, bk, dtype, low_rank, ws[:n].view(dtype))
    _check(f"prompt {i} V", v_out, len_v, xv, Wv, bv, dtype, low_rank, ws[n:2 * n].view(dtype))


@pytest.mark.gpu
def test_special_values_and_unaligned_outputs(dev):
    """Outputs at an odd element offset (element stores) hold what aligned ones do, and rows with
    infinite or NaN inputs come out as from the 8-wave kernel, row by row."""
    G, D, M, dtype = 4, 128, 700, torch.bfloat16
    print("[gpu] cutoff prompt: special values, unaligned outputs", flush=True)
    x, W, b = _inputs(G, D, M, dtype, 3.0, seed=8300)
    x[3, 5], x[4, 200], x[5, 7], x[6, :] = float("inf"), float("-inf"), float("nan"), 0.0
    x[7, 130] = 3.0e38
    t = lambda a: torch.from_numpy(a).to(device=dev, dtype=dtype)  # noqa: E731
    xd, bd = t(x), t(b)
    head = CK.CutoffHead(t(W), bd, t(W), bd, groups=G)
    k, _, lk, lv, _, _ = head.kv_process_fused(xd, xd)
    few, _, lf, _, _, _ = head.kv_process_fused(xd[:16], xd[:16])
    assert torch.equal(lk[:16], lf) and torch.equal(lk, lv)
    assert torch.equal(k[:16].view(torch.int16), few.view(torch.int16))

    lib = _lib.load()
    H = G * D
    out = torch.zeros(2, M * H + 1, dtype=dtype, device=dev)
    ln = torch.zeros(2, M, G, dtype=torch.int32, device=dev)
    ws = torch.zeros(2 * M * H + 1, dtype=dtype, device=dev)
    rc = lib.dkv_cutoff_kv(
        _lib.stream_of(xd), _lib.dtype_code(dtype), xd.data_ptr(), xd.data_ptr(), H,
        head.wt_k.data_ptr(), head.wt_v.data_ptr(), head.b_k.data_ptr(), head.b_v.data_ptr(), 0.1,
        -1, out[0, 1:].data_ptr(), out[1, 1:].data_ptr(), H, ln[0].data_ptr(), ln[1].data_ptr(), G,
        ws[1:].data_ptr(), 2 * M * H * 2, M, G, D)
    assert rc == _lib.DKV_OK
    torch.cuda.synchronize()
    assert torch.equal(ln[0], lk)
    assert torch.equal(out[0, 1:].view(M, H).view(torch.int16), k.view(torch.int16))


@pytest.mark.gpu
@pytest.mark.parametrize("D,dtype", [(128, torch.bfloat16), (128, torch.float16),
                                     (64, torch.bfloat16)])
def test_prompt_counts_equal_decode_counts(dev, D, dtype):
    """A prompt in one call gives every row the count and the masked copy that the decode-size
    kernel gives it, bit for bit: sums in one order, so rounding ties fall alike."""
    G, M = 8, 8192
    print(f"[gpu] cutoff prompt against decode sizes D={D} {dtype}", flush=True)
    x, W, b = _inputs(G, D, M, dtype, 3.0, seed=8400 + D)
    t = lambda a: torch.from_numpy(a).to(device=dev, dtype=dtype)  # noqa: E731
    xd, wd, bd = t(x), t(W), t(b)
    head = CK.CutoffHead(wd, bd, wd, bd, groups=G)
    k, _, lk, _, _, _ = head.kv_process_fused(xd, xd)
    for r in range(0, M, 128):
        few, _, lf, _, _, _ = head.kv_process_fused(xd[r:r + 128], xd[r:r + 128])
        assert torch.equal(lk[r:r + 128], lf), r
        assert torch.equal(k[r:r + 128].view(torch.int16), few.view(torch.int16)), r
