"""The wide head's logits (256 to 1024 inputs) sum each quarter of the inputs by itself in both
kernels, the tiled one of prompts (32- and 64-row tiles) and the split one of few rows: a prompt in
one call leaves the workspace logits, the counts and the masked copies of the same rows in
decode-size calls, bit for bit."""
import pytest
import torch

from dynakv_amd.kernels import cutoff as CK

from test_gpu_cutoff import _inputs

# (D, rows of a prompt): 32-row tiles, then 64-row ones; the last tile of one row
CASES = [(256, 897), (256, 2689), (512, 673), (512, 1409), (1024, 481), (1024, 705)]
SPLIT_ROWS = {256: 384, 512: 192, 1024: 96}  # the most rows that the split kernel takes, one group


def _logits(dev, M, D, dtype):
    ws = CK._WS_CACHE[(dev.index, torch.cuda.current_stream(dev).cuda_stream)]
    return ws[:2 * M * D * 2].view(dtype).view(2, M, D).clone()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D,M", CASES)
def test_prompt_equals_decode_sizes(dev, D, M, dtype):
    print(f"[gpu] wide cutoff D={D} M={M} {dtype}", flush=True)
    n = SPLIT_ROWS[D]
    # the lines between the kernels: more than three split workgroups per CU; 320 tiles of 32 rows
    assert D // 16 * (n // 16) * 2 == 3 * 256
    assert (D // 128 * -(-M // 32) * 2 <= 320) == ((D, M) in CASES[::2])
    x, W, b = _inputs(1, D, 2 * M, dtype, 3.0, seed=8500 + D + M)
    t = lambda a: torch.from_numpy(a).to(device=dev, dtype=dtype)  # noqa: E731
    xk, xv, wd, bd = t(x[:M]), t(x[M:]), t(W[0]), t(b)
    head = CK.CutoffHead(wd, bd, wd.flip(0).contiguous(), bd)
    k, v, lk, lv, _, _ = head.kv_process_fused(xk, xv)
    torch.cuda.synchronize()
    logits = _logits(dev, M, D, dtype)
    bits = lambda a: a.view(torch.int16)  # noqa: E731
    for r in range(0, M, n):
        rows = slice(r, min(M, r + n))
        fk, fv, fl, fm, _, _ = head.kv_process_fused(xk[rows], xv[rows])
        torch.cuda.synchronize()
        assert torch.equal(bits(_logits(dev, rows.stop - r, D, dtype)), bits(logits[:, rows]))
        assert torch.equal(fl, lk[rows]) and torch.equal(fm, lv[rows])
        assert torch.equal(bits(fk), bits(k[rows])) and torch.equal(bits(fv), bits(v[rows]))
