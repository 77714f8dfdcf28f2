"""fp16 cutoff probabilities round twice, as the reference's softmax does: the fp32 quotient first,
then to fp16. The rows below have a probability whose fp32 quotient is a tie of fp16 while the
exact quotient is not, so one rounding instead of two gives the other fp16 neighbour, and the
threshold is the larger of the two: the count says which was taken."""
import numpy as np
import pytest
import torch

from dynakv_amd.kernels.compressed_cache import CustomDynamicCache
from dynakv_amd.kernels.cutoff import CutoffHead
from dynakv_amd.kernels.layer import DecodeLayerPlan

# (D, k, t, L): logits 0 at the first k positions, L at the next t, the lowest fp16 after them
ROWS = [
    (64, 5, 59, -9.2265625),
    (128, 3, 64, -9.671875),
    (128, 10, 118, -9.2265625),
    (256, 5, 251, -6.578125),
    (256, 17, 239, -6.2890625),
    (512, 10, 502, -6.578125),
    (512, 21, 491, -7.234375),
    (1024, 8, 1016, -10.59375),
    (1024, 11, 512, -7.40625),
]


def _logits(D, k, t, L):
    z = np.full(D, -65504.0, np.float32)
    z[:k] = 0.0
    z[k:k + t] = L
    return z


def _sum(D, k, t, L, rel=0.0):
    """The row's softmax denominator in fp32, in the kernels' order: D / 64 consecutive terms per
    lane, then a tree over neighbouring lanes. ``rel``: relative error put on exp(L)."""
    x = np.zeros((64, D // 64), np.float32)
    flat = x.reshape(-1)
    flat[:k] = 1.0
    flat[k:k + t] = np.float32(np.exp(np.float64(L)) * (1.0 + rel))
    p = np.zeros(64, np.float32)
    for e in range(D // 64):
        p = p + x[:, e]
    while p.size > 1:
        p = p[0::2] + p[1::2]
    return p[0]


def _tie(D, k, t, L):
    """(probability of the first positions rounded twice, rounded once)."""
    s = _sum(D, k, t, L)
    return np.float16(np.float32(1.0) / s), np.float16(1.0 / np.float64(s))


def _expected(D, k, t, L):
    two, one = _tie(D, k, t, L)
    return float(max(two, one)), D if two > one else D - 1


@pytest.mark.parametrize("row", ROWS)
def test_rows_sit_on_a_tie(row):
    """The frozen rows are what they claim, whatever the last bits of the device's exp(L)."""
    D, k, t, L = row
    assert float(np.float16(L)) == L and k + t <= D
    assert _sum(*row) == _sum(*row, rel=2.0 ** -22) == _sum(*row, rel=-(2.0 ** -22))
    two, one = _tie(*row)
    assert two != one and abs(int(two.view(np.int16)) - int(one.view(np.int16))) == 1
    thr, n = _expected(*row)
    # the first prefix sum is the first probability; the second passes the threshold either way
    assert (float(two) >= thr) == (n == D) and 2 * float(min(two, one)) >= thr


def _head(row, G, dev):
    D = row[0]
    thr, n = _expected(*row)
    w = torch.zeros(G, D, D, dtype=torch.float16, device=dev)
    b = torch.from_numpy(_logits(*row)).to(dev, torch.float16).expand(G, D).contiguous()
    return CutoffHead(w, b, w, b, groups=G, threshold=thr), n


@pytest.mark.gpu
@pytest.mark.parametrize("M", [5, 353, 1400])  # decode rows, a prompt's, the 64-row logit tiles
@pytest.mark.parametrize("row", ROWS)
def test_counts_round_twice(dev, row, M):
    D = row[0]
    G = 8 if D <= 128 else 1
    print(f"[gpu] cutoff fp16 ties D={D} M={M}", flush=True)
    head, n = _head(row, G, dev)
    x = torch.randn(M, G * D, device=dev).to(torch.float16)
    for rows in (x, x.flip(0)):
        k, v, lk, lv, _, _ = head.kv_process_fused(rows, rows)
        assert (lk == n).all() and (lv == n).all()
        want = rows.view(M, G, D).clone()
        want[..., n:] *= 0
        assert torch.equal(k, want.view(M, G * D)) and torch.equal(v, k)


@pytest.mark.gpu
@pytest.mark.parametrize("row", [r for r in ROWS if r[0] <= 128])
def test_layer_step_counts_round_twice(dev, row):
    D, B, G, Hq, S0 = row[0], 3, 2, 4, 20
    print(f"[gpu] layer step fp16 ties D={D}", flush=True)
    head, n = _head(row, G, dev)
    basis = torch.randn(G, D, 128, device=dev).to(torch.float16)
    cache = CustomDynamicCache()
    for S in (S0, 1):  # the prompt, then the append that grows the buffers
        x = torch.randn(B * G, S, D, device=dev).to(torch.float16)
        ln = torch.full((B * G, S), D, dtype=torch.int32, device=dev)
        cache.update_sp(x, ln, x, ln, D, 0, D)
    plan = DecodeLayerPlan(cache, 0, head, basis, basis, batch=B, heads=Hq, theta=1e4)
    assert plan.can_step()
    q = torch.randn(B, Hq, 128, device=dev).to(torch.float16)
    c = torch.randn(B, G * D, device=dev).to(torch.float16)
    plan.step(q, c, c, S0 + 1)
    for slot in (cache.key_cache_sp[0], cache.value_cache_sp[0]):
        assert (slot[1][:, S0 + 1] == n).all()
