"""Prefill attention's launch shapes (two query blocks x 4 waves, 1 x 8, 1 x 4, chosen by the
number of 128-query workgroups) at the edges of their query blocks and key tiles, against the
oracle to the bars of the other prefill tests."""
import numpy as np
import pytest
import torch

from dynakv_amd.kernels.prefill import prefill_attention
from oracle import prefill as P

from helpers import assert_close, cast_np

# (B, Hq, Hkv, Sq, Sk, causal, dtype, padded): 128-query workgroups below 257, up to 1024, above
CASES = [
    (1, 4, 2, 63, 63, True, torch.bfloat16, False),
    (1, 4, 1, 65, 193, True, torch.float16, True),
    (8, 32, 8, 128, 128, True, torch.bfloat16, True),    # 256: the last of the small shape
    (9, 32, 4, 127, 140, True, torch.bfloat16, False),   # 288: 8 waves
    (9, 32, 8, 17, 64, True, torch.float16, False),
    (16, 32, 8, 129, 129, True, torch.float16, True),    # 1024, a block of one query
    (33, 32, 8, 33, 65, True, torch.bfloat16, False),    # 1056: two query blocks per wave
    (33, 32, 2, 128, 128, True, torch.float16, True),
    (34, 32, 8, 20, 130, False, torch.bfloat16, False),
]


@pytest.mark.gpu
@pytest.mark.parametrize("i", range(len(CASES)))
def test_launch_shapes_against_oracle(dev, i):
    B, Hq, Hkv, Sq, Sk, causal, dtype, padded = CASES[i]
    print(f"[gpu] prefill shape {CASES[i]}", flush=True)
    rng = np.random.default_rng(9100 + i)
    q = cast_np(2.0 * rng.standard_normal((B, Hq, Sq, 128)).astype(np.float32), dtype)
    k = cast_np(rng.standard_normal((B, Hkv, Sk, 128)).astype(np.float32), dtype)
    v = cast_np(rng.standard_normal((B, Hkv, Sk, 128)).astype(np.float32), dtype)
    start = rng.integers(0, Sk + 1, B).astype(np.int32) if padded else None
    t = lambda a: torch.from_numpy(a).to(device=dev, dtype=dtype)  # noqa: E731
    ks = None if start is None else torch.from_numpy(start).to(dev)
    # rows of a wider buffer whose tail holds NaN: keys past Sk are never read into a result
    kd = torch.full((B, Hkv, Sk + 64, 128), float("nan"), dtype=dtype, device=dev)
    vd = kd.clone()
    kd[:, :, :Sk], vd[:, :, :Sk] = t(k), t(v)
    got = prefill_attention(t(q), kd[:, :, :Sk], vd[:, :, :Sk], causal=causal, kstart=ks,
                            out_dtype=torch.float32)
    low = prefill_attention(t(q), kd[:, :, :Sk], vd[:, :, :Sk], causal=causal, kstart=ks)
    torch.cuda.synchronize()
    rows = sorted({0, B // 2, B - 1})
    ref = P.attention(q[rows], k[rows], v[rows], causal=causal,
                      **({} if start is None else dict(kstart=start[rows])))
    assert_close(got[rows], ref, f"prefill shape {i}")
    assert torch.equal(low, got.to(dtype))
