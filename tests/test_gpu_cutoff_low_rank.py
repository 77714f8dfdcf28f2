"""``low_rank`` of any size: caps past the width, and negative ones, keep every count."""
import sys

import pytest
import torch

from dynakv_amd.kernels.cutoff import CutoffHead


@pytest.mark.gpu
@pytest.mark.parametrize("low_rank", [128, 1 << 31, 1 << 40, sys.maxsize, -1, -(1 << 40)])
def test_low_rank_past_the_width(dev, low_rank):
    print(f"[gpu] cutoff low_rank {low_rank}", flush=True)
    g = torch.Generator().manual_seed(9)
    r = lambda *d: torch.randn(*d, generator=g).to(dev, torch.bfloat16)  # noqa: E731
    w, b, x = r(2, 128, 128) * 0.2, r(2, 128), r(1, 20, 256)
    want = CutoffHead(w, b, w, b, groups=2).kv_process_fused(x, x)
    got = CutoffHead(w, b, w, b, groups=2, low_rank=low_rank).kv_process_fused(x, x)
    for a, e in zip(got[:4], want[:4]):
        assert torch.equal(a, e)
