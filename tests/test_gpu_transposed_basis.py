"""Transposed bases (unit rank stride) are read in place: decode attention and the prefill
reconstruction give the bits they give from rank-major copies, over ranks, split structures, the
separate merge kernel, shared and offset bases; other strides still take a copy."""
import numpy as np
import pytest
import torch

from dynakv_amd.kernels import decode as D
from dynakv_amd.kernels import prefill as P
from dynakv_amd.synthetic import make_case

from helpers import assert_close, oracle_grouped, packed_from_case

# (B, G, Hq, S, R, dtype, route, split_len): one split, several, pairs of tiles, ranks below 128,
# 16 heads per group, more units than arrival counters
CASES = [
    (1, 8, 32, 96, 128, torch.bfloat16, "short_fused", 0),
    (2, 4, 16, 700, 128, torch.float16, "long_two_stage", 0),
    (1, 2, 32, 513, 72, torch.bfloat16, "long_two_stage", 128),
    (3, 2, 4, 1100, 8, torch.float16, "short_fused", 512),
    (2, 8, 32, 2050, 64, torch.bfloat16, "long_two_stage", 0),
    (2049, 8, 8, 17, 16, torch.bfloat16, "long_two_stage", 0),
]


def _t(b: torch.Tensor) -> torch.Tensor:
    return b.transpose(1, 2).contiguous().transpose(1, 2)


@pytest.mark.gpu
@pytest.mark.parametrize("i", range(len(CASES)))
def test_decode_matches_rank_major(dev, i):
    B, G, Hq, S, R, dtype, route, sl = CASES[i]
    print(f"[gpu] transposed basis {CASES[i]}", flush=True)
    case = make_case(B=B, G=G, Hq=Hq, S=S, R=R, mean=0.4, force_frac=0.05, seed=60 + i)
    d = packed_from_case(case, dtype, dev)
    kt, vt = _t(d["k_basis"]), _t(d["v_basis"])
    assert kt.stride(1) == 1 and D.splitk_layout(d["q"], kt, vt, d["k_flat"], d["v_flat"]).transposed
    run = lambda k, v: D.grouped_decode_attention(  # noqa: E731
        d["q"], d["k_flat"], d["v_flat"], d["lens_k"], d["offs_k"], d["lens_v"], d["offs_v"], k, v,
        theta=case.theta, route=route, split_len=sl, out_dtype=torch.float32)
    got, want = run(kt, vt), run(d["k_basis"], d["v_basis"])
    assert torch.equal(got, want)
    # mixed orders take copies
    assert not D.splitk_layout(d["q"], kt, d["v_basis"], d["k_flat"], d["v_flat"]).transposed
    assert torch.equal(run(kt, d["v_basis"]), want)
    if B <= 3:
        assert_close(got, oracle_grouped(case, d["host"], route, str(dtype)[6:]), f"transposed {i}")


@pytest.mark.gpu
def test_decode_views(dev):
    """A shared basis (zero head stride), bases cut from wider buffers, and strides the kernel does
    not take (odd dim stride, ranks that are not a multiple of 8)."""
    print("[gpu] transposed basis views", flush=True)
    case = make_case(B=2, G=1, Hq=4, S=300, R=64, mean=0.4, seed=80)
    d = packed_from_case(case, torch.bfloat16, dev)
    kb, vb = d["k_basis"], d["v_basis"]
    run = lambda k, v: D.grouped_decode_attention(  # noqa: E731
        d["q"], d["k_flat"], d["v_flat"], d["lens_k"], d["offs_k"], d["lens_v"], d["offs_v"], k, v,
        theta=case.theta, out_dtype=torch.float32)
    want = run(kb, vb)
    for ld in (64, 72, 96, 67):
        wide = [torch.zeros(1, 130, ld, dtype=kb.dtype, device=dev) for _ in range(2)]
        for w, b in zip(wide, (kb, vb)):
            w[:, 1:129, :64] = b.transpose(1, 2)
        k, v = (w[:, 1:129, :64].transpose(1, 2) for w in wide)
        lay = D.splitk_layout(d["q"], k, v, d["k_flat"], d["v_flat"])
        assert lay.transposed == (ld % 8 == 0)
        assert torch.equal(run(k, v), want)
    lay = D.splitk_layout(d["q"], _t(kb).expand(4, -1, -1), _t(vb).expand(4, -1, -1), d["k_flat"],
                          d["v_flat"])
    assert lay.transposed and lay.n_kv == 1
    odd = make_case(B=1, G=2, Hq=4, S=40, R=60, mean=0.5, seed=81)
    o = packed_from_case(odd, torch.float16, dev)
    assert not D.splitk_layout(o["q"], _t(o["k_basis"]), _t(o["v_basis"]), o["k_flat"],
                               o["v_flat"]).transposed


@pytest.mark.gpu
@pytest.mark.parametrize("B,G,S,R,dtype", [(2, 4, 77, 128, torch.float16),
                                           (16, 8, 300, 72, torch.bfloat16),
                                           (1, 2, 1, 8, torch.bfloat16)])
def test_recon_matches_rank_major(dev, B, G, S, R, dtype):
    print(f"[gpu] recon transposed basis {B} {G} {S} {R}", flush=True)
    rng = np.random.default_rng(S)
    t = lambda *d: torch.from_numpy(rng.standard_normal(d).astype(np.float32)).to(dev, dtype)  # noqa: E731
    ck, cv, kb, vb = t(B * G, S, R), t(B * G, S, R), t(G, R, 128), t(G, R, 128)
    kw = dict(batch=B, theta=500000.0, pos0=9)
    want = P.recon_kv(ck, cv, kb, vb, **kw)
    for k, v in ((_t(kb), _t(vb)), (_t(kb), vb)):
        got = P.recon_kv(ck, cv, k, v, **kw)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
