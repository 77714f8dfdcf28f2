"""The joint scores' two launch shapes (few workgroups: 128 tokens of one basis head each; else 256
of two or 512 of one) on both sides of their boundary: against the vector kernel with the bounds of
the other scores tests, and a batch row's scores the same bits from either shape."""
import pytest
import torch

from dynakv_amd.kernels import joint as J

from test_gpu_joint import THETA, ULP, _case, _dev, _generic_scores

# (B, S, R, n_basis, Hq): 128 and 130 workgroups of two heads, 129 of one head, tokens one past a
# 128-token range, one chunk, five chunks (a remainder of the four-chunk loop)
CASES = [
    (64, 129, 64, 2, 8),
    (65, 129, 64, 2, 8),
    (43, 513, 160, 3, 12),
    (9, 2049, 32, 2, 2),
    (17, 1025, 224, 4, 16),
]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("i", range(len(CASES)))
def test_scores_launch_shapes(dev, i, dtype):
    B, S, R, nb, Hq = CASES[i]
    print(f"[gpu] joint scores shape {CASES[i]} {dtype}", flush=True)
    d = _dev(_case(B, S, R, nb, Hq=Hq, dtype=dtype, seed=500 + i, exact_end=True), dev, dtype)
    for mode, odt in ((0, dtype), (1, torch.float32)):
        kw = dict(theta=THETA, mode=mode, out_dtype=odt)
        got = J.joint_scores(d["q"], d["kb"], d["fk"], d["lk"], d["ok"], **kw)
        ref = _generic_scores(d, d["kb"], mode, odt).float()
        fin = torch.isfinite(ref)
        assert torch.equal(torch.isfinite(got.float()), fin)
        err = (got.float()[fin] - ref[fin]).abs()
        tol = (2 * ULP[dtype] if mode == 0 else 1e-4) * ref[fin].abs() + 1e-4
        assert (err <= tol).all(), float(err.max())
        for b in (0, B - 1):  # one row alone: always the small shape
            one = J.joint_scores(d["q"][b:b + 1], d["kb"], d["fk"][b:b + 1], d["lk"][b:b + 1],
                                 d["ok"][b:b + 1], **kw)
            assert torch.equal(one[0], got[b])
