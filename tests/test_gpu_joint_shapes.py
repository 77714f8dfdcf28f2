"""The joint scores' launch shapes (32 tokens of one basis head with the ranks split over the waves,
128 of one head, else 256 of two or 512 of one) on both sides of their boundaries: against the
vector kernel with the bounds of the other scores tests, and a batch row's scores from the shapes
that sum the ranks in one order the same bits. The V pass on both sides of its shortest split."""
import numpy as np
import pytest
import torch

from dynakv_amd import _lib
from dynakv_amd.kernels import joint as J

from helpers import assert_close, cast_np
from test_gpu_joint import THETA, ULP, _case, _dev, _generic_av, _generic_scores

# (B, S, R, n_basis, Hq): with two heads per workgroup 48, 128 and 130 workgroups, with one head
# 128, 129 (half the rows: 66) and 258, tokens one past a 128-token range, one chunk, five chunks (a
# remainder of the four-chunk loop)
CASES = [
    (8, 1025, 64, 2, 8),
    (64, 129, 64, 2, 8),
    (65, 129, 64, 2, 8),
    (43, 513, 160, 3, 12),
    (9, 2049, 32, 2, 2),
    (17, 1025, 224, 4, 16),
    (43, 290, 160, 3, 12),
    (128, 129, 96, 1, 4),
]


def _shape(B, S, nb):
    """The scores' launch shape: "32" (tokens of one head), "128" (of one head), or the large one."""
    if _wg32(B, S, nb) <= 512:
        return "32"
    win = 2048 if S >= 2048 else -(-S // 512) * 512
    tok, heads = (512, 1) if nb % 2 else (256, 2)
    return "128" if -(-S // win) * (win // tok) * (nb // heads) * B <= 128 else f"{tok}x{heads}"


def test_cases_cross_the_boundaries():
    """The listed cases take every shape, and their halves other ones than the whole."""
    whole = [_shape(*c[:2], c[3]) for c in CASES]
    half = [_shape((c[0] + 1) // 2, c[1], c[3]) for c in CASES]
    assert set(whole) == {"128", "256x2", "512x1"}
    crossed = {(w, h) for w, h, c in zip(whole, half, CASES)
               if w != h and _wg32(c[0] // 2, c[1], c[3]) > 512}
    assert crossed >= {("256x2", "128"), ("512x1", "128")}


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
        half = (B + 1) // 2
        if _wg32(B // 2, S, nb) > 512:  # half the rows: the 128-token shape beside the large one
            rows = slice(0, half)
            part = J.joint_scores(d["q"][rows], d["kb"], d["fk"][rows], d["lk"][rows],
                                  d["ok"][rows], **kw)
            assert torch.equal(part, got[rows])


def _wg32(B, S, nb):
    return B * ((S + 31) // 32) * nb


# (B, S, R, n_basis, Hq): the 32-token shape up to 512 workgroups: fewer chunks than waves, chunks
# that do not divide among them, a last block of one token, 1 to 8 query heads per basis
FEW = [
    (1, 1, 32, 1, 8),
    (2, 33, 96, 8, 32),
    (1, 17, 1024, 8, 32),
    (3, 65, 288, 3, 24),
    (1, 2048, 512, 8, 8),
    (16, 512, 128, 2, 4),
]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("i", range(len(FEW)))
def test_scores_of_few_tokens(dev, i, dtype):
    B, S, R, nb, Hq = FEW[i]
    assert _wg32(B, S, nb) <= 512
    print(f"[gpu] joint scores few tokens {FEW[i]} {dtype}", flush=True)
    d = _dev(_case(B, S, R, nb, Hq=Hq, dtype=dtype, seed=600 + i, exact_end=True), dev, dtype)
    for mode, odt in ((0, dtype), (1, torch.float32)):
        got = J.joint_scores(d["q"], d["kb"], d["fk"], d["lk"], d["ok"], theta=THETA, mode=mode,
                             out_dtype=odt).float()
        ref = _generic_scores(d, d["kb"], mode, odt).float()
        fin = torch.isfinite(ref)
        assert torch.equal(torch.isfinite(got), fin)
        err = (got[fin] - ref[fin]).abs()
        tol = (2 * ULP[dtype] if mode == 0 else 1e-4) * ref[fin].abs() + 1e-4
        assert (err <= tol).all(), float(err.max())
        if mode == 0:
            masked = (d["lk"] == 0)[:, None, :]
            assert torch.equal(got.masked_select(masked), ref.masked_select(masked))


@pytest.mark.gpu
@pytest.mark.parametrize("S", [800, 801, 1025])  # 50 splits of 16; 26 of 32, the last of one token
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_v_pass_shortest_split(dev, S, dtype):
    B, R, nb, Hq = 2, 160, 4, 16
    floats = _lib.load().dkv_joint_av_workspace_floats(B, Hq, S, R)
    assert floats == B * Hq * ({800: 50, 801: 26, 1025: 33}[S] * (4 + 1024) + 256)
    print(f"[gpu] joint av split line S={S} {dtype}", flush=True)
    d = _dev(_case(B, S, R, nb, Hq=Hq, dtype=dtype, seed=S, exact_end=True), dev, dtype)
    z = cast_np(np.random.default_rng(S).standard_normal((B, Hq, S)) * 2, dtype)
    sc = torch.from_numpy(z).to(dev, dtype)
    got = J.joint_av(sc, d["vb"], d["fv"], d["lv"], d["ov"], mode=0, out_dtype=torch.float32)
    ref = _generic_av(sc, d, d["vb"], 0, torch.float32)
    # the bounds of the other V-pass tests: fp16 caches hold P in fp16, 2^-11 per term
    assert_close(got, ref.cpu().numpy(), "av", tol_rel=2e-3,
                 tol_abs=2e-4 if dtype == torch.bfloat16 else 1e-3)
