"""``joint_flops`` against a count over the launch's own blocks, on either side of the line between
the 32-token shape and the window-sorted ones."""
import pytest
import torch

from dynakv_amd.kernels.joint import joint_flops


def _count(lens, R, nb):
    """32-rank chunks times token slots, block by block, for all basis heads."""
    B, S = lens.shape
    few = B * -(-S // 32) * nb <= 512
    win = 32 if few else (2048 if S >= 2048 else -(-S // 512) * 512)
    total = 0
    for row in lens.tolist():
        for w in range(0, S, win):
            c = [-(-min(max(n, 0), R) // 32) for n in row[w:w + win]]
            c += [0] * (win - len(c))
            if few:
                total += win * max(c)
            else:
                c.sort()
                total += sum(16 * c[i + 15] for i in range(0, win, 16))
    return total * nb


@pytest.mark.parametrize("B,S,R,nb", [(1, 1, 32, 1), (2, 70, 256, 8), (1, 2048, 1024, 8),
                                      (1, 2080, 1024, 8), (3, 1500, 160, 3), (40, 513, 96, 2),
                                      (2, 5000, 512, 8)])
def test_joint_flops(B, S, R, nb):
    g = torch.Generator().manual_seed(S)
    lens = torch.randint(-1, R + 9, (B, S), generator=g, dtype=torch.int32)
    assert joint_flops(lens, R, nb, B) == _count(lens, R, nb) * 2 * 128 * 32
