"""Tail marks gathered by ranges in LDS (lists that lose a quarter of their items
or more), in every form that marks by itself, against the CPU oracle: the edges of
the rule, of ranges, chunks and words."""
import pytest
import torch

import redzone_amd as rz
from redzone_amd import workloads as W
from tests.parity import announce, expected_canonical, gpu_remove_parity

pytestmark = pytest.mark.gpu

# one launch with slices of 2^10 and 2^12 pairs, fused, three kernels, dense with marks of its own kernel
SHAPES = [(256, 4, 512, 6, 12, 1), (512, 8, 512, 6, 12, 1), (512, 4, 512, 4, 0, 1), (256, 4, 512, 0, 0, 1),
          (512, 8, 1024, 5, 10, 1)]


@pytest.mark.parametrize("esz,pattern", [(4, "uniform"), (8, "tail_heavy"), (16, "uniform"), (4, "clustered")])
@pytest.mark.parametrize("k", [(1 << 15) - 1, 1 << 15, (1 << 16) + 33, 3 * 131072 + 1, (1 << 20) - 31, (1 << 20) + 1])
def test_range_marks(ctx, oracle, esz, pattern, k):
    top = 17 * k // 4  # the rule's last n, and the first beyond it
    for n in (k + 1, 2 * k + 5, top, top + 1):
        if n > 3 * k and (k > 1 << 18 or pattern == "clustered"):
            continue
        A = W.payload(esz, n, seed=k % 97)
        R = W.removals(pattern, n, k, seed=k % 89)
        want = expected_canonical(oracle, A.numpy(), R.numpy())
        for s in SHAPES:
            announce("range marks", esz, pattern, k, n, s)
            gpu_remove_parity(ctx, oracle, A, R, config=rz.TileConfig(*s), want=want)
    assert ctx.check_errors() == 0


def test_range_marks_counted(ctx):
    """The tail removals counted by the one-launch form are those of the list."""
    k, n = 70001, 150000
    R = W.removals("uniform", n, k, seed=3)
    d = W.payload(4, n, seed=4).cuda()
    ctx.remove(d, R.cuda(), flags=rz.RZ_STATS, config=rz.TileConfig(512, 4, 512, 6, 12, 1))
    torch.cuda.synchronize()
    assert ctx.last_stats().tail_removals == int((R >= n - k).sum())


@pytest.mark.parametrize("order", ["rising", "falling", "pairs", "sorted"])
def test_range_marks_of_runs(ctx, oracle, order):
    """Removals whose neighbours share bitmap words, in every order of a row."""
    k = 40000 + 77
    n = 2 * k + 3
    R = torch.arange(n - k - k // 3, n - k // 3, dtype=torch.int32)
    if order == "falling":
        R = R.flip(0).contiguous()
    elif order == "pairs":  # two runs that alternate lane by lane
        R = torch.stack([R[: k // 2], R[k - k // 2:]], 1).reshape(-1)[: k - 1].contiguous()
    elif order == "sorted":
        R = W.uniform_removals(n, k, seed=9).sort().values.contiguous()
    A = W.payload(4, n, seed=8)
    want = expected_canonical(oracle, A.numpy(), R.numpy())
    for s in SHAPES:
        announce("range marks runs", order, s)
        gpu_remove_parity(ctx, oracle, A, R, config=rz.TileConfig(*s), want=want)
    d = A.cuda()
    assert ctx.partition(d, R.cuda()) == n - len(R)
    keep = torch.ones(n, dtype=torch.bool)
    keep[R.long()] = False
    assert torch.equal(d[: n - len(R)].cpu(), A[keep])
