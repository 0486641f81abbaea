"""Tail marks gathered by ranges in LDS (lists that lose a quarter of their items
or more), in every form that marks by itself, against the CPU oracle: the edges of
the rule, of ranges, chunks and words."""
import pytest
import torch

import redzone_amd as rz
from redzone_amd import workloads as W
from tests.parity import announce, expected_canonical, first_mismatch, gpu_remove_parity

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


@pytest.mark.parametrize("order", ["random", "sorted", "sorted sparse", "tail block", "falling block", "pairs", "last row"])
@pytest.mark.parametrize("k", [1000, 16384 - 5, 20001])
def test_marks_one_by_one_or_in_runs(ctx, oracle, order, k):
    """Fewer removals than the ranges take: rounds that look for runs of marks in
    one word, in every form that marks by itself, and the partition's atomics."""
    n = 300 * k if order == "sorted sparse" else 2 * k + 7
    R = W.uniform_removals(n, k, seed=k)
    if order.startswith("sorted"):
        R = R.sort().values.contiguous()
    elif order in ("tail block", "falling block", "pairs"):
        R = torch.arange(n - k - k // 5, n - k // 5, dtype=torch.int32)
        if order == "falling block":
            R = R.flip(0).contiguous()
        elif order == "pairs":  # two runs that alternate lane by lane
            R = torch.stack([R[: k // 2], R[k - k // 2:]], 1).reshape(-1)[: k - 1].contiguous()
    elif order == "last row":  # a run in the last removals only
        R = torch.cat([torch.arange(0, k - 200), torch.arange(n - 200, n)]).to(torch.int32)
    A = W.payload(4, n, seed=9)
    want = expected_canonical(oracle, A.numpy(), R.numpy())
    for s in ((256, 4, 512, 6, 12, 1), (256, 2, 4096, 6, 10, 1), (512, 4, 512, 6, 10, 1), (256, 4, 1024, 6, 11, 1),
              (256, 4, 512, 4, 0, 1), (256, 4, 512, 0, 0, 1), (256, 4, 512, 1, 0, 1), (256, 8, 0, 2, 1, 1),
              (256, 4, 4096, 3, 0, 1), (512, 8, 1024, 5, 10, 0)):
        for flags in ((0, rz.RZ_SORTED) if order.startswith("sorted") or order in ("tail block", "last row") else (0,)):
            announce("marks", order, k, s, flags)
            gpu_remove_parity(ctx, oracle, A, R, config=rz.TileConfig(*s), flags=flags, want=want)
    k = R.shape[0]
    d, dR = A.cuda(), R.cuda()
    b = ctx.batch([(d, dR)], flags=rz.RZ_PRESERVE_REMOVALS)
    b.launch()
    torch.cuda.synchronize()
    assert first_mismatch(d.cpu().numpy()[: n - k], want[: n - k]) < 0
    d = A.cuda()
    assert ctx.partition(d, dR) == n - k
    keep = torch.ones(n, dtype=torch.bool)
    keep[R.long()] = False
    assert torch.equal(d[: n - k].cpu(), A[keep])
    assert ctx.check_errors() == 0


@pytest.mark.parametrize("k,n", [(1 << 21, 4 * (1 << 21) // 3), ((1 << 21) + 1, 4 * (1 << 21) // 3), ((1 << 23) - 1, 11000000),
                                 (1 << 23, 11000000), ((1 << 22) + 33, 17 * ((1 << 22) + 33) // 4),
                                 ((1 << 22) + 33, 17 * ((1 << 22) + 33) // 4 + 1)])
def test_range_marks_of_long_lists(ctx, oracle, k, n):
    """The largest ranges (2^18 positions), the removals from which marks are made one
    by one again, and the rule's last n for many removals."""
    A, R = W.payload(4, n, seed=21), W.uniform_removals(n, k, seed=22)
    want = expected_canonical(oracle, A.numpy(), R.numpy())
    for s in ((512, 8, 768, 4, 0, 1), (512, 8, 4096, 0, 0, 1)):
        announce("range marks, long", k, n, s)
        gpu_remove_parity(ctx, oracle, A, R, config=rz.TileConfig(*s), want=want)
    assert ctx.check_errors() == 0
