"""The dense form (variant 5) at the edges of its passes, against the CPU
oracle: tiles of the split (16,384 pairs of 4-byte items), move regions (one
per XCD), bin chunks, 128 KiB head windows and the red zone's last word."""
import pytest
import torch

import redzone_amd as rz
from redzone_amd import workloads as W
from tests.parity import announce, expected_canonical, first_mismatch, gpu_remove_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("esz", [4, 8, 16])
@pytest.mark.parametrize("k", [1, 63, 65, 16383, 16385, 8 * 16384 - 1, 8 * 16384 + 33, 300001])
def test_dense_tile_edges(ctx, oracle, esz, k):
    window = (1 << 17) // esz
    for head in (1, window - 1, window, 2 * window + 1, 40 * window + 7):
        n = k + head
        for pattern in ("uniform", "clustered"):
            A = W.payload(esz, n, seed=k)
            R = W.removals(pattern, n, k, seed=k + head)
            want = expected_canonical(oracle, A.numpy(), R.numpy())
            for cfg in ((1024, 8 if esz < 16 else 4, 5, 12, 2), (256, 4, 5, 3, 2), (512, 4, 5, 9, 0)):
                announce("dense edges", esz, k, head, pattern, cfg)
                wg, it, v, lg, ch = cfg
                gpu_remove_parity(ctx, oracle, A, R, config=rz.TileConfig(wg, it, 1024, v, lg, ch), want=want)


def test_dense_keeps_unnamed_items(ctx):
    """Items of the head that no removal names keep their bits, and the red zone is only read."""
    n, k = 1 << 22, 1 << 20
    A = W.edge_payload(4, n, seed=3)
    R = W.uniform_removals(n, k, seed=4)
    dA, dR = A.cuda(), R.cuda()
    ctx.remove(dA, dR, config=rz.TileConfig(1024, 8, 1024, 5, 12, 2), flags=rz.RZ_PRESERVE_REMOVALS)
    keep = torch.ones(n, dtype=torch.bool)
    keep[R.long()] = False
    keep[n - k:] = False
    assert first_mismatch(dA.cpu()[keep].numpy(), A[keep].numpy()) < 0
    assert torch.equal(dR.cpu(), R)
    assert torch.equal(dA.cpu()[n - k:], A[n - k:])


@pytest.mark.parametrize("esz,n,k", [(4, (1 << 28) + 77, (1 << 25) + 3), (8, (1 << 26) + 70001, 1 << 21),
                                     (8, (1 << 27) - 3, 50000001), (16, (1 << 26) + (1 << 23) + 1, 1 << 20),
                                     (16, (1 << 27) + 5, 40000003)])
@pytest.mark.parametrize("pattern", ["uniform", "block"])
def test_dense_single_stores(ctx, esz, n, k, pattern):
    """Lists whose bins are written one store per entry: every item of the list
    beside the three-kernel form's, removals at random and in one block (bins
    filled to their last position)."""
    announce("dense stores", esz, n, k, pattern)
    A = torch.empty((n,) if esz == 4 else (n, esz // 4), dtype=torch.int32, device="cuda")
    ctx.gen_payload(A, 11)
    want = A.clone()
    if pattern == "uniform":
        R = torch.empty(k, dtype=torch.int32, device="cuda")
        ctx.gen_uniform_removals(R, n, 12)
    else:
        R = torch.arange(1000, 1000 + k, dtype=torch.int32, device="cuda")
    ctx.remove(want, R, config=rz.TileConfig(512, 8, 4096, 0, 0, 1), flags=rz.RZ_PRESERVE_REMOVALS)
    for lg in (12, 11, 3):
        B = A.clone()
        cfg = rz.TileConfig(1024, 8 if esz < 16 else 4, 1024, 5, lg, 2)
        assert ctx.remove(B, R, config=cfg, flags=rz.RZ_PRESERVE_REMOVALS) == n - k
        assert ctx.check_errors() == 0
        assert torch.equal(B[: n - k], want[: n - k]), lg
        assert torch.equal(B[n - k:], A[n - k:]), "the red zone is only read"
        del B
