"""Device memory that a context holds after a call: buffers that are whole
powers of two for lists of 2^m items take no more than that."""
import pytest
import torch

import redzone_amd as rz
from tests.parity import announce

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def _held(n, k, call):
    """MiB that a fresh context takes for one call on n 4-byte items, the second
    context that makes it (the first one's call loads the kernels and what the
    runtime keeps for them)."""
    A = torch.empty(n, dtype=torch.int32, device="cuda")
    R = torch.empty(k, dtype=torch.int32, device="cuda")
    for _ in range(2):
        ctx = rz.Context(0)
        ctx.gen_payload(A, 1)
        ctx.gen_uniform_removals(R, n, 2)
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        call(ctx, A, R)
        torch.cuda.synchronize()
        held = (before - torch.cuda.mem_get_info()[0]) / MIB
        assert ctx.check_errors() == 0
        ctx.close()
    return held


def test_partition_scratch():
    """Entries of 4 bytes an item and the n-bit bitmap."""
    n = 1 << 26
    held = _held(n, n // 4, lambda c, a, r: c.partition(a, r))
    announce("scratch partition", n, held)
    assert held <= (4 * n + n // 8) / MIB + 32


def test_dense_scratch():
    """Tail marks' entries (4 k), moves and bins (8 bytes a removal, 8 an item of
    the head), and orphans (4 and 4 bytes for half of the removals, and one more,
    rounded up to a power of two)."""
    n, k = 1 << 26, 1 << 25
    cfg = rz.TileConfig(1024, 8, 1024, 5, 12, 2)
    held = _held(n, k, lambda c, a, r: c.remove(a, r, config=cfg, flags=rz.RZ_PRESERVE_REMOVALS))
    announce("scratch dense", n, held)
    # the flag keeps a copy of the removals aside in the forms that write them (4 k)
    assert held <= (4 * k + 8 * k + 8 * (n - k) + 8 * k + 4 * k + k // 8) / MIB + 32
