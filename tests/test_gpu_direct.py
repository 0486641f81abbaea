"""The direct form (variant 7: independent workgroups, maps of all pairs in
LDS) and the added items that rz_add_remove reads in place, against the CPU
oracle: bit-exact survivors at the edges of words, steps, slices and of the
form's range."""
import numpy as np
import pytest
import torch

import redzone_amd as rz
from redzone_amd import workloads as W
from tests.parity import announce, expected_canonical, first_mismatch, gpu_remove_parity

pytestmark = pytest.mark.gpu

SHAPES = [(256, 1), (256, 2), (256, 4), (512, 1), (512, 2), (512, 4), (1024, 1), (1024, 2)]
MAX_K = 1 << 17


@pytest.mark.parametrize("esz", [4, 8, 16])
@pytest.mark.parametrize("k", [1, 63, 64, 65, 255, 256, 1023, 1025, 4096, 4097, 16384 + 1])
def test_direct_edges(ctx, oracle, esz, k):
    for pattern, n in (("uniform", 40 * k + 7), ("uniform", 2 * k + 1), ("tail_heavy", 3 * k + 5),
                       ("clustered", k + k // 3 + 2)):
        A = W.payload(esz, n, seed=k)
        R = W.removals(pattern, n, k, seed=k + 1)
        want = expected_canonical(oracle, A.numpy(), R.numpy())
        for wg, it in SHAPES:
            announce("direct", esz, k, pattern, wg, it)
            gpu_remove_parity(ctx, oracle, A, R, config=rz.TileConfig(wg, it, 0, 7, 0, 1), want=want)


@pytest.mark.parametrize("k", [MAX_K - 1, MAX_K, MAX_K + 1])
def test_direct_range_end(ctx, oracle, k):
    """The largest k of the form, and one above it (refused)."""
    n = 2 * k + 11
    A = W.payload(4, n, seed=5)
    R = W.uniform_removals(n, k, seed=6)
    for wg, it in ((256, 4), (1024, 1)):
        announce("direct end", k, wg, it)
        if k > MAX_K:
            with pytest.raises(rz.RedzoneError):
                ctx.remove(A.cuda(), R.cuda(), config=rz.TileConfig(wg, it, 0, 7, 0, 1))
        else:
            gpu_remove_parity(ctx, oracle, A, R, config=rz.TileConfig(wg, it, 0, 7, 0, 1))


def test_direct_flags(ctx, oracle):
    n, k = 50000, 20001
    A, R = W.payload(8, n, seed=7), torch.sort(W.uniform_removals(n, k, seed=8)).values.contiguous()
    cfg = rz.TileConfig(512, 2, 0, 7, 0, 1)
    want = expected_canonical(oracle, A.numpy(), R.numpy())
    sz = n - k
    dead = np.zeros(k, bool)
    dead[R.numpy()[R.numpy() >= sz] - sz] = True
    for flags in (0, rz.RZ_PRESERVE_REMOVALS, rz.RZ_SORTED, rz.RZ_VALIDATE | rz.RZ_SORTED, rz.RZ_ANY_PAIRING,
                  rz.RZ_STATS, rz.RZ_PROFILE, rz.RZ_COOPERATIVE):
        announce("direct flags", flags)
        _, dR = gpu_remove_parity(ctx, oracle, A, R, config=cfg, flags=flags, want=want)
        if flags & rz.RZ_PRESERVE_REMOVALS:
            assert torch.equal(dR.cpu(), R)
        if flags & rz.RZ_STATS:
            st = ctx.last_stats()
            assert st.tail_removals == int(dead.sum())
            assert st.orphan_pairs == int((dead & (R.numpy() < sz)).sum())
    dup = R.clone()
    dup[0] = dup[k - 1]  # the last tail item twice: one source more than holes
    dA, dR = A.cuda(), dup.cuda()
    announce("direct mismatch")
    with pytest.raises(rz.RedzoneError):
        ctx.remove(dA, dR, config=cfg, flags=rz.RZ_STATS)
    gpu_remove_parity(ctx, oracle, A, R, config=cfg, want=want)
    announce("direct premarked")
    bits = torch.zeros((k + 31) // 32, dtype=torch.int32, device="cuda")
    dA, dR = A.cuda(), R.cuda()
    ctx.mark_removals(dR, n, bits)
    ctx.remove_premarked(dA, dR, bits, config=cfg)
    assert first_mismatch(dA.cpu().numpy()[:sz], want[:sz]) < 0 and int(bits.abs().sum()) == 0
    for bad in (rz.TileConfig(1024, 4, 0, 7, 0, 1), rz.TileConfig(256, 8, 0, 7, 0, 1), rz.TileConfig(128, 1, 0, 7, 0, 1)):
        with pytest.raises(rz.RedzoneError):
            ctx.remove(dA, dR, config=bad)


@pytest.mark.parametrize("k", [1, 97, 5000, 20001])
def test_direct_stages(ctx, oracle, k):
    """RZ_PROFILE on small removals through the tuned table: the slices' timeline,
    without the stages that the direct form does not have."""
    n = 3 * k + 40
    A, R = W.payload(4, n, seed=k), W.uniform_removals(n, k, seed=k + 1)
    announce("direct stages", k)
    gpu_remove_parity(ctx, oracle, A, R, flags=rz.RZ_PROFILE)
    st = ctx.last_stages()
    assert st["slices"] == (k + 511) // 512 and st["mark_groups"] == 0
    assert 0 <= st["first_slice_start"] <= st["last_slice_start"]
    assert 0 < st["lookback_end"] <= st["moves_end"] <= st["exit"] < 10_000
    assert st["marks_done"] == st["ready_raised"] == st["ready_wait_end"] == st["exchange_end"] == 0


@pytest.mark.parametrize("esz", [4, 8, 16])
@pytest.mark.parametrize("k,variant", [(300, 7), (5000, 7), (70001, 6), (70001, 4), (70001, 0)])
def test_add_remove_sources(oracle, esz, k, variant):
    """Added items read where the caller has them (fused and direct forms) or
    copied first (the others; unaligned items; items inside the list)."""
    ctx = rz.Context(0)
    b = k.bit_length() - 1
    ctx.set_table(esz, b, rz.TileConfig(256, 4, 512, variant, 12 if variant == 6 else 0, 1))
    n = 3 * k + 17
    for g in (1, k // 2, k, k + 1, 2 * k):
        m = n + g
        full = W.payload(esz, m, seed=g)
        R = W.uniform_removals(m, k, seed=g + 1)
        want = expected_canonical(oracle, full.numpy(), R.numpy())
        announce("add sources", esz, k, variant, g)
        cap = torch.zeros((m + 3,) + tuple(full.shape[1:]), dtype=torch.int32, device="cuda")
        cap[:n] = full[:n].cuda()
        guard = cap[m:].clone()
        add = full[n:].cuda()
        assert ctx.add_remove(cap, n, add, R.cuda()) == m - k
        assert first_mismatch(cap[: m - k].cpu().numpy(), want[: m - k]) < 0
        assert torch.equal(cap[m:], guard)
        if esz > 4:  # items at an address the kernels cannot load them from
            raw = torch.empty(add.numel() + 1, dtype=torch.int32, device="cuda")
            off = raw[1:].view(add.shape)
            off.copy_(add)
            cap[:n] = full[:n].cuda()
            assert ctx.add_remove(cap, n, off, R.cuda()) == m - k
            assert first_mismatch(cap[: m - k].cpu().numpy(), want[: m - k]) < 0
        if g <= n:  # the added items are a part of the list itself
            cap[:n] = full[:n].cuda()
            src = full.clone()
            src[n:] = full[:g]
            want2 = expected_canonical(oracle, src.numpy(), R.numpy())
            assert ctx.add_remove(cap, n, cap[:g], R.cuda()) == m - k
            assert first_mismatch(cap[: m - k].cpu().numpy(), want2[: m - k]) < 0
    assert ctx.check_errors() == 0
    ctx.close()


@pytest.mark.parametrize("k", [500, 40000])
@pytest.mark.parametrize("share", [0.4, 1, 2.5])
@pytest.mark.parametrize("bad", ["duplicate", "range"])
def test_add_remove_refused(oracle, k, share, bad):
    """Removals that RZ_VALIDATE refuses: the added items are in the list behind the
    others, and the corrected removals work on them."""
    ctx = rz.Context(0)
    n, g = 3 * k, int(share * k)
    m = n + g
    full, R = W.payload(8, m, seed=31), W.uniform_removals(m, k, seed=32)
    cap = torch.zeros((m, 2), dtype=torch.int32, device="cuda")
    cap[:n] = full[:n].cuda()
    wrong = R.clone()
    wrong[k // 2] = m if bad == "range" else wrong[3]
    announce("add refused", k, share, bad)
    with pytest.raises(rz.RedzoneError) as e:
        ctx.add_remove(cap, n, full[n:].cuda(), wrong.cuda(), flags=rz.RZ_VALIDATE)
    assert e.value.status == (2 if bad == "range" else 3)
    assert torch.equal(cap.cpu(), full)
    want = expected_canonical(oracle, full.numpy(), R.numpy())
    assert ctx.remove(cap, R.cuda(), flags=rz.RZ_VALIDATE) == m - k
    assert first_mismatch(cap[: m - k].cpu().numpy(), want[: m - k]) < 0
    ctx.close()


@pytest.mark.parametrize("esz", [4, 8, 16])
@pytest.mark.parametrize("p", [1, 1000, 8192, 8193, 64 * 8192, 64 * 8192 + 1, 65 * 4096 + 3, (1 << 22) + 17])
def test_gather_tiles(ctx, esz, p):
    """The one-pass gather's tiles and its search for the tiles that read from
    a tile's outputs: kept items in one run at the end, behind a gap, in runs,
    spread out, and dense at first then sparse (so that the guessed position is
    wrong), in one context with calls of both tile sizes."""
    keep = {"run at the end": torch.arange(p) + p // 2,
            "gap": torch.cat([torch.arange(p // 2), torch.arange(p // 2, p) + p // 3 + 5]),
            "spread": torch.arange(p) * 3 + 1,
            "sparse then dense": torch.cat([torch.arange(p // 8) * 30, p // 8 * 30 + torch.arange(p - p // 8)]),
            "dense then sparse": torch.cat([torch.arange(p - p // 8), p - p // 8 + torch.arange(p // 8) * 30]),
            "all": torch.arange(p)}
    for name, P in keep.items():
        n = int(P[-1]) + 1
        if p * 8 < n or n * esz > 1 << 28:
            continue
        announce("gather tiles", esz, p, name)
        A = torch.empty((n,) if esz == 4 else (n, esz // 4), dtype=torch.int32, device="cuda")
        ctx.gen_payload(A, p)
        want = A[P.cuda()].clone()
        assert ctx.gather_preserve(A, P.to(torch.int32).cuda(), n=n) == p
        assert torch.equal(A[:p], want)
    assert ctx.check_errors() == 0


@pytest.mark.parametrize("n,p", [(4000000, 3499999), (4000000, 3500000), (22000000, 3000000), (22000001, 3000000),
                                 ((1 << 27) + 3, 3 << 23)])
def test_gather_forms(ctx, n, p):
    """4-byte gathers at the edges of the band that takes two passes, and a large
    sparse one whose tiles follow each other."""
    announce("gather forms", n, p)
    A = torch.empty(n, dtype=torch.int32, device="cuda")
    ctx.gen_payload(A, p)
    R = torch.empty(p, dtype=torch.int32, device="cuda")
    ctx.gen_uniform_removals(R, n, p + 1)
    P = torch.sort(R).values.contiguous()
    want = A[P.long()]
    rest = A[p:].clone()
    assert ctx.gather_preserve(A, P) == p
    assert torch.equal(A[:p], want) and torch.equal(A[p:], rest)
    assert ctx.check_errors() == 0


@pytest.mark.parametrize("given", [False, True])
def test_calls_run_on_the_stream_they_name(ctx, given):
    """The caller's current stream, or the stream it passes, on every call (not
    only the first): the list is filled on that stream right before."""
    n, k = 60000, 700
    s = torch.cuda.Stream()
    R = torch.arange(5, 5 + k, dtype=torch.int32, device="cuda")
    new = torch.arange(n, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    for _ in range(3):
        data = torch.empty_like(new)
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            data.copy_(new)
            if not given:
                assert ctx.remove(data, R, flags=rz.RZ_PRESERVE_REMOVALS) == n - k
        if given:
            assert ctx.remove(data, R, flags=rz.RZ_PRESERVE_REMOVALS, stream=s) == n - k
        s.synchronize()
        got = data[: n - k].cpu()
        assert torch.equal(got.sort().values, torch.cat([new[:5], new[5 + k:]]).cpu())


def test_tensors_that_are_refused(ctx):
    data = torch.zeros(64, dtype=torch.int32, device="cuda")
    R = torch.zeros(4, dtype=torch.int32, device="cuda")
    for bad in ((data.cpu(), R), (data, R.cpu()), (data[::2], R), (data, R.long()), (data, R[::2]), (data, R.float())):
        with pytest.raises(ValueError):
            ctx.remove(*bad)
    with pytest.raises(ValueError):
        ctx.remove(data, R, k=5)
    with pytest.raises(ValueError):
        ctx.remove(data, R, n=65)
    with pytest.raises(ValueError):
        ctx.add_remove(data, 60, R, R.long())
    torch.cuda.synchronize()
