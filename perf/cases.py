"""Performance cases: what programs that use redzone_amd have it do.

Every pass is one step of a program in a steady state, so it can be repeated
on the same buffers.  A removal leaves the end of the list free, and the
program fills that end with new items before the next removal: through
Context.add_remove, or with a copy of its own ("arrivals") before
Context.remove, remove_auto, partition and the batch.  A pass's result then
depends only on the inputs and never on what the library left in the scratch
part of a list.  The program keeps its removal list (RZ_PRESERVE_REMOVALS), for
instance to free the removed items' handles.

Outputs are the survivors, moved bit for bit, so they have no rounding and
exact() has nothing to add for them; only the dispatch network's training
gradient is computed, and exact() gives it in float64.
"""
import math

import numpy as np
import torch

import redzone_amd as rz
from redzone_amd import workloads as W
from redzone_amd.dispatch import NC, NF, NH, NP, Dispatcher, init_params

KEEP = rz.RZ_PRESERVE_REMOVALS


def listed():
    return [
        # one frame of a small particle system: 16-byte records, a few dozen
        # spawned and as many removed; the call's fixed cost is everything
        {"name": "frame_rec16_small", "kind": "add_remove", "elem_bytes": 16, "n": 4001, "k": 97,
         "pattern": "uniform"},
        # the small plain list: 2^20 4-byte items, 2^14 removals
        {"name": "remove_u32_2e20", "kind": "remove", "elem_bytes": 4, "n": 1 << 20, "k": 1 << 14,
         "pattern": "uniform"},
        # a mid-size list that loses a quarter of its 8-byte items: many removals
        # fall in the red zone, so marks and orphan pairs count as much as moves
        {"name": "remove_u64_quarter", "kind": "remove", "elem_bytes": 8, "n": 4200001, "k": 1050000,
         "pattern": "uniform"},
        # the headline: 1 GiB of 4-byte items, 1% removed at random
        {"name": "remove_u32_1pct", "kind": "remove", "elem_bytes": 4, "n": 1 << 28, "k": (1 << 28) // 100,
         "pattern": "uniform"},
        # a large simulation's frame: 16-byte records, 3% replaced, removals in runs
        {"name": "frame_rec16_runs", "kind": "add_remove", "elem_bytes": 16, "n": 30000007, "k": 900001,
         "pattern": "clustered"},
        # the densest removal for which Redzone is meant: half of a 1 GiB list
        {"name": "remove_u32_half", "kind": "remove", "elem_bytes": 4, "n": 1 << 28, "k": 1 << 27,
         "pattern": "uniform"},
        # survivors in their order: the stable partition of a 1 GiB list
        {"name": "partition_u32", "kind": "partition", "elem_bytes": 4, "n": (1 << 28) - 17, "k": 1 << 26,
         "pattern": "uniform"},
        # the same for a mid-size list of 16-byte records with removals towards the end
        {"name": "partition_rec16", "kind": "partition", "elem_bytes": 16, "n": 1500001, "k": 600000,
         "pattern": "tail_heavy"},
        # a program that knows the survivors instead: the in-place gather
        {"name": "gather_u64", "kind": "gather", "elem_bytes": 8, "n": 5000003, "p": 2000001},
        # thousands of independent lists in one planned launch (size classes of
        # a slab allocator, 2^8 to 2^20 items, up to 30% removed)
        {"name": "batch_u32_4096", "kind": "batch", "elem_bytes": 4, "lists": 4096, "classes": 32, "log2_min": 8.0,
         "log2_max": 20.0, "r_max": 0.3},
        # the method chosen per list by the learned dispatcher
        {"name": "auto_u64", "kind": "auto", "elem_bytes": 8, "n": 3000017, "k": 400001, "pattern": "uniform"},
        # one gradient of the dispatch network (forward and backward) on its training set's size
        {"name": "mlp_grad", "kind": "mlp_grad", "batch": 4000},
    ]


# kind -> (weight, smallest and largest bytes of the list) of a drawn case
_KINDS = (("add_remove", 3), ("remove", 4), ("partition", 2), ("gather", 2), ("batch", 1), ("auto", 1),
          ("mlp_grad", 1))


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choices([k for k, _ in _KINDS], [w for _, w in _KINDS])[0]
    if kind == "mlp_grad":
        return {"kind": kind, "batch": int(_log_uniform(rng, 32, 8000))}
    esz = rng.choice([4, 8, 16])
    if kind == "batch":
        return {"kind": kind, "elem_bytes": esz, "lists": int(_log_uniform(rng, 64, 4096)),
                "classes": rng.randint(8, 32), "log2_min": round(rng.uniform(6.0, 10.0), 2),
                "log2_max": round(rng.uniform(12.0, 18.0), 2), "r_max": round(rng.uniform(0.05, 0.6), 3)}
    if kind == "gather":
        n = int(_log_uniform(rng, 1 << 12, (1 << 28) // esz))
        return {"kind": kind, "elem_bytes": esz, "n": n, "p": max(1, int(n * rng.uniform(0.05, 0.99)))}
    pattern = rng.choice(["uniform", "uniform", "clustered", "tail_heavy"])
    # the clustered and tail-heavy generators hold several 8-byte words per position
    n = int(_log_uniform(rng, 1 << 12, ((1 << 30) if pattern == "uniform" else (1 << 27)) // esz))
    if kind == "partition":
        f = rng.uniform(0.01, 0.5)
    else:
        f = _log_uniform(rng, 1e-4, 0.4)
    return {"kind": kind, "elem_bytes": esz, "n": n, "k": max(1, int(n * f)), "pattern": pattern}


def _empty_items(rows, elem_bytes):
    shape = (rows,) if elem_bytes == 4 else (rows, elem_bytes // 4)
    return torch.empty(shape, dtype=torch.int32, device="cuda")


def _items(ctx, rows, elem_bytes, seed):
    """`rows` items; the first word of an item is a keyed bijection of its index (unique)."""
    A = _empty_items(rows, elem_bytes)
    ctx.gen_payload(A, seed)
    return A


def _removals(ctx, pattern, n, k, seed):
    if pattern == "uniform":
        R = torch.empty(k, dtype=torch.int32, device="cuda")
        ctx.gen_uniform_removals(R, n, seed)
        return R
    if pattern == "clustered":
        return W.clustered_removals(n, k, seed, mean=64, device="cuda")
    return W.tail_heavy_removals(n, k, seed, device="cuda")


def _batch_classes(case):
    """(n, k, lists) of every size class: n spread over the logarithm, k/n over [0, r_max)."""
    out = []
    c = case["classes"]
    for i in range(c):
        lists = case["lists"] // c + (1 if i < case["lists"] % c else 0)
        log2n = case["log2_min"] + (case["log2_max"] - case["log2_min"]) * (i + 0.5) / c
        n = int(2 ** log2n)
        if lists:
            out.append((n, int(n * case["r_max"] * ((0.618034 * (i + 1)) % 1.0)), lists))
    return out


def prepare(case, seed):
    ctx = rz.default_context(0)
    kind = case["kind"]
    s = {"kind": kind, "ctx": ctx}
    if kind == "mlp_grad":
        disp, X, T, M = _mlp_inputs(case, seed)
        s["disp"] = Dispatcher(ctx, params=disp)
        s["X"], s["T"], s["M"] = X.cuda(), T.cuda(), M.cuda()
        return s
    esz = case["elem_bytes"]
    if kind == "batch":
        s["heads"], s["tails"], s["arrivals"], lists = [], [], [], []
        for i, (n, k, m) in enumerate(_batch_classes(case)):
            arena = _items(ctx, m * n, esz, seed + 1000 * i).view((m, n) if esz == 4 else (m, n, esz // 4))
            R = torch.empty((m, max(1, k)), dtype=torch.int32, device="cuda")
            for j in range(m):
                if k:
                    ctx.gen_uniform_removals(R[j], n, seed + 7919 * i + 31 * j)
                    lists.append((arena[j], R[j]))
            s["heads"].append(arena[:, : n - k])
            if k:
                s["tails"].append(arena[:, n - k:])
                s["arrivals"].append(arena[:, n - k:].clone())
        s["batch"] = ctx.batch(lists, flags=KEEP)
        s["lists"] = lists
        return s
    n = case["n"]
    if kind == "gather":
        p = case["p"]
        s["data"] = _items(ctx, n, esz, seed)
        s["keep"] = torch.sort(_removals(ctx, "uniform", n, p, seed + 1)).values.contiguous()
        s["p"] = p
        return s
    k = case["k"]
    s["k"] = k
    if kind == "add_remove":
        s["n"] = n
        s["data"] = _items(ctx, n + k, esz, seed)  # capacity for the k items of a frame
        s["add"] = _items(ctx, k, esz, seed + 3)
        s["R"] = _removals(ctx, case["pattern"], n + k, k, seed + 1)
        return s
    s["n"] = n
    s["data"] = _items(ctx, n, esz, seed)
    s["tail"] = s["data"][n - k:]
    s["arrivals"] = s["tail"].clone()
    s["R"] = _removals(ctx, case["pattern"], n, k, seed + 1)
    return s


def run(s):
    kind, ctx = s["kind"], s["ctx"]
    if kind == "mlp_grad":
        loss, grad = s["disp"].grad(s["X"], s["T"], s["M"])
        return {"loss": loss, "grad": grad}
    if kind == "batch":
        for tail, arrivals in zip(s["tails"], s["arrivals"]):
            tail.copy_(arrivals)
        s["batch"].launch()
        return s["heads"]
    if kind == "gather":
        return s["data"][: ctx.gather_preserve(s["data"], s["keep"])]
    if kind == "add_remove":
        return s["data"][: ctx.add_remove(s["data"], s["n"], s["add"], s["R"], flags=KEEP)]
    s["tail"].copy_(s["arrivals"])
    if kind == "partition":
        return s["data"][: ctx.partition(s["data"], s["R"])]
    if kind == "auto":
        return s["data"][: ctx.remove_auto(s["data"], s["R"], flags=KEEP)[0]]
    return s["data"][: ctx.remove(s["data"], s["R"], flags=KEEP)]


def work(case):
    """Bytes and operations a pass cannot do without, the program's own copy of
    the arrivals not counted."""
    kind = case["kind"]
    if kind == "mlp_grad":
        b = case["batch"]
        # forward, and twice as much backward; the inputs, the parameters and the gradient once
        return {"bytes": 4 * (b * (NF + 2 * NC) + 2 * NP), "flops": 6 * b * NP}
    esz = case["elem_bytes"]
    if kind == "batch":
        total = 0
        for n, k, m in _batch_classes(case):
            total += m * _remove_bytes(esz, n, k)
        return {"bytes": total, "flops": 0}
    if kind == "gather":
        return {"bytes": (4 + 2 * esz) * case["p"], "flops": 0}
    n, k = case["n"], case["k"]
    if kind == "partition":
        return {"bytes": 4 * k + esz * n + esz * (n - k), "flops": 0}
    if kind == "add_remove":
        return {"bytes": _remove_bytes(esz, n + k, k), "flops": 0}
    return {"bytes": _remove_bytes(esz, n, k), "flops": 0}


def _remove_bytes(esz, n, k):
    """The removal list and the red zone read, the holes written (k^2/n removals fall in the red zone)."""
    return int(4 * k + esz * k + esz * (k - k * k / n)) if k else 0


# --------------------------------------------------------------------------
# the dispatch network
# --------------------------------------------------------------------------

def _mlp_inputs(case, seed):
    """Parameters as training starts them, features in the ranges of
    rz_features, targets log2 microseconds; one list in ten lacks a method's
    timing."""
    b = case["batch"]
    g = torch.Generator().manual_seed(seed)
    u = torch.rand((b, NF), generator=g)
    X = torch.empty((b, NF), dtype=torch.float32)
    log2n = 12 + 14 * u[:, 0]
    frac = 10 ** (-5 + 4.95 * u[:, 1])
    X[:, 0] = log2n / 32
    X[:, 1] = (log2n + torch.log2(frac)).clamp_min(0) / 32
    X[:, 2] = frac
    X[:, 3] = (torch.log2(frac) / 20).clamp_min(-1)
    X[:, 4] = 4.0 * 2 ** torch.floor(3 * u[:, 4]) / 16
    X[:, 5:11] = u[:, 5:11]
    X[:, 11] = 1
    T = 3 + 9 * torch.rand((b, NC), generator=g)
    M = (torch.rand((b, NC), generator=g) > 0.1).to(torch.float32)
    M[0] = 1
    return init_params(seed), X, T, M


def exact(case, seed):
    """The loss and the gradient in float64; the other cases move bits."""
    if case["kind"] != "mlp_grad":
        return None
    p, X, T, M = _mlp_inputs(case, seed)
    flat = torch.from_numpy(np.asarray(p, np.float64)).requires_grad_(True)
    h, at = X.double(), 0
    for nin, nout in ((NF, NH), (NH, NH), (NH, NH), (NH, NC)):
        w = flat[at: at + nin * nout].view(nout, nin)
        bias = flat[at + nin * nout: at + nin * nout + nout]
        at += nin * nout + nout
        h = h @ w.t() + bias
        if nout == NH:
            h = torch.relu(h)
    M = M.double()
    loss = (M * (h - T.double()) ** 2).sum() / M.sum()
    loss.backward()
    return {"loss": loss.detach().reshape(1), "grad": flat.grad}
