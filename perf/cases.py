"""Measured cases: sorted-set intersection as a user's program calls it, on one GPU.

Each family stands for one way the library is used (the comment at its entry in ``listed`` says
which), over the sizes the repository's own benchmark, generators and tests use: pairs of 2^6 to
2^18 elements, size ratios of 1 to 4,096, plain and BSR sets, uint32 and int32 elements, results
written or only counted.  ``draw`` gives further cases from the same ranges.
"""
import ctypes
import math

import numpy as np
import torch

DEV = "cuda"
KSET_WORDS = 1 << 22  # result words a request loop's slot holds


def listed():
    return [
        # one small pair from host memory: the per-pair drop-in of a harness that times int32 sets
        # of a datafile; latency and launches are all of it
        dict(name="host_pair", kind="host_pair", entry="hip_branchless_merge", na=1000, nb=1300, signed=True),
        # one k-set query from host memory, sizes 2^18 / (i + 1) as the k-set generator plans them
        dict(name="host_kset", kind="host_kset", entry="hip_branchless_merge", k=5, size=1 << 18),
        # one pair whose sets are on the device already: 2^16 against 2^16 over 2^20
        dict(name="dev_pair", kind="dev_pair", entry="hip_branchless_merge", na=1 << 16, nb=1 << 16, signed=False),
        # a small batch of uneven int32 pairs (one datafile's worth), results written
        dict(name="batch_small", kind="batch", entry="hip_branchless_merge", pairs=601, lmin=6.0, lmax=14.0, skew=10.0,
             signed=True, count_only=False, bsr=False),
        # the batched workload: 65,536 uneven pairs, compacted results, offsets and counts
        dict(name="batch_uneven", kind="batch", entry="hip_branchless_merge", pairs=65536, lmin=6.0, lmax=14.0,
             skew=10.0, signed=False, count_only=False, bsr=False),
        # similarity counts: the same kind of pairs, only counted
        dict(name="batch_count", kind="batch", entry="hip_branchless_merge", pairs=40001, lmin=6.0, lmax=14.0,
             skew=10.0, signed=False, count_only=True, bsr=False),
        # the same kind of pairs as base and state words, results written
        dict(name="batch_bsr", kind="batch", entry="hip_branchless_merge_bsr", pairs=65536, lmin=6.0, lmax=14.0,
             skew=10.0, signed=False, count_only=False, bsr=True),
        # a resident, indexed set of 2^24 against 4,096 small ones; the entry from the tuning table
        dict(name="resident", kind="resident", entry="hip_auto", large=1 << 24, sets=4096, small=256),
        # strongly skewed pairs, each with its own larger set: the galloping entry, no index
        dict(name="gallop", kind="batch", entry="hip_galloping", pairs=3000, lmin=12.0, lmax=16.0, skew=12.0,
             signed=False, count_only=False, bsr=False),
        # one step of a request loop: new k-set queries over an indexed corpus, results copied back
        dict(name="kset_step", kind="kset_step", entry="hip_galloping", lists=12000, queries=200),
        # neighbour intersections of every edge of an R-MAT graph, counted, one merge entry
        dict(name="graph_merge", kind="graph", scale=16, split=False),
        # the same on a larger graph as the graph module splits it: skewed edges to the indexed search entry
        dict(name="graph_split", kind="graph", scale=17, split=True),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["host_pair", "host_kset", "dev_pair", "batch", "batch", "batch", "resident", "gallop",
                       "kset_step", "graph"])
    if kind in ("host_pair", "dev_pair"):
        return dict(kind=kind, entry="hip_branchless_merge", na=_log_int(rng, 1 << 6, 1 << 17),
                    nb=_log_int(rng, 1 << 6, 1 << 17), signed=rng.random() < 0.5)
    if kind == "host_kset":
        return dict(kind=kind, entry=rng.choice(["hip_branchless_merge", "hip_galloping", "hip_small_adaptive"]),
                    k=rng.randint(3, 8), size=_log_int(rng, 1 << 12, 1 << 18))
    if kind == "batch":
        bsr = rng.random() < 0.3
        skew, most = rng.choice([(0.0, 30000), (3.0, 45000), (6.0, 55000), (10.0, 60000)])
        return dict(kind="batch", entry="hip_branchless_merge_bsr" if bsr else "hip_branchless_merge",
                    pairs=_log_int(rng, 60, most), lmin=6.0, lmax=14.0, skew=skew,
                    signed=(not bsr) and rng.random() < 0.4, count_only=rng.random() < 0.35, bsr=bsr)
    if kind == "gallop":
        return dict(kind="batch", entry=rng.choice(["hip_galloping", "hip_binary_search"]), pairs=_log_int(rng, 40, 3000),
                    lmin=12.0, lmax=16.0, skew=12.0, signed=rng.random() < 0.4, count_only=rng.random() < 0.35,
                    bsr=False)
    if kind == "resident":
        return dict(kind=kind, entry="hip_auto", large=_log_int(rng, 1 << 20, 1 << 24), sets=_log_int(rng, 100, 4096),
                    small=_log_int(rng, 16, 256))
    if kind == "kset_step":
        return dict(kind=kind, entry="hip_galloping", lists=_log_int(rng, 3000, 12000), queries=_log_int(rng, 3, 1000))
    return dict(kind="graph", scale=rng.randint(12, 16), split=rng.random() < 0.5)


# ---- inputs ------------------------------------------------------------------------------------


def _planted(gen, na, nb, ns, gap):
    """Pairs of sorted sets as (A, a_off, B, b_off): pair p draws about na + nb - ns values with the
    mean distance gap, each in A, in B or (about ns of them) in both."""
    nu = (na + nb - ns).to(torch.int64).clamp_(min=1)
    end = torch.cumsum(nu, 0)
    pid = torch.repeat_interleave(torch.arange(nu.numel(), device=DEV), nu)
    n = pid.numel()
    v = torch.rand(n, device=DEV, generator=gen)
    v = torch.log1p(-v).neg_().mul_((gap - 1).clamp_(min=0).to(torch.float32)[pid])
    v = torch.cumsum(v.to(torch.int64).add_(1), 0)
    base = torch.cat([v.new_zeros(1), v[end[:-1] - 1]])
    v = (v - base[pid]).to(torch.int32)
    r = torch.rand(n, device=DEV, generator=gen)
    in_b = r < (nb / nu).to(torch.float32)[pid]
    in_a = r >= (1 - na / nu).to(torch.float32)[pid]
    sets = []
    for m in (in_a, in_b):
        off = torch.zeros(nu.numel() + 1, dtype=torch.int64, device=DEV)
        off[1:] = torch.cumsum(m, 0)[end - 1]
        sets += [v[m], off]
    return sets


def _bsr(v, off):
    """Base and state words of the sets v[off[p] .. off[p+1])."""
    lens = off[1:] - off[:-1]
    pid = torch.repeat_interleave(torch.arange(lens.numel(), device=DEV), lens)
    base = v >> 5
    new = torch.ones(v.numel(), dtype=torch.bool, device=DEV)
    new[1:] = (base[1:] != base[:-1]) | (pid[1:] != pid[:-1])
    bits = torch.cumsum(torch.ones((), dtype=torch.int64, device=DEV) << (v & 31).to(torch.int64), 0)
    last = torch.cat([torch.nonzero(new).flatten()[1:] - 1, torch.tensor([v.numel() - 1], device=DEV)])
    upto = bits[last]
    states = upto - torch.cat([upto.new_zeros(1), upto[:-1]])
    states = torch.where(states >= 1 << 31, states - (1 << 32), states).to(torch.int32)
    words = torch.zeros(lens.numel() + 1, dtype=torch.int64, device=DEV)
    words[1:] = torch.cumsum(torch.bincount(pid[new], minlength=lens.numel()), 0)
    return base[new].contiguous(), states, words


def _pair_sizes(case, seed):
    g = torch.Generator().manual_seed(seed)
    p = case["pairs"]
    larger = torch.floor(2.0 ** (case["lmin"] + (case["lmax"] - case["lmin"]) * torch.rand(p, generator=g, dtype=torch.float64)))
    smaller = torch.floor(larger / 2.0 ** (case["skew"] * torch.rand(p, generator=g, dtype=torch.float64))).clamp_(min=1)
    shared = torch.round(smaller * torch.rand(p, generator=g, dtype=torch.float64))
    return smaller.to(DEV), larger.to(DEV), shared.to(DEV)


def _mean_sizes(case):
    """Mean sizes of a pair's smaller and larger set."""
    lo, hi, s = case["lmin"], case["lmax"], case["skew"] * math.log(2)
    larger = (2.0 ** hi - 2.0 ** lo) / ((hi - lo) * math.log(2))
    return larger * ((1 - math.exp(-s)) / s if s else 1.0), larger


def _clear(batch, room=None):
    """Outputs start as zeros, so that what lies behind the results is defined; with `room`, the
    results go to buffers of that many words, kept for batches of such sizes."""
    if room is not None:
        if room < batch.capacity:
            raise ValueError("the output buffers are too small")
        batch.d_out = torch.zeros(room, dtype=torch.int32, device=DEV)
        batch.d_out_s = torch.zeros(room, dtype=torch.int32, device=DEV) if batch.bsr else None
    for t in (batch.d_out, batch.d_out_s, batch.d_out_off, batch.d_counts, batch.d_totals):
        if t is not None:
            t.zero_()


def _prepare_batch(case, seed):
    from simd_set_operations_amd.batch import DeviceBatch

    gen = torch.Generator(device=DEV).manual_seed(seed)
    na, nb, ns = _pair_sizes(case, seed)
    gap = 10 * nb / (na + nb - ns).clamp(min=1)
    A, a_off, B, b_off = _planted(gen, na, nb, ns, gap)
    As = Bs = None
    if case["bsr"]:
        A, As, a_off = _bsr(A, a_off)
        B, Bs, b_off = _bsr(B, b_off)
    if case["signed"]:
        # each pair's values spread to both sides of zero
        for v, off in ((A, a_off), (B, b_off)):
            v -= torch.repeat_interleave((5 * nb).to(torch.int32), off[1:] - off[:-1])
    db = DeviceBatch(case["entry"], A, a_off.cpu().numpy(), B, b_off.cpu().numpy(), A_states=As, B_states=Bs,
                     signed=case["signed"])
    _clear(db, None if case["count_only"] else int(2 * case["pairs"] * _mean_sizes(case)[0] + 4 * 2.0 ** case["lmax"]))
    return dict(kind="batch", batch=db, count_only=case["count_only"])


def _host_sets(seed, sizes, universe, shared):
    """Sorted unique int32 sets over {0 .. universe - 1} with `shared` common elements."""
    rng = np.random.default_rng(seed)
    common = rng.choice(universe, shared, replace=False)
    out = []
    for n in sizes:
        more = rng.integers(0, universe, 2 * n + 64)
        more = np.setdiff1d(more, common)
        rng.shuffle(more)
        out.append(np.sort(np.concatenate([common, more[:n - shared]])))
    return out


def _prepare_pair(case, seed):
    from simd_set_operations_amd import intersect

    na, nb = case["na"], case["nb"]
    a, b = _host_sets(seed, (na, nb), 16 * max(na, nb), int(0.3 * min(na, nb)))
    if case["signed"]:
        a, b = ((x - 8 * max(na, nb)).astype(np.int32) for x in (a, b))
    else:
        a, b = (x.astype(np.uint32) for x in (a, b))
    intersect.init(0)
    cap = min(a.size, b.size)
    if case["kind"] == "host_pair":
        return dict(kind="host_pair", entry=case["entry"], a=a, b=b, out=np.zeros(cap, a.dtype))
    from simd_set_operations_amd import _native

    algo = intersect.algo_id(case["entry"]) | (_native.SIGNED_I32 if case["signed"] else 0)
    return dict(kind="dev_pair", algo=algo, a=torch.from_numpy(a.view(np.int32)).to(DEV),
                b=torch.from_numpy(b.view(np.int32)).to(DEV), out=torch.zeros(cap, dtype=torch.int32, device=DEV),
                totals=torch.zeros(2, dtype=torch.int64, device=DEV))


def _prepare_host_kset(case, seed):
    from simd_set_operations_amd import intersect

    intersect.init(0)
    sizes = [max(8, case["size"] // (i + 1)) for i in range(case["k"])][::-1]
    sets = _host_sets(seed, sizes, 100 * case["size"], max(1, sizes[0] // 10))
    return dict(kind="host_kset", entry=case["entry"], sets=[s.astype(np.uint32) for s in sets])


def _prepare_resident(case, seed):
    from simd_set_operations_amd.batch import GatherBatch

    gen = torch.Generator(device=DEV).manual_seed(seed)
    large, sets, small = case["large"], case["sets"], case["small"]
    gaps = torch.log1p(-torch.rand(large, device=DEV, generator=gen)).mul_(-15.0).to(torch.int64).add_(1)
    L = torch.cumsum(gaps, 0)
    # one value of each of `small` equal parts of the large set: a tenth of them members, the rest
    # between two members
    part = torch.arange(small, device=DEV).to(torch.float64) + torch.rand(sets, small, device=DEV, generator=gen,
                                                                        dtype=torch.float64)
    i = (part * (large / small)).to(torch.int64).clamp_(max=large - 2)
    between = (torch.rand(sets, small, device=DEV, generator=gen) * (gaps[i + 1] - 1)).to(torch.int64).add_(1)
    between.clamp_(max=gaps[i + 1] - 1)
    member = torch.rand(sets, small, device=DEV, generator=gen) < 0.1
    S = torch.where(member, L[i], L[i] + between).to(torch.int32).flatten().contiguous()
    beg = np.arange(sets, dtype=np.uint64) * np.uint64(small)
    gb = GatherBatch(case["entry"], S, beg, beg + np.uint64(small), L.to(torch.int32), np.zeros(sets, np.uint64),
                     np.full(sets, large, np.uint64), signed=False, index=True)
    _clear(gb)
    return dict(kind="batch", batch=gb, count_only=False)


def _prepare_kset_step(case, seed):
    from simd_set_operations_amd import _native
    from simd_set_operations_amd.intersect import algo_id, init
    from simd_set_operations_amd.serving import Corpus, make_queries

    init(0)
    lib = _native.hip()
    c = Corpus(nlists=case["lists"], seed=seed)
    nq = case["queries"]
    ids, ks = make_queries(c, nq, seed=seed + 1)
    one = torch.zeros(4, dtype=torch.int64, device=DEV)
    h = ctypes.c_void_p()
    _native.check(lib.setops_hip_batch_create_gather(
        ctypes.byref(h), algo_id(case["entry"]), c.pool.data_ptr(), None, c.pool.numel(), one.data_ptr(),
        one.data_ptr() + 8, c.pool.data_ptr(), None, c.pool.numel(), one.data_ptr() + 16, one.data_ptr() + 24, 1))
    na, nb = c.lens[ids[:, 0]], c.lens[ids[:, 1]]
    need = int(na.sum())
    if need + 64 > KSET_WORDS:
        raise ValueError("the result buffers are too small")
    _native.check(lib.setops_hip_batch_reserve(h, nq, need))
    _native.check(lib.setops_hip_batch_index_b(h))
    # the step's rows: pair bounds, further-set offsets and bounds
    further = np.array([i for q in range(nq) for i in ids[q, 2:ks[q]]], np.int64)
    xoff = np.concatenate([[0], np.cumsum(ks - 2)])
    rows = np.concatenate([c.beg[ids[:, 0]], c.beg[ids[:, 0]] + na, c.beg[ids[:, 1]], c.beg[ids[:, 1]] + nb,
                           xoff.astype(np.uint64), c.beg[further], c.beg[further] + c.lens[further]])
    rows = rows.astype(np.uint64).view(np.int64)
    return dict(kind="kset_step", lib=lib, handle=_Handle(lib, h), corpus=c, nq=nq, nx=further.size,
                na=np.ascontiguousarray(na, np.uint64), nb=np.ascontiguousarray(nb, np.uint64), words=need + 64,
                h_idx=torch.from_numpy(rows).pin_memory(), d_idx=torch.zeros(rows.size, dtype=torch.int64, device=DEV),
                out=torch.zeros(KSET_WORDS, dtype=torch.int32, device=DEV),
                off=torch.zeros(nq + 1, dtype=torch.int64, device=DEV),
                counts=torch.zeros(nq, dtype=torch.int32, device=DEV),
                totals=torch.zeros(2, dtype=torch.int64, device=DEV),
                h_off=torch.zeros(nq + 1, dtype=torch.int64).pin_memory(),
                h_out=torch.zeros(KSET_WORDS, dtype=torch.int32).pin_memory())


class _Handle:
    """A batch handle that goes with its state."""

    def __init__(self, lib, h):
        self.lib, self.h = lib, h

    def __del__(self):
        self.lib.setops_hip_batch_destroy(self.h)


def _prepare_graph(case, seed):
    from simd_set_operations_amd import tuning
    from simd_set_operations_amd.graph import EdgeIntersections, split_by_skew

    gen = torch.Generator(device=DEV).manual_seed(seed)
    n, m = 1 << case["scale"], 16 << case["scale"]
    u = torch.zeros(m, dtype=torch.int64, device=DEV)
    v = torch.zeros(m, dtype=torch.int64, device=DEV)
    for _ in range(case["scale"]):
        # R-MAT quadrants 0.57, 0.19, 0.19, 0.05
        r = torch.rand(m, device=DEV, generator=gen)
        u = 2 * u + (r >= 0.76)
        v = 2 * v + (((r >= 0.57) & (r < 0.76)) | (r >= 0.95))
    keep = u != v
    u, v = u[keep], v[keep]
    # undirected edges without repeats, as many as every draw of this size has
    key = torch.unique(torch.minimum(u, v) * n + torch.maximum(u, v))
    key = key[torch.randperm(key.numel(), device=DEV, generator=gen)[:10 << case["scale"]]]
    u, v = key // n, key % n
    key = torch.sort(torch.cat([key, v * n + u])).values
    src, col = key // n, (key % n).to(torch.int32)
    rowptr = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    rowptr[1:] = torch.cumsum(torch.bincount(src, minlength=n), 0)
    rp = rowptr.cpu().numpy().astype(np.uint64)
    fwd = src < col
    eu, ev = src[fwd].cpu().numpy(), col[fwd].cpu().numpy().astype(np.int64)
    beg, end = rp[:-1], rp[1:]
    if not case["split"]:
        parts = [EdgeIntersections("hip_branchless_merge", col, beg, end, eu, ev)]
    else:
        deg = end - beg
        skewed = split_by_skew(deg[eu], deg[ev], tuning.graph_split_threshold())
        parts = [EdgeIntersections("hip_branchless_merge", col, beg, end, eu, ev, select=~skewed),
                 EdgeIntersections("hip_galloping", col, beg, end, eu, ev, select=skewed, index=True)]
    # one count per edge and one offset per edge (and one past each part's last), over all parts
    parts = [p for p in parts if p.batch is not None]
    counts = torch.zeros(eu.size, dtype=torch.int32, device=DEV)
    off = torch.zeros(eu.size + 2, dtype=torch.int64, device=DEV)
    totals = torch.zeros(2, 2, dtype=torch.int64, device=DEV)
    at = 0
    for k, p in enumerate(parts):
        p.batch.d_counts = counts[at:at + p.pairs]
        p.batch.d_out_off = off[at + k:at + k + p.pairs + 1]
        p.batch.d_totals = totals[k]
        at += p.pairs
    return dict(kind="graph", parts=parts, outputs=[off, counts, totals])


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        return _prepare_batch(case, seed)
    if kind in ("host_pair", "dev_pair"):
        return _prepare_pair(case, seed)
    if kind == "host_kset":
        return _prepare_host_kset(case, seed)
    if kind == "resident":
        return _prepare_resident(case, seed)
    if kind == "kset_step":
        return _prepare_kset_step(case, seed)
    return _prepare_graph(case, seed)


# ---- one pass ------------------------------------------------------------------------------------


def _outputs(batch, count_only):
    if count_only:
        return [batch.d_out_off, batch.d_counts, batch.d_totals]
    return [batch.d_out, batch.d_out_off, batch.d_counts, batch.d_totals] + ([batch.d_out_s] if batch.bsr else [])


def run(state):
    kind = state["kind"]
    if kind == "batch":
        state["batch"].run(count_only=state["count_only"])
        return _outputs(state["batch"], state["count_only"])
    if kind == "graph":
        for p in state["parts"]:
            p.run()
        return state["outputs"]
    if kind == "kset_step":
        from simd_set_operations_amd import _native

        s = state
        _native.check(s["lib"].setops_hip_batch_step(
            s["handle"].h, s["h_idx"].data_ptr(), s["d_idx"].data_ptr(), s["nq"], s["nx"], s["na"].ctypes.data,
            s["nb"].ctypes.data, s["out"].data_ptr(), KSET_WORDS, s["off"].data_ptr(), s["counts"].data_ptr(),
            s["totals"].data_ptr(), s["h_off"].data_ptr(), s["h_out"].data_ptr(), s["words"],
            torch.cuda.current_stream().cuda_stream))
        return [s["h_off"], s["h_out"], s["counts"], s["totals"]]
    from simd_set_operations_amd import intersect

    if kind == "host_pair":
        n = intersect.intersect2_c(state["entry"], state["a"], state["b"], state["out"])
        return [state["out"], n]
    if kind == "host_kset":
        return intersect.run_kset(state["sets"], state["entry"])
    from simd_set_operations_amd import _native

    a, b, out = state["a"], state["b"], state["out"]
    _native.check(_native.hip().setops_hip_intersect2_dev(
        state["algo"], a.data_ptr(), None, a.numel(), b.data_ptr(), None, b.numel(), out.data_ptr(), None, out.numel(),
        state["totals"].data_ptr(), torch.cuda.current_stream().cuda_stream))
    return [out, state["totals"]]


# ---- what a pass cannot do without -----------------------------------------------------------------


def work(case):
    """Bytes: every input element read once (of a searched larger set, the 128-byte lines its probes
    end in, where those are fewer), every result, offset and count written once."""
    kind = case["kind"]
    if kind in ("host_pair", "dev_pair"):
        return dict(bytes=4 * (case["na"] + case["nb"]) + 4 * 0.3 * min(case["na"], case["nb"]) + 16, flops=0)
    if kind == "host_kset":
        sizes = [max(8, case["size"] // (i + 1)) for i in range(case["k"])]
        return dict(bytes=4 * sum(sizes) + 0.4 * min(sizes), flops=0)
    if kind == "batch":
        p = case["pairs"]
        smaller, larger = _mean_sizes(case)
        if case["bsr"]:
            # a tenth of the element space: about three elements of the larger set share a word
            larger, smaller, each = 0.302 * larger, 0.75 * smaller, 8
        else:
            each = 4
        if "merge" not in case["entry"]:
            larger = min(larger, 32 * smaller)
        found = 0 if case["count_only"] else 0.5 * smaller
        return dict(bytes=p * (each * (larger + smaller + found) + 28), flops=0)
    if kind == "resident":
        probes = case["sets"] * case["small"]
        return dict(bytes=4 * probes + min(4 * case["large"], 128 * probes) + 0.4 * probes + 44 * case["sets"], flops=0)
    if kind == "kset_step":
        # a query's smallest list has about 750 elements
        return dict(bytes=case["queries"] * (750 * (4 + 128) + 100), flops=0)
    # graph: the neighbour lists once, each edge's bounds, count and offset
    edges = 10 << case["scale"]
    return dict(bytes=8 * edges + 44 * edges, flops=0)
