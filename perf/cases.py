"""What this framework's callers have it do, as measurable cases.

A case is a dict of plain values; `prepare` builds what a program holds
before the call (allocator, plan, tables, device inputs), `run` is one pass
through the package's entry points, and `work` is what that pass cannot do
without.  The sizes are those of bench.py's configurations and of the GPU
tests, and ragged ones around them.

Kinds:
  churn    the mixed malloc/free churn, every allocation filled and verified
           (`words` false) or one word of it written and checked (true); per
           thread as device code calls malloc and free, or in workgroup
           batches
  big      one step of whole-block and multi-segment requests
  stream   a batched request stream: captured plan, or one launch per batch
  table    insert, look up and remove a batch of keys on the growing hash table
  chain    build a chaining table from a batch, answer it, give it back
  queue    a batch through a FIFO: linked nodes, ring of queues or block nodes
  serving  one step of the session loop on the global allocator
"""
import numpy as np
import torch

import gallatin_amd as G
from gallatin_amd import serving
from gallatin_amd.batch_streams import lognormal_sizes

MIB, GIB = 1 << 20, 1 << 30
GLOBAL_BYTES = 80 * GIB  # the global allocator behind tables, chains and serving


def listed():
    return [
        # The headline workload: 2^24 request streams of ten rounds in
        # workgroup batches on an 8 GiB pool (one partition per XCD).
        dict(name="churn_batched", kind="churn", words=False, batched=True, pool_gib=8,
             n=1 << 24, rounds=10, threads=1024),
        # Device code that calls malloc and free per thread from a pool too
        # small for XCD partitions; a ragged thread count.
        dict(name="churn_thread_small_pool", kind="churn", words=False, batched=False,
             pool_gib=4, n=1_000_003, rounds=10, threads=256),
        # Per-thread malloc and free of the same sizes with one word used, the
        # allocator's own rate on a partitioned pool.
        dict(name="churn_word_thread", kind="churn", words=True, batched=False, pool_gib=8,
             n=1 << 22, rounds=10, threads=256),
        # The smallest call: a thousand threads, latency and launches.
        dict(name="churn_word_tiny", kind="churn", words=True, batched=False, pool_gib=1,
             n=1000, rounds=3, threads=256),
        # Large buffers: 64 KiB to 64 MiB and 256 MiB to 2 GiB, half the pool.
        dict(name="big_blocks", kind="big", pool_gib=48, n_small=576, n_large=5),
        # A stream of batches of very different sizes as one captured plan, at
        # the geometry the autotuner picks.
        dict(name="stream_plan", kind="stream", plan=True, batched=1, threads=1024,
             segment_mib=16, smallest=128, pool_gib=32, nbatches=256, max_count=1 << 19),
        # Small batches, one launch each, as a program that launches per batch.
        dict(name="stream_launches", kind="stream", plan=False, batched=0, threads=256,
             segment_mib=16, smallest=16, pool_gib=8, nbatches=100, max_count=4096),
        # A million keys through the large hash table, which holds as many
        # others: the rate of a key-value store's batch.
        dict(name="table_large", kind="table", large=True, held=1 << 20, n=1 << 20,
             absent=0.25),
        # A thousand keys through the small table: a request's latency.
        dict(name="table_small", kind="table", large=False, held=5000, n=1000, absent=0.5),
        # Grouping a batch of pairs by key and reading it back.
        dict(name="chain_build_query", kind="chain", layout=0, n=500_000, load=1.0,
             absent=0.25),
        # A batch of work items through a queue on an allocator.
        dict(name="queue_pass", kind="queue", form="linked", pool_gib=4, n=65_003),
        # One step of a serving loop at its steady number of sessions, with
        # table traffic beside the appends.
        dict(name="serving_step", kind="serving", sessions=16384, life=48, ht_ops=1 << 16),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(("churn", "churn", "churn", "big", "stream", "stream", "table", "table",
                       "chain", "queue", "serving"))
    if kind == "churn":
        batched = rng.random() < 0.5
        return dict(kind=kind, words=rng.random() < 0.5, batched=batched,
                    pool_gib=rng.choice((2, 4, 8, 16)), n=_log(rng, 1000, 1 << 23),
                    rounds=rng.randint(2, 10),
                    threads=rng.choice((512, 1024)) if batched else rng.choice((64, 256, 512)))
    if kind == "big":
        f = 0.1 + 0.9 * rng.random()
        return dict(kind=kind, pool_gib=48, n_small=int(576 * f), n_large=int(5 * f))
    if kind == "stream":
        plan = rng.random() < 0.5
        batched = rng.choice((0, 1, 2))
        return dict(kind=kind, plan=plan, batched=batched,
                    threads=rng.choice((256, 512, 1024)) if batched else 256,
                    segment_mib=rng.choice((16, 64)), smallest=rng.choice((16, 128)),
                    pool_gib=32, nbatches=_log(rng, 16, 256 if plan else 100),
                    max_count=_log(rng, 1024, 1 << 19) if plan else _log(rng, 256, 8192))
    if kind == "table":
        large = rng.random() < 0.5
        return dict(kind=kind, large=large, held=_log(rng, 1000, (1 << 20) if large else 200_000),
                    n=_log(rng, 200, (1 << 20) if large else 200_000),
                    absent=round(rng.random(), 2))
    if kind == "chain":
        return dict(kind=kind, layout=rng.randrange(5), n=_log(rng, 2000, 500_000),
                    load=rng.choice((0.5, 1.0, 2.0)), absent=round(rng.random(), 2))
    if kind == "queue":
        return dict(kind=kind, form=rng.choice(("linked", "ring", "block256", "block16")),
                    pool_gib=4, n=_log(rng, 300, 65_003))
    return dict(kind=kind, sessions=_log(rng, 1024, 16384), life=rng.randint(16, 48),
                ht_ops=_log(rng, 1 << 10, 1 << 16))


def _global():
    """The process's global allocator, made at its first use."""
    if not G.lib().gal_global_handle():
        G.init_global_allocator(GLOBAL_BYTES, 42, print_info=False)


class _Held:
    """Objects a program keeps between calls, given back together."""

    def __init__(self, **kw):
        self.__dict__.update(kw)

    def __del__(self):
        for name in ("plan", "table", "queue", "loop"):
            if name in self.__dict__:
                getattr(self, name).destroy()
        if "alloc" in self.__dict__:
            torch.cuda.synchronize()
            self.alloc.free_on_device()


def _cuda(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _distinct(rng, n, bits):
    """n distinct keys in [1, 2^bits]: an odd multiple of a random range."""
    start = int(rng.integers(1 << (bits - 1)))
    mult = int(rng.integers(1 << 40)) * 2 + 1
    k = (np.arange(n, dtype=np.uint64) + np.uint64(start)) * np.uint64(mult)
    return ((k & np.uint64((1 << bits) - 1)) + np.uint64(1)).astype(np.int64)


def _zipf_counts(nbatches, max_count, s=1.2):
    """The nbatches quantiles of Zipf(s) on [1, max_count]."""
    cdf = np.cumsum(np.arange(1, max_count + 1, dtype=np.float64) ** -s)
    return np.searchsorted(cdf / cdf[-1], (np.arange(nbatches) + 0.5) / nbatches) + 1


def _stream_ops(seed, nbatches, max_count, p_malloc=0.6):
    """Batches of Zipf sizes in random order; each request a malloc of a
    lognormal(6, 2) size or the free of a random live pointer of an earlier
    batch."""
    rng = np.random.default_rng(seed)
    counts = rng.permutation(_zipf_counts(nbatches, max_count))
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.uint64)
    ops = np.zeros(int(offsets[-1]), G.BATCH_OP_DTYPE)
    live, slots = np.empty(0, np.uint32), 0
    for b, n in enumerate(counts):
        o = ops[int(offsets[b]):int(offsets[b + 1])]
        nf = min(len(live), int(rng.binomial(int(n), 1 - p_malloc)))
        is_free = np.zeros(n, bool)
        is_free[rng.permutation(int(n))[:nf]] = True
        live = rng.permutation(live)
        o["kind"][is_free] = 1
        o["slot"][is_free] = live[:nf]
        new = np.arange(slots, slots + int(n) - nf, dtype=np.uint32)
        o["slot"][~is_free] = new
        o["arg"][~is_free] = lognormal_sizes(rng, len(new), 6.0, 2.0, 16 * MIB)
        slots += len(new)
        live = np.concatenate([live[nf:], new])
    return ops, offsets, slots


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    h = _Held(kind=kind, case=case, seed=int(seed))
    if kind == "churn":
        h.alloc = G.Gallatin(16 * MIB, 16, 4096).generate_on_device(
            case["pool_gib"] * GIB, 1234, print_info=False,
            slots_min=32 if case["pool_gib"] >= 8 else 4)
    elif kind == "big":
        h.alloc = G.Gallatin(16 * MIB, 16, 4096).generate_on_device(
            case["pool_gib"] * GIB, 1234, print_info=False)
        # how many requests a step has varies by some percent
        h.n_small = case["n_small"] - int(rng.integers(case["n_small"] // 8 + 2))
        h.n_large = case["n_large"]
        h.ptrs = torch.zeros(h.n_small + h.n_large, dtype=torch.int64, device="cuda")
        h.step = 0
    elif kind == "stream":
        h.alloc = G.Gallatin(case["segment_mib"] * MIB, case["smallest"], 4096) \
            .generate_on_device(case["pool_gib"] * GIB, 1234, print_info=False, slots_min=32,
                                flags=G.GAL_FLAG_NO_PAYLOAD_FENCE)
        h.stream = G.BatchStream(*_stream_ops(seed, case["nbatches"], case["max_count"]))
        h.counters = torch.zeros(G.CTR_COUNT, dtype=torch.int64, device="cuda")
        if case["plan"]:
            h.plan = G.BatchPlan(h.alloc, h.stream, h.counters, threads=case["threads"],
                                 batched=case["batched"])
    elif kind == "table":
        _global()
        keys = _distinct(rng, case["held"] + 2 * case["n"], 40)
        held, new, other = np.split(keys, (case["held"], case["held"] + case["n"]))
        h.table = G.Table(1 if case["large"] else 0, seed=42)
        h.table.insert(_cuda(held), _cuda(held * 3))
        h.keys = _cuda(rng.permutation(new))
        h.vals = _cuda(rng.integers(1 << 62, size=case["n"]))
        h.asked = _cuda(np.where(rng.random(case["n"]) < case["absent"], other, new))
    elif kind == "chain":
        _global()
        dt = np.int64 if G.ChainTable.KINDS[case["layout"]][0] == 8 else np.int32
        keys = _distinct(rng, 2 * case["n"], 40 if dt == np.int64 else 30)
        new, other = np.split(keys, 2)
        h.keys = _cuda(rng.permutation(new).astype(dt))
        h.vals = _cuda(rng.integers(1 << 30, size=case["n"]).astype(dt))
        h.asked = _cuda(np.where(rng.random(case["n"]) < case["absent"], other, new).astype(dt))
        h.nslots = max(64, int(case["n"] / case["load"]))
    elif kind == "queue":
        if case["form"].startswith("block"):
            _global()
            h.queue = G.BlockQueue(0 if case["form"] == "block256" else 1)
        else:
            h.alloc = G.Gallatin(16 * MIB, 16, 4096).generate_on_device(
                case["pool_gib"] * GIB, 1234, print_info=False)
            h.queue = G.Queue(h.alloc, ring=case["form"] == "ring")
        h.items = _cuda(_distinct(rng, case["n"], 40))
    else:
        _global()
        p_end = 1.0 / case["life"]
        h.loop = serving.Serving(case["sessions"], seed=h.seed)
        h.p_end = p_end
        h.arrivals = rng.poisson(0.5 * case["sessions"] * p_end, 4096)
        h.counters = torch.zeros(16, dtype=torch.int64, device="cuda")
        h.step = 0
        for _ in range(3 * case["life"]):
            _serve(h)
    return h


def _serve(h):
    h.loop.step(h.step, int(h.arrivals[h.step % len(h.arrivals)]), 64, h.p_end,
                h.case["ht_ops"], h.counters)
    h.step += 1


def run(h):
    c = h.case
    if h.kind == "churn":
        if c["words"]:
            return h.alloc.run_churn_word(h.seed, c["n"], c["rounds"], batched=c["batched"],
                                          threads=c["threads"])
        if c["batched"]:
            return h.alloc.run_churn_batched(h.seed, c["n"], c["rounds"], threads=c["threads"])
        return h.alloc.run_churn(h.seed, c["n"], c["rounds"], block_threads=c["threads"])
    if h.kind == "big":
        h.step += 1
        return h.alloc.run_big(h.seed, h.step, h.n_small, h.n_large, ptrs=h.ptrs)[1]
    if h.kind == "stream":
        h.counters.zero_()
        if c["plan"]:
            h.plan.launch()
        else:
            G.run_batches(h.alloc, h.stream, h.counters, threads=c["threads"],
                          batched=c["batched"])
        # pairs, misses, bad tags, bytes, mallocs, timeouts, frees skipped;
        # the words after them are the waits' polls and clock ticks
        return h.counters[:7]
    if h.kind == "table":
        stored = h.table.insert(h.keys, h.vals)
        vals, found = h.table.query(h.asked)
        removed = h.table.remove(h.keys)
        return stored, vals, found, removed
    if h.kind == "chain":
        t = G.ChainTable(c["layout"], nslots=h.nslots, default_key=0)
        stored = t.insert(h.keys, h.vals)
        vals, found = t.query(h.asked)
        t.destroy()
        return stored, vals, found
    if h.kind == "queue":
        put = h.queue.enqueue(h.items)
        out, got = h.queue.dequeue(c["n"])
        if c["form"].startswith("block"):
            h.queue.reclaim()
        # items of one launch come out in any order: sorted by their ids
        return put, torch.sort(out)[0], got
    _serve(h)
    # sessions, words and chunks so far and keys inserted; how many removes
    # found their key depends on the order of the step's table operations
    return h.counters[:9]


def work(case):
    k = case["kind"]
    if k == "churn":
        pairs = case["n"] * (1 + (case["rounds"] - 1) / 2)
        return {"bytes": pairs * (16 if case["words"] else 991), "flops": 0}
    if k == "big":
        return {"bytes": 48 * (case["n_small"] + case["n_large"]), "flops": 0}
    if k == "stream":
        n = float(_zipf_counts(case["nbatches"], case["max_count"]).sum())
        return {"bytes": n * 16 + 0.6 * n * 32, "flops": 0}
    if k == "table":
        # pairs in, stored pairs written; keys asked, values out; keys removed
        return {"bytes": case["n"] * (16 + 16 + 1 + 8 + 16 + 9 + 8 + 8 + 1), "flops": 0}
    if k == "chain":
        w = G.ChainTable.KINDS[case["layout"]][0]
        return {"bytes": case["n"] * (2 * w + 2 * w + 1 + w + 2 * w + w + 1), "flops": 0}
    if k == "queue":
        return {"bytes": case["n"] * (8 + 16 + 1 + 16 + 8 + 1), "flops": 0}
    # words appended by the live sessions (mean 33 tokens of 256 B), table pairs
    live = 0.5 * case["sessions"]
    return {"bytes": live * 33 * 256 + case["ht_ops"] * 16, "flops": 0}
