"""The calls this library spends its users' time in, over the sizes they are made at.

Every case is one public entry point of the C ABI, called as a plugin or a tool calls it: inputs,
outputs and plans are in hand, one call is a pass.  `listed()` names the ones looked at first,
`draw()` gives more of the same ranges.
"""
import ctypes

import numpy as np
import torch

import aws_ofi_nccl_amd as m
from aws_ofi_nccl_amd import synthetic

SIGNAL_BASE = 0x7F5500000000
RX_STRIDE = 8320         # an rx buffer: 8 bytes of header and 8184 of payload on a 128-byte boundary
GIN_THREADS = 4          # NCCL runs up to four GIN proxy threads
SWEEP_COLLS = (4, 2, 3)  # AllReduce, AllGather, ReduceScatter


def listed():
    return [
        # what one progress call of a busy proxy hands to the scheduler: latency
        dict(name="stripe_1000", path="stripe", n=1000, rails=4, min_stripe=131072, max_small=64),
        # the configured striping batch
        dict(name="stripe_1000000", path="stripe", n=1000000, rails=4, min_stripe=131072, max_small=64),
        # the largest batch striping is used at: the output no longer fits any cache
        dict(name="stripe_16000000", path="stripe", n=16000000, rails=4, min_stripe=131072, max_small=64),
        # the configured bounce batch: eager buffers scattered over a 2 GiB arena, flushed
        dict(name="bounce_65536", path="bounce", n=65536, max_len=8192, arena=2 << 30, flush=True),
        # the eager arrivals of one receive round with the usual 64 messages in flight
        dict(name="eager_64", path="eager", n=64, max_len=8184, host_rx=False, truncate=False),
        # eager arrivals by the rx pool: any destination alignment
        dict(name="eager_65536", path="eager", n=65536, max_len=8184, host_rx=False, truncate=False),
        # a launch group of one-sided writes, 8 B to 1 MiB as the GIN traffic mixes them
        dict(name="writes_2048", path="writes", n=2048, lo=3, hi=20, align=8),
        # signals released by a launch group's writes, in the pinned memory the receiver fills
        dict(name="signals_16384", path="signals", n=16384, slots=512, regions=1, pinned=True),
        # the configured cost-model grids: 2 platforms x 32 pipeline depths
        dict(name="model_64_grids", path="model", variants=64, per_octave=4, octaves=35, nodes=11),
        # a decision sweep of the four platforms, 16 sizes an octave and 4 node counts an octave
        dict(name="region_sweep", path="region", platforms=4, per_octave=16, octaves=35, nodes=44),
        # what a communicator's start evaluates ahead: a ladder of sizes for every collective
        dict(name="queries_259", path="queries", n=259),
        # GPU-initiated puts: device producers, pinned rings, proxy threads that derive wire records
        dict(name="gin_256x1000", path="gin", contexts=256, ops=1000, capacity=4096),
    ]


def _log_int(rng, lo, hi):
    """Log-uniform whole number in [lo, hi], odd ones as likely as even ones."""
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    path = rng.choice(["stripe", "stripe", "bounce", "eager", "writes", "signals", "model", "region", "queries", "gin"])
    if path == "stripe":
        return dict(path=path, n=_log_int(rng, 64, 16000000), rails=rng.randint(1, 4),
                    min_stripe=rng.choice([131072, 131072, 65536, 100000]), max_small=rng.choice([64, 64, 0, 8192]))
    if path == "bounce":
        n = _log_int(rng, 16, 65536)
        return dict(path=path, n=n, max_len=rng.choice([8192, 8192, 4096, 1000]), arena=n * 32768,
                    flush=rng.random() < 0.75)
    if path == "eager":
        host_rx = rng.random() < 0.25
        return dict(path=path, n=_log_int(rng, 16, 2048 if host_rx else 65536), max_len=rng.choice([8184, 8184, 4000, 500]),
                    host_rx=host_rx, truncate=rng.random() < 0.25)
    if path == "writes":
        # a few long stripes of rendezvous messages, or many one-sided writes of mixed size
        hi = rng.randint(13, 26)
        lo = rng.choice([3, max(3, hi - 6), hi - 1])
        most = max(16, min(16384, (1 << 30) // int(_mean_len(lo, hi))))
        return dict(path=path, n=_log_int(rng, 4, most), lo=lo, hi=hi, align=rng.choice([1, 8, 128]))
    if path == "signals":
        return dict(path=path, n=_log_int(rng, 64, 1 << 18), slots=rng.choice([1, 64, 512, 65536]),
                    regions=rng.randint(1, 16), pinned=rng.random() < 0.5)
    if path == "model":
        return dict(path=path, variants=_log_int(rng, 1, 256), per_octave=rng.choice([1, 2, 4]), octaves=rng.randint(20, 35),
                    nodes=rng.randint(3, 16))
    if path == "region":
        return dict(path=path, platforms=rng.randint(1, 4), per_octave=_log_int(rng, 1, 16), octaves=rng.randint(20, 35),
                    nodes=_log_int(rng, 4, 44))
    if path == "queries":
        return dict(path=path, n=_log_int(rng, 16, 1200))
    return dict(path=path, contexts=_log_int(rng, 8, 256), ops=_log_int(rng, 100, 1000), capacity=rng.choice([1024, 4096]))


class State:
    """What a caller keeps between calls; library objects are given back with it."""

    def __init__(self, case):
        self.case = case
        self.stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        self.plan = self.rings = None

    def __del__(self):
        if self.plan:
            m.load().ofi_amd_tuner_plan_destroy(self.plan)
        if self.rings:
            m.load().ofi_amd_gin_rings_destroy(self.rings)


def _dev(a):
    """numpy array -> device tensor with the same bytes (unsigned types travel as signed)."""
    signed = {1: np.uint8, 2: np.int16, 4: np.int32, 8: np.int64}[a.dtype.itemsize]
    return torch.from_numpy(np.ascontiguousarray(a).view(signed)).cuda()


def _log_lens(gen, n, lo, hi):
    """Whole lengths in [2^lo, 2^hi): uniform octave, uniform inside it."""
    e = torch.randint(lo, hi, (n,), generator=gen, device="cuda")
    one = torch.ones_like(e)
    return (one << e) | (torch.randint(0, 1 << 62, (n,), generator=gen, device="cuda") & ((one << e) - 1))


def _mean_len(lo, hi):
    return 1.5 * ((1 << hi) - (1 << lo)) / (hi - lo)


def prepare(case, seed):
    lib = m.load()
    m.check(lib.ofi_amd_gpu_init(), "gpu_init")
    s = State(case)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    rng = np.random.default_rng(seed)
    globals()["_prepare_" + case["path"]](lib, s, case, seed, gen, rng)
    return s


def run(s):
    return globals()["_run_" + s.case["path"]](m.load(), s)


# ---- rail striping: one scheduler's batches, chained on a stream through the state in HBM ----

def _prepare_stripe(lib, s, case, seed, gen, rng):
    n = s.n = case["n"]
    s.sizes = _log_lens(gen, n, 0, 28)
    st = m.SchedState(int(rng.integers(0, case["rails"])), int(rng.integers(0, case["rails"])), case["max_small"],
                      case["min_stripe"], case["rails"], 0)
    s.sched = _dev(np.frombuffer(bytes(st), dtype=np.uint8).copy())
    s.num = torch.zeros(n, dtype=torch.int32, device="cuda")
    s.xfers = torch.zeros(n * 12, dtype=torch.int64, device="cuda")


def _run_stripe(lib, s):
    m.check(lib.ofi_amd_sched_batch(s.sched.data_ptr(), s.sizes.data_ptr(), s.n, 128, s.num.data_ptr(),
                                    s.xfers.data_ptr(), s.stream), "sched_batch")
    return s.num, s.xfers, s.sched


# ---- bounce copy and flush: packed source, 64-byte-aligned destinations, flush words in pinned memory ----

def _prepare_bounce(lib, s, case, seed, gen, rng):
    w = synthetic.bounce_workload(seed, case["n"], case["max_len"], case["arena"])
    s.n, s.arena_bytes = case["n"], case["arena"]
    s.src = torch.randint(0, 256, (w["src_bytes"] + 16,), dtype=torch.uint8, generator=gen, device="cuda")
    s.arena = torch.zeros(s.arena_bytes, dtype=torch.uint8, device="cuda")
    s.src_off, s.dst_off, s.len = _dev(w["src_off"]), _dev(w["dst_off"]), _dev(w["len"])
    s.flush = torch.zeros(s.n, dtype=torch.int32).pin_memory() if case["flush"] else None


def _run_bounce(lib, s):
    m.check(lib.ofi_amd_bounce_scatter(s.src.data_ptr(), s.src.numel(), s.arena.data_ptr(), s.arena_bytes,
                                       s.src_off.data_ptr(), s.dst_off.data_ptr(), s.len.data_ptr(), s.n,
                                       s.flush.data_ptr() if s.flush is not None else None, s.stream), "bounce_scatter")
    return s.arena, s.flush


# ---- eager arrivals: rx buffers in arrival order, destinations at any alignment ----

def _prepare_eager(lib, s, case, seed, gen, rng):
    n = s.n = case["n"]
    s.rx = torch.randint(0, 256, (n * RX_STRIDE,), dtype=torch.uint8, generator=gen, device="cuda")
    if case["host_rx"]:
        s.rx = s.rx.cpu().pin_memory()
    lens = rng.integers(0, case["max_len"] + 1, n).astype(np.uint32)
    room = np.where(rng.random(n) < 0.25, lens // 2, lens).astype(np.uint32) if case["truncate"] else lens
    s.rx_off = _dev(rng.permutation(n).astype(np.uint64) * np.uint64(RX_STRIDE))
    s.recv_len, s.dst_len = _dev(lens), _dev(room)
    s.dst_off = _dev(rng.permutation(2 * n)[:n].astype(np.uint64) * np.uint64(16384) + rng.integers(0, 64, n).astype(np.uint64))
    s.dst = torch.zeros(2 * n * 16384, dtype=torch.uint8, device="cuda")
    s.copied = torch.zeros(n, dtype=torch.int32, device="cuda")
    s.flush = torch.zeros(n, dtype=torch.int32, device="cuda")


def _run_eager(lib, s):
    m.check(lib.ofi_amd_eager_copy_batch(s.rx.data_ptr(), s.rx_off.data_ptr(), s.recv_len.data_ptr(), s.dst.data_ptr(),
                                         s.dst_off.data_ptr(), s.dst_len.data_ptr(), s.n, s.copied.data_ptr(),
                                         s.flush.data_ptr(), s.stream), "eager_copy_batch")
    return s.dst, s.copied, s.flush


# ---- one-sided writes and rendezvous stripes: a table in the pinned memory the proxy fills ----

def _prepare_writes(lib, s, case, seed, gen, rng):
    n, align = case["n"], case["align"]
    lens = _log_lens(gen, n, case["lo"], case["hi"]).cpu().numpy()
    room = (lens + 255) // 128 * 128           # ranges of a batch are disjoint
    order = rng.permutation(n)
    at = np.zeros(n, dtype=np.int64)
    at[order] = np.cumsum(room[order]) - room[order]
    src_at = np.cumsum(room) - room + rng.integers(0, 128, n) // align * align
    # the windows a program registers ahead: the same size whatever the lengths come out as
    mean = _mean_len(case["lo"], case["hi"])
    total = int(min(n << case["hi"], 1.35 * n * mean + (8 << case["hi"]))) + 256 * n + 256
    if int(room.sum()) + 256 > total:
        raise RuntimeError("the writes of this seed do not fit their window")
    s.n, s.max_len = n, int(lens.max())
    s.src = torch.randint(0, 1 << 62, (total // 8 + 1,), generator=gen, device="cuda").view(torch.uint8)
    s.dst = torch.zeros(total, dtype=torch.uint8, device="cuda")
    at = at + rng.integers(0, 128, n) // align * align
    s.src_addr = torch.from_numpy(src_at + s.src.data_ptr()).pin_memory()
    s.dst_addr = torch.from_numpy(at + s.dst.data_ptr()).pin_memory()
    s.len = torch.from_numpy(lens.astype(np.int32)).pin_memory()


def _run_writes(lib, s):
    m.check(lib.ofi_amd_copy_table_pieces(s.src_addr.data_ptr(), s.dst_addr.data_ptr(), s.len.data_ptr(), s.n, s.max_len,
                                          s.stream), "copy_table_pieces")
    return s.dst


# ---- signal delivery: folded work items onto counters in HBM ----

def _prepare_signals(lib, s, case, seed, gen, rng):
    n, slots, regions = case["n"], case["slots"], case["regions"]
    s.n, s.n_regions = n, regions
    s.counters = torch.randint(0, 1 << 40, (regions * slots,), generator=gen, device="cuda")
    s.regions = (m.GinSignalRegion * regions)(*[
        m.GinSignalRegion(SIGNAL_BASE + (r << 32), 8 * slots, s.counters.data_ptr() + 8 * slots * r) for r in range(regions)])
    item = np.dtype([("base", "<u8"), ("offset", "<u8"), ("value", "<u8"), ("peer", "<u4"), ("gate_seq", "<u2"),
                     ("run_len", "<u2")])
    work = np.zeros(n, dtype=item)
    work["base"] = SIGNAL_BASE + (rng.integers(0, regions, n).astype(np.uint64) << np.uint64(32))
    work["offset"] = 8 * rng.integers(0, slots, n)
    work["value"] = rng.integers(1, 65537, n)
    work["peer"] = rng.integers(0, 256, n)
    work["gate_seq"] = rng.integers(0, 8192, n)
    work["run_len"] = 1
    words = torch.from_numpy(work.view(np.int64))
    s.work = words.pin_memory() if case["pinned"] else words.cuda()
    s.rejected = torch.zeros(1, dtype=torch.int32, device="cuda")


def _run_signals(lib, s):
    m.check(lib.ofi_amd_gin_signal_apply(s.work.data_ptr(), s.n, s.regions, s.n_regions, s.rejected.data_ptr(), s.stream),
            "gin_signal_apply")
    return s.counters, s.rejected


# ---- tuner: cost-model grids, decision grids, point queries ----

def _plan(lib, s, case, rng, nodes):
    step = 1.0 / case["per_octave"]
    sizes = np.round(2.0 ** (step * (np.arange(case["octaves"] * case["per_octave"]) + rng.random()))).astype(np.uint64)
    colls = np.array(SWEEP_COLLS, dtype=np.int32)
    ppn = np.array([1, 2, 4, 8], dtype=np.uint32)
    algos = np.array([1, 0, 6], dtype=np.int32)          # Ring, Tree, PAT
    s.plan = ctypes.c_void_p()
    m.check(lib.ofi_amd_tuner_plan_create(colls.ctypes.data, len(colls), sizes.ctypes.data, len(sizes), nodes.ctypes.data,
                                          len(nodes), ppn.ctypes.data, len(ppn), algos.ctypes.data, len(algos),
                                          ctypes.byref(s.plan)), "plan_create")
    s.points, s.cells = lib.ofi_amd_tuner_plan_points(s.plan), lib.ofi_amd_tuner_plan_cells(s.plan)


def _prepare_model(lib, s, case, seed, gen, rng):
    _plan(lib, s, case, rng, (1 << np.arange(case["nodes"])).astype(np.uint64))
    s.nv = case["variants"]
    channels = int(rng.integers(4, 17))
    s.variants = (m.TunerVariant * s.nv)(*[m.TunerVariant(i % 2, 1 + (i // 2) % 32, channels + i // 64, 3) for i in range(s.nv)])
    s.cost = torch.zeros(s.nv * s.cells, dtype=torch.float64, device="cuda")
    s.choice = torch.zeros(s.nv * s.points * 2, dtype=torch.int8, device="cuda")


def _run_model(lib, s):
    m.check(lib.ofi_amd_tuner_model_grid(s.plan, s.variants, s.nv, s.cost.data_ptr(), s.choice.data_ptr(), s.stream),
            "model_grid")
    return s.cost, s.choice


def _prepare_region(lib, s, case, seed, gen, rng):
    # node counts from 1 up to 1024 at most, spread over the octaves
    nodes = np.unique(np.round(2.0 ** (np.arange(case["nodes"]) * 10.0 / max(1, case["nodes"] - 1))).astype(np.uint64))
    _plan(lib, s, case, rng, nodes)
    s.platforms = np.arange(case["platforms"], dtype=np.int32)
    s.choice = torch.zeros(len(s.platforms) * s.points * 4, dtype=torch.int8, device="cuda")


def _run_region(lib, s):
    m.check(lib.ofi_amd_tuner_region_grid(s.plan, s.platforms.ctypes.data, len(s.platforms), s.choice.data_ptr(), s.stream),
            "region_grid")
    return s.choice


def _prepare_queries(lib, s, case, seed, gen, rng):
    n = s.n = case["n"]
    nodes = rng.choice([4, 8, 16, 32, 64, 128], n)
    ppn = rng.choice([1, 8], n)
    s.queries = (m.TunerQuery * n)(*[
        m.TunerQuery(int(rng.integers(0, 4)), i % 3, SWEEP_COLLS[int(rng.integers(0, 3))], 1, 8, 3, 0 if i % 2 else 6,
                     1 if i % 2 else 2, (1 << 21) - 1, 0, int(2.0 ** (34 * rng.random())), int(nodes[i] * ppn[i]),
                     int(nodes[i])) for i in range(n)])
    s.answers = np.zeros(2 * n, dtype=np.int64)
    m.check(lib.ofi_amd_tuner_query_prepare(n), "query_prepare")


def _run_queries(lib, s):
    m.check(lib.ofi_amd_tuner_query(s.queries, s.n, s.answers.ctypes.data), "query")
    return s.answers


# ---- GIN puts: produced on the GPU, drained and derived by proxy threads ----

def _prepare_gin(lib, s, case, seed, gen, rng):
    nctx = s.nctx = case["contexts"]
    s.ops, s.seed = case["ops"], seed
    s.rings = ctypes.c_void_p()
    m.check(lib.ofi_amd_gin_rings_create(nctx, case["capacity"], ctypes.byref(s.rings)), "rings_create")
    s.comms, s.fresh = (m.GinComm * nctx)(), (m.GinComm * nctx)()
    for c in range(nctx):
        lib.ofi_amd_gin_comm_init(ctypes.byref(s.fresh[c]), c % 1024, 4, 131072, 64, 1)
    s.mrs = (m.GinMr * 3)()
    for i in range(3):
        s.mrs[i].local_base = 0x7F0000000000 + (i << 36)
        s.mrs[i].remote_address = 0x7F5500000000 + (i << 36)
        s.mrs[i].remote_address_offset = i << 36
        for r in range(4):
            s.mrs[i].key[r] = 0x1000 * (i + 1) + r
    s.stats = m.GinProxyStats()
    s.wires = np.zeros(nctx * s.ops * 28, dtype=np.int64)


def _run_gin(lib, s):
    ctypes.memmove(s.comms, s.fresh, ctypes.sizeof(s.fresh))
    m.check(lib.ofi_amd_gin_produce_seeded(s.rings, s.seed, s.ops, 1, 64, 1, 1, 0, s.stream), "produce_seeded")
    m.check(lib.ofi_amd_gin_proxy_drain_mt(s.rings, s.ops, 2, None, s.comms, s.mrs, 3, s.wires.ctypes.data, 20000,
                                           GIN_THREADS, ctypes.byref(s.stats)), "proxy_drain")
    return s.wires, np.frombuffer(s.comms, dtype=np.uint8)


def work(case):
    path = case["path"]
    n = case.get("n", 0)
    if path == "stripe":                                  # 8 read, 4 + 96 written
        return {"bytes": 108.0 * n}
    if path == "bounce":                                  # payload twice, its table, the flush word
        return {"bytes": n * (case["max_len"] + 20.0 + (8 if case["flush"] else 0))}
    if path == "eager":
        return {"bytes": n * (case["max_len"] * (7 / 8 if case["truncate"] else 1.0) + 24.0 + 12.0)}
    if path == "writes":
        return {"bytes": n * (2 * _mean_len(case["lo"], case["hi"]) + 20.0)}
    if path == "signals":
        return {"bytes": 32.0 * n + 16.0 * min(n, case["slots"] * case["regions"])}
    points = len(SWEEP_COLLS) * 4.0 * case.get("octaves", 0) * case.get("per_octave", 0) * case.get("nodes", 0)
    if path == "model":                                   # 9 cells of 8 bytes and a decision of 2 per point
        return {"bytes": case["variants"] * points * 74, "flops": case["variants"] * points * 9 * 8}
    if path == "region":
        return {"bytes": case["platforms"] * points * 4}
    if path == "queries":
        return {"bytes": 80.0 * n}
    return {"bytes": case["contexts"] * case["ops"] * (64.0 + 4.0 + 224.0)}


def tolerance(case):
    # rails, bytes, counters, decisions and wire words are whole; the model's costs are rounded as
    # the reference rounds them, operation by operation
    return "exact"
