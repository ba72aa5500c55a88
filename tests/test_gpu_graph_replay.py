"""The launch-bound entry points recorded into one HIP graph and replayed: striping (two
launches), bounce copy, eager-format copy and signal delivery.  None of them allocates or
synchronises once its stream has been used, so they can be captured; every replay is
checked against the oracle, with eager work and synchronisations between replays."""
import ctypes

import numpy as np
import pytest
import torch

import _gpu
import _oracle
import aws_ofi_nccl_amd as m
from aws_ofi_nccl_amd import synthetic

pytestmark = pytest.mark.gpu
SCRATCH_WORDS = 29_760  # of a stream's striping scratch, kScratchWords in csrc/sched_stripe.hip


def test_graph_of_hot_path_launches_replays_exactly(lib, oracle, gpu):
    rng = np.random.default_rng(77)
    s = torch.cuda.Stream()
    sp = ctypes.c_void_p(s.cuda_stream)

    # striping inputs; the scheduler state lives on the device and advances with every replay
    n_msg = 50_000
    sizes = synthetic.stripe_sizes(5, n_msg)
    st = m.SchedState(2, 1, 64, 131072, 4, 0)
    d_state = _gpu.to_dev(np.frombuffer(bytes(st), dtype=np.uint8).copy())
    d_sizes = _gpu.to_dev(sizes)
    d_num = torch.zeros(n_msg, dtype=torch.int32, device="cuda")
    d_xf = torch.zeros(n_msg * 12, dtype=torch.int64, device="cuda")

    # bounce copy inputs
    w = synthetic.bounce_workload(9, n=2048, arena_bytes=32 << 20)
    src = synthetic.random_bytes(9, w["src_bytes"] + 16)
    d_src, d_so, d_do, d_len = (_gpu.to_dev(x) for x in (src, w["src_off"], w["dst_off"], w["len"]))
    d_arena = torch.zeros(w["arena_bytes"], dtype=torch.uint8, device="cuda")
    d_flush = torch.zeros(2048, dtype=torch.int32, device="cuda")
    want_arena = np.zeros(w["arena_bytes"], dtype=np.uint8)
    want_flush = np.zeros(2048, dtype=np.uint32)
    oracle.oracle_bounce_scatter(_oracle.ptr(src), _oracle.ptr(want_arena), _oracle.ptr(w["src_off"]),
                                 _oracle.ptr(w["dst_off"]), _oracle.ptr(w["len"]), 2048,
                                 _oracle.ptr(want_flush))

    # signal delivery inputs: counters accumulate across replays
    n_sig, base = 10_000, 0x7F0000000000
    work = np.zeros(n_sig, dtype=np.dtype([("base", "<u8"), ("offset", "<u8"), ("value", "<u8"),
                                            ("peer", "<u4"), ("gate_seq", "<u2"), ("run_len", "<u2")]))
    work["base"], work["run_len"] = base, 1
    work["offset"] = 8 * rng.integers(0, 128, n_sig).astype(np.uint64)
    work["value"] = rng.integers(0, 1 << 64, n_sig, dtype=np.uint64)
    d_work = _gpu.to_dev(work.view(np.uint8))
    d_cnt = torch.zeros(128, dtype=torch.int64, device="cuda")
    regions = (m.GinSignalRegion * 1)(m.GinSignalRegion(base, 1024, d_cnt.data_ptr()))
    per_replay = np.zeros(128, dtype=np.uint64)
    with np.errstate(over="ignore"):
        np.add.at(per_replay, (work["offset"] // 8).astype(np.int64), work["value"])

    # eager-format copy and table copy out of the same source bytes
    n_e, stride = 512, 8320
    e_len = rng.integers(0, 8185, n_e).astype(np.uint32)
    e_rx = (rng.permutation(n_e).astype(np.uint64) * np.uint64(stride))
    e_dst = (np.arange(n_e, dtype=np.uint64) * np.uint64(8192 + 64) + rng.integers(0, 16, n_e).astype(np.uint64))
    d_earena = torch.zeros(n_e * (8192 + 64), dtype=torch.uint8, device="cuda")
    d_erx, d_elen, d_edst = _gpu.to_dev(e_rx), _gpu.to_dev(e_len), _gpu.to_dev(e_dst)
    d_copied = torch.zeros(n_e, dtype=torch.int32, device="cuda")
    want_earena = np.zeros(n_e * (8192 + 64), dtype=np.uint8)
    oracle.oracle_eager_copy_batch(_oracle.ptr(src), _oracle.ptr(e_rx), _oracle.ptr(e_len), _oracle.ptr(want_earena),
                                   _oracle.ptr(e_dst), _oracle.ptr(e_len), n_e, None)
    n_t = 300
    t_len = rng.integers(1, 70000, n_t).astype(np.uint32)
    t_src_off = rng.integers(0, w["src_bytes"] - 70000, n_t).astype(np.uint64)
    t_dst_off = np.concatenate(([0], np.cumsum(t_len.astype(np.uint64) + np.uint64(3))[:-1])).astype(np.uint64)
    d_tarena = torch.zeros(int(t_dst_off[-1]) + 70000, dtype=torch.uint8, device="cuda")
    d_tsrc = _gpu.to_dev(t_src_off + np.uint64(d_src.data_ptr()))
    d_tdst = _gpu.to_dev(t_dst_off + np.uint64(d_tarena.data_ptr()))
    d_tlen = _gpu.to_dev(t_len)
    d_parena = torch.zeros_like(d_tarena)    # the same table through the launch with a wavefront per 8 KiB
    d_pdst = _gpu.to_dev(t_dst_off + np.uint64(d_parena.data_ptr()))
    want_tarena = np.zeros(d_tarena.numel(), dtype=np.uint8)
    for a, b, l in zip(t_src_off, t_dst_off, t_len):
        want_tarena[int(b):int(b) + int(l)] = src[int(a):int(a) + int(l)]

    def launches():
        assert lib.ofi_amd_eager_copy_batch(d_src.data_ptr(), d_erx.data_ptr(), d_elen.data_ptr(),
                                            d_earena.data_ptr(), d_edst.data_ptr(), d_elen.data_ptr(), n_e,
                                            d_copied.data_ptr(), None, sp) == 0
        assert lib.ofi_amd_copy_table(d_tsrc.data_ptr(), d_tdst.data_ptr(), d_tlen.data_ptr(), n_t, sp) == 0
        assert lib.ofi_amd_copy_table_pieces(d_tsrc.data_ptr(), d_pdst.data_ptr(), d_tlen.data_ptr(), n_t, 70000,
                                             sp) == 0
        assert lib.ofi_amd_sched_batch(d_state.data_ptr(), d_sizes.data_ptr(), n_msg, 128, d_num.data_ptr(),
                                       d_xf.data_ptr(), sp) == 0
        assert lib.ofi_amd_bounce_scatter(d_src.data_ptr(), d_src.numel(), d_arena.data_ptr(), w["arena_bytes"],
                                          d_so.data_ptr(), d_do.data_ptr(), d_len.data_ptr(), 2048,
                                          d_flush.data_ptr(), sp) == 0
        assert lib.ofi_amd_gin_signal_apply(d_work.data_ptr(), n_sig, regions, 1, None, sp) == 0

    # first use of the stream sets up the per-stream striping scratch (an allocation): outside capture
    with torch.cuda.stream(s):
        launches()
    s.synchronize()
    ost = _oracle.Sched(2, 1, 64, 131072, 4, 0)
    num = np.zeros(n_msg, dtype=np.uint32)
    xf = np.zeros((n_msg, 4, 3), dtype=np.uint64)
    oracle.oracle_sched_batch(ctypes.byref(ost), _oracle.ptr(sizes), n_msg, 128, _oracle.ptr(num),
                              _oracle.ptr(xf))
    assert np.array_equal(_gpu.to_host(d_xf, np.uint64).reshape(n_msg, 4, 3), xf)
    counters = per_replay.copy()

    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        launches()

    for replay in range(4):
        # eager work and a synchronisation between replays; outputs wiped so a replay must rewrite them
        d_arena.zero_()
        d_earena.zero_()
        d_tarena.zero_()
        d_parena.zero_()
        d_copied.zero_()
        d_flush.zero_()
        d_num.fill_(-1)
        d_xf.fill_(-1)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        # the oracle advances its own state by one batch: replay k continues where k-1 stopped
        oracle.oracle_sched_batch(ctypes.byref(ost), _oracle.ptr(sizes), n_msg, 128, _oracle.ptr(num),
                                  _oracle.ptr(xf))
        assert np.array_equal(_gpu.to_host(d_num, np.uint32), num), replay
        assert np.array_equal(_gpu.to_host(d_xf, np.uint64).reshape(n_msg, 4, 3), xf), replay
        got_state = m.SchedState.from_buffer_copy(d_state.cpu().numpy().tobytes())
        assert (got_state.rr_small_counter, got_state.rr_counter) == (ost.rr_small_counter, ost.rr_counter)
        assert np.array_equal(d_arena.cpu().numpy(), want_arena), replay
        assert np.array_equal(d_earena.cpu().numpy(), want_earena), replay
        assert np.array_equal(_gpu.to_host(d_copied, np.uint32), e_len), replay
        assert np.array_equal(d_tarena.cpu().numpy(), want_tarena), replay
        assert np.array_equal(d_parena.cpu().numpy(), want_tarena), replay
        assert np.array_equal(_gpu.to_host(d_flush, np.uint32), want_flush), replay
        with np.errstate(over="ignore"):
            counters += per_replay
        assert np.array_equal(_gpu.to_host(d_cnt, np.uint64), counters), replay
    assert _gpu.fetch_async_errors(lib) == 0


@pytest.mark.parametrize("n", [1000, 30_001])
def test_batch_first_called_while_its_stream_is_captured(lib, oracle, gpu, n):
    """The scratch of a stream is made by the call that the stream is being captured in (a capture mode that lets a
    call allocate): batches called before the first replay, the replay and batches after it all match the oracle,
    whatever the memory held.  1000 messages are one launch when called, whose workgroups count themselves in the
    scratch, 30,001 one whose workgroups publish totals there, and both two when captured."""
    s = torch.cuda.Stream()
    sp = ctypes.c_void_p(s.cuda_stream)
    assert lib.ofi_amd_sched_stream_release(sp) == 0
    # memory of the scratch's size, left dirty for the allocator to hand out again
    dirty = [torch.full((SCRATCH_WORDS,), -1, dtype=torch.int32, device="cuda") for _ in range(8)]
    torch.cuda.synchronize()
    del dirty
    torch.cuda.empty_cache()
    sizes = synthetic.stripe_sizes(6, n)
    st = m.SchedState(2, 1, 64, 131072, 4, 0)
    d_state = _gpu.to_dev(np.frombuffer(bytes(st), dtype=np.uint8).copy())
    d_sizes = _gpu.to_dev(sizes)
    d_num = torch.zeros(n, dtype=torch.int32, device="cuda")
    d_xf = torch.zeros(n * 12, dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()

    def call():
        return lib.ofi_amd_sched_batch(d_state.data_ptr(), d_sizes.data_ptr(), n, 128, d_num.data_ptr(), d_xf.data_ptr(), sp)

    g = torch.cuda.CUDAGraph()
    probe = ctypes.c_void_p()
    with torch.cuda.graph(g, stream=s, capture_error_mode="relaxed"):
        can_allocate = lib.ofi_amd_gpu_mem_alloc(ctypes.byref(probe), 1 << 20) == 0
        rc = call()
    if not can_allocate:
        pytest.skip("this runtime refuses allocations during a capture")
    assert rc == 0 and lib.ofi_amd_gpu_mem_free(probe) == 0
    seeds = (2, 1)
    for step in ("call", "replay", "call", "replay"):
        if step == "call":
            assert call() == 0
        else:
            with torch.cuda.stream(s):
                g.replay()
        s.synchronize()
        want_num, want_xf, ost = _oracle.sched_batch(oracle, sizes, 4, 131072, 64, seeds)
        assert np.array_equal(_gpu.to_host(d_num, np.uint32), want_num), step
        assert np.array_equal(_gpu.to_host(d_xf, np.uint64).reshape(n, 4, 3), want_xf), step
        now = m.SchedState.from_buffer_copy(d_state.cpu().numpy().tobytes())
        seeds = (ost.rr_small_counter, ost.rr_counter)
        assert (now.rr_small_counter, now.rr_counter) == seeds, step
    assert lib.ofi_amd_sched_stream_release(sp) == 0


def test_small_batch_replayed_on_another_stream_beside_its_own_streams_batches(lib, oracle, gpu):
    """A small batch captured on one stream and replayed on another while the first stream runs small batches of
    its own (one launch each, with the same scratch): both schedulers' results and counters match the
    oracle at the end of every round, and so does the next round."""
    s, t = torch.cuda.Stream(), torch.cuda.Stream()
    sp = ctypes.c_void_p(s.cuda_stream)
    cases = []
    for n, seeds in ((3001, (2, 1)), (5000, (0, 3))):
        sizes = synthetic.stripe_sizes(n, n)
        d_state = _gpu.to_dev(np.frombuffer(bytes(m.SchedState(*seeds, 64, 131072, 4, 0)), dtype=np.uint8).copy())
        cases.append(dict(n=n, seeds=seeds, sizes=sizes, d_state=d_state, d_sizes=_gpu.to_dev(sizes),
                          d_num=torch.zeros(n, dtype=torch.int32, device="cuda"),
                          d_xf=torch.zeros(n * 12, dtype=torch.int64, device="cuda")))
    torch.cuda.synchronize()

    def call(c):
        assert lib.ofi_amd_sched_batch(c["d_state"].data_ptr(), c["d_sizes"].data_ptr(), c["n"], 128, c["d_num"].data_ptr(),
                                       c["d_xf"].data_ptr(), sp) == 0

    captured, direct = cases
    call(direct)                                    # the stream's scratch is there before the capture
    s.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s, capture_error_mode="relaxed"):
        call(captured)
    times = {3001: 0, 5000: 1}
    for _ in range(3):
        for _ in range(20):
            with torch.cuda.stream(t):
                g.replay()
            call(direct)
        times = {n: k + 20 for n, k in times.items()}
        torch.cuda.synchronize()
        for c in cases:
            ost = c["seeds"]
            for _ in range(times[c["n"]]):
                want_num, want_xf, st = _oracle.sched_batch(oracle, c["sizes"], 4, 131072, 64, ost)
                ost = (st.rr_small_counter, st.rr_counter)
            assert np.array_equal(_gpu.to_host(c["d_num"], np.uint32), want_num)
            assert np.array_equal(_gpu.to_host(c["d_xf"], np.uint64).reshape(c["n"], 4, 3), want_xf)
            now = m.SchedState.from_buffer_copy(c["d_state"].cpu().numpy().tobytes())
            assert (now.rr_small_counter, now.rr_counter) == ost
    assert lib.ofi_amd_sched_stream_release(sp) == 0
