"""GPU parity of the striping form in which a tile adds up what the tiles before it have published, against the CPU oracle:
its smallest and largest batches, with and without waiting for the others."""
import ctypes

import numpy as np
import pytest
import torch

import _gpu
import _oracle
import aws_ofi_nccl_amd as m
from aws_ofi_nccl_amd import synthetic

pytestmark = pytest.mark.gpu
TILE = 512


def dev_state(rails, min_stripe, max_small, seeds):
    st = m.SchedState(seeds[0], seeds[1], max_small, min_stripe, rails, 0)
    return _gpu.to_dev(np.frombuffer(bytes(st), dtype=np.uint8).copy())


def messages(seed, n):
    sizes = synthetic.stripe_sizes(seed, n)
    sizes[::5] = sizes[::5] % np.uint64(200)
    return sizes


class Chain:
    """Batches of one scheduler, queued in a row, and what the oracle makes of them."""

    def __init__(self, n, count, rails, max_small, seed):
        self.n, self.rails, self.max_small = n, rails, max_small
        self.seeds = (rails - 1, rails // 2)
        self.sizes = [messages(seed + k, n) for k in range(count)]
        self.d_state = dev_state(rails, 100000, max_small, self.seeds)
        self.d_sizes = [_gpu.to_dev(s) for s in self.sizes]
        self.out = [(torch.full((n,), -1, dtype=torch.int32, device="cuda"),
                     torch.full((n * 12,), -1, dtype=torch.int64, device="cuda")) for _ in range(count)]

    def queue(self, call, k, stream):
        num, xf = self.out[k]
        assert call(self.d_state.data_ptr(), self.d_sizes[k].data_ptr(), self.n, 128, num.data_ptr(), xf.data_ptr(), stream) == 0

    def check(self, oracle):
        seeds = self.seeds
        for k, (num, xf) in enumerate(self.out):
            want_num, want_xf, ost = _oracle.sched_batch(oracle, self.sizes[k], self.rails, 100000, self.max_small, seeds)
            seeds = (ost.rr_small_counter, ost.rr_counter)
            assert np.array_equal(_gpu.to_host(num, np.uint32), want_num), k
            assert np.array_equal(_gpu.to_host(xf, np.uint64).reshape(self.n, 4, 3), want_xf), k
        st = m.SchedState.from_buffer_copy(self.d_state.cpu().numpy().tobytes())
        assert (st.rr_small_counter, st.rr_counter) == seeds
        assert (st.max_small_msg_size, st.min_stripe_size, st.num_rails) == (self.max_small, 100000, self.rails)


# the smallest batches, with whole and ragged last tiles, both sides of a wavefront's share of the words, the largest batch
# and the one after it
@pytest.mark.parametrize("n", [9984, 9985, 10240, 10241, 20 * TILE + 513, 64 * TILE, 64 * TILE + 1, 65 * TILE + 1,
                               TILE * TILE - 1, TILE * TILE, TILE * TILE + 1])
@pytest.mark.parametrize("rails,max_small", [(4, 64), (3, 5000), (1, 0)])
def test_batches_of_published_totals(lib, oracle, gpu, n, rails, max_small):
    """Three in a row without a wait between them: each starts from the counters the one before has moved on, and none
    takes a word of another for its own."""
    chain = Chain(n, 3, rails, max_small, n + rails)
    for k in range(3):
        chain.queue(lib.ofi_amd_sched_batch, k, _gpu.stream())
    _gpu.sync()
    chain.check(oracle)
    assert _gpu.fetch_async_errors(lib) == 0


@pytest.mark.parametrize("looks", [0, 1])
@pytest.mark.parametrize("n", [9985, 10241, 65 * TILE + 1, TILE * TILE])
@pytest.mark.parametrize("rails,max_small", [(4, 64), (3, 5000)])
def test_tiles_that_do_not_wait_add_up_by_themselves(lib, oracle, gpu, n, rails, max_small, looks):
    """What a tile does that has looked for the others' words in vain, for all of them and for those that one look finds
    incomplete, between batches that wait."""
    call = lib.ofi_amd_sched_batch_looks
    call.argtypes = [ctypes.c_void_p] * 2 + [ctypes.c_uint64] * 2 + [ctypes.c_void_p] * 3 + [ctypes.c_uint32]
    chain = Chain(n, 4, rails, max_small, 7 * n + rails)
    for k in range(4):
        chain.queue(lambda *a: call(*a, looks) if k % 2 else lib.ofi_amd_sched_batch(*a), k, _gpu.stream())
    _gpu.sync()
    chain.check(oracle)
    assert _gpu.fetch_async_errors(lib) == 0


def test_several_streams_at_once_and_the_fixed_scratch(lib, oracle, gpu):
    """Four schedulers on four streams, whose tiles run between each other's, each with scratch of its own; then the entry point
    that allocates nothing, small batches and larger forms between."""
    streams = [torch.cuda.Stream() for _ in range(4)]
    chains = [Chain(n, 3, rails, 64, 100 + rails) for n, rails in ((200_001, 4), (150_003, 3), (262_144, 2), (99_999, 1))]
    torch.cuda.synchronize()
    for k in range(3):
        for s, chain in zip(streams, chains):
            chain.queue(lib.ofi_amd_sched_batch, k, ctypes.c_void_p(s.cuda_stream))
    torch.cuda.synchronize()
    for s, chain in zip(streams, chains):
        chain.check(oracle)
        assert lib.ofi_amd_sched_stream_release(ctypes.c_void_p(s.cuda_stream)) == 0
    assert lib.ofi_amd_gpu_init() == 0
    for n in (30_001, 700, 400_001, 262_144, 12_000):
        chain = Chain(n, 2, 4, 64, n)
        for k in range(2):
            chain.queue(lib.ofi_amd_sched_batch_noalloc, k, _gpu.stream())
        _gpu.sync()
        chain.check(oracle)
    assert _gpu.fetch_async_errors(lib) == 0


@pytest.mark.parametrize("n", [50_000, 300_000, 6_300_000])
def test_an_unusable_state_ends_every_tile(lib, gpu, n):
    for rails, min_stripe in [(5, 131072), (0, 131072), (4, 0)]:
        d_state = dev_state(rails, min_stripe, 64, (0, 0))
        d_sizes = _gpu.to_dev(messages(1, n))
        num = torch.full((n,), -1, dtype=torch.int32, device="cuda")
        xf = torch.full((n * 12,), -1, dtype=torch.int64, device="cuda")
        assert lib.ofi_amd_sched_batch(d_state.data_ptr(), d_sizes.data_ptr(), n, 128, num.data_ptr(), xf.data_ptr(),
                                       _gpu.stream()) == 0
        _gpu.sync()
        assert int(num.max()) == -1 and int(xf.max()) == -1 and _gpu.fetch_async_errors(lib) & 4
