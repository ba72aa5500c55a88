"""Eager arrivals out of rx buffers in host memory: batches on both sides of the line between the kernels, last workgroups of
one to four buffers, payloads on both sides of the length from which wavefronts take turns, none at all, and a graph."""
import ctypes

import numpy as np
import pytest
import torch

import _gpu
import test_gpu_eager_copy as eager

pytestmark = eager.pytestmark
EDGES = np.array([0, 1, 3, 4, 1023, 1024, 1025, 8184], dtype=np.uint32)


def host_case(oracle, n, max_len):
    rng = np.random.default_rng(n + max_len)
    rx, rx_off, recv_len, dst_off, dst_len, arena_bytes = eager.make_case(rng, n, max_len)
    if max_len > EDGES.max() - 1:                 # some at the edges, where the destination has room for them
        edges = rng.choice(EDGES, n)
        recv_len = np.where(rng.random(n) < 0.5, np.minimum(edges, recv_len), recv_len).astype(np.uint32)
    want = eager.expected(oracle, rx, rx_off, recv_len, dst_off, dst_len, arena_bytes, 0x5A)
    return torch.from_numpy(rx).pin_memory(), (rx_off, recv_len, dst_off, dst_len, arena_bytes), want


@pytest.mark.parametrize("n", [1, 127, 128, 129, 130, 131, 1500])
@pytest.mark.parametrize("max_len", [40, 8184])
def test_rx_buffers_in_host_memory(lib, oracle, gpu, n, max_len):
    rx, case, want = host_case(oracle, n, max_len)
    for base in (0, 3):
        got = eager.run_gpu(lib, rx.data_ptr(), *case, 0x5A, base_offset=base)
        for g, w in zip(got, want):
            assert np.array_equal(g, w)
    got = eager.run_gpu(lib, rx.data_ptr(), *case, 0x5A, want_flush=False)
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])


@pytest.mark.parametrize("n", [100, 702])
def test_rx_buffers_in_host_memory_in_a_graph(lib, oracle, gpu, n):
    rx, (rx_off, recv_len, dst_off, dst_len, arena_bytes), want = host_case(oracle, n, 8184)
    arena = torch.full((arena_bytes,), 0x5A, dtype=torch.uint8, device="cuda")
    table = [_gpu.to_dev(x) for x in (rx_off, recv_len, dst_off, dst_len)]
    copied, flush = (torch.zeros(n, dtype=torch.int32, device="cuda") for _ in range(2))
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        rc = lib.ofi_amd_eager_copy_batch(rx.data_ptr(), table[0].data_ptr(), table[1].data_ptr(), arena.data_ptr(),
                                          table[2].data_ptr(), table[3].data_ptr(), n, copied.data_ptr(), flush.data_ptr(),
                                          ctypes.c_void_p(stream.cuda_stream))
    assert rc == 0
    for _ in range(3):
        arena.fill_(0x5A)
        copied.zero_()
        flush.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for got, w in zip((arena, copied, flush), want):
            assert np.array_equal(_gpu.to_host(got, w.dtype), w)
