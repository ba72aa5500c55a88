"""Eager batches whose workgroups read their buffers' first bytes back together: last workgroups of one to four buffers,
last runs over the XCDs, buffers of fewer bytes than are read back, neighbours in one line, with and without counts."""
import numpy as np
import pytest

import _gpu
import test_gpu_eager_copy as eager

pytestmark = eager.pytestmark


@pytest.mark.parametrize("n", [9001, 9002, 9003, 9004, 9216, 9217])
@pytest.mark.parametrize("max_len", [6, 300])
def test_first_bytes_read_back_by_one_wavefront_of_a_workgroup(lib, oracle, gpu, n, max_len):
    rng = np.random.default_rng(n + max_len)
    rx, rx_off, recv_len, dst_off, dst_len, arena_bytes = eager.make_case(rng, n, max_len)
    want = eager.expected(oracle, rx, rx_off, recv_len, dst_off, dst_len, arena_bytes, 0x5A)
    d_rx = _gpu.to_dev(rx)
    for base in (0, 3):
        got = eager.run_gpu(lib, d_rx.data_ptr(), rx_off, recv_len, dst_off, dst_len, arena_bytes, 0x5A, base_offset=base)
        for g, w in zip(got, want):
            assert np.array_equal(g, w)
