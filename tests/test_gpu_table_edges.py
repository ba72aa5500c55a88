"""GPU parity of the table copy by pieces at the edges of its pieces, which lie on 64-byte boundaries of the destination."""
import numpy as np
import pytest
import torch

import _gpu

pytestmark = pytest.mark.gpu
PIECE = 8192
LENS = [0, 1, 63, 64, PIECE - 64, PIECE - 1, PIECE, PIECE + 1, PIECE + 63, PIECE + 64, 2 * PIECE - 1, 2 * PIECE, 2 * PIECE + 1,
        3 * PIECE + 62, 9 * PIECE + 5]


@pytest.mark.parametrize("skew", [0, 1, 40, 63])
@pytest.mark.parametrize("src_skew", [0, 1, 2, 7, 12])
@pytest.mark.parametrize("max_len", [max(LENS), 200 * PIECE, 1024 * PIECE])
def test_pieces_of_an_entry_meet_without_a_gap(lib, gpu, skew, src_skew, max_len):
    """Every byte of an entry once, none beside it, from any source alignment to any destination alignment; each way of
    dealing pieces out."""
    room = 11 * PIECE
    gen = np.random.default_rng(skew * 100 + src_skew)
    src = gen.integers(0, 256, room * len(LENS), dtype=np.uint8)
    want = gen.integers(0, 256, room * len(LENS), dtype=np.uint8)
    d_src, d_dst = _gpu.to_dev(src), _gpu.to_dev(want)
    at = np.arange(len(LENS), dtype=np.uint64) * np.uint64(room)
    s_at, d_at, lens = at + np.uint64(128 + src_skew), at + np.uint64(128 + skew), np.array(LENS, dtype=np.uint32)
    tables = [_gpu.to_dev(s_at + np.uint64(d_src.data_ptr())), _gpu.to_dev(d_at + np.uint64(d_dst.data_ptr())), _gpu.to_dev(lens)]
    assert lib.ofi_amd_copy_table_pieces(*[t.data_ptr() for t in tables], len(LENS), max_len, _gpu.stream()) == 0
    torch.cuda.synchronize()
    for s, d, n in zip(s_at.astype(int), d_at.astype(int), LENS):
        want[d:d + n] = src[s:s + n]
    assert np.array_equal(d_dst.cpu().numpy().view(np.uint8), want)
    assert _gpu.fetch_async_errors(lib) == 0
