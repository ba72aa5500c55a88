"""Bounce batches of more buffers than each read their own flush word back, out of a source whose rows stay in the L2s: a
workgroup's words read back together behind kept rows, from 11,001 buffers on."""
import pytest

import test_gpu_bounce as bounce

pytestmark = bounce.pytestmark


@pytest.mark.parametrize("n", [8001, 8004, 8008, 8449, 11000, 11001, 11004, 11008, 11521])
@pytest.mark.parametrize("flush", [False, True])
def test_words_of_kept_rows_read_back_by_one_wavefront(lib, oracle, gpu, n, flush):
    """Last workgroups of one, four and eight buffers and a last run over the XCDs, with buffers outside the arena or the
    source among them, from a source just within what the rows are kept for."""
    bounce.test_forms_by_the_size_of_the_source(lib, oracle, gpu, 31, n, flush)
