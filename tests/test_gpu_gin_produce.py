"""GPU parity: the seeded GIN producer at the lines where a context gets fewer wavefronts and at the edges of their groups."""
import numpy as np
import pytest

from test_gpu_gin import drain_descs, make_rings, oracle_stream, produce_and_drain, SEED
import _gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nctx", [15, 16, 31, 32])
@pytest.mark.parametrize("ops", [1, 63, 65, 193, 700])
def test_groups_of_few_and_many_contexts(lib, oracle, gpu, nctx, ops):
    """Launch after launch on rings that wrap: full groups and short ones, slots seen free ahead and slots waited for."""
    rings = make_rings(lib, nctx, 256)
    want = oracle_stream(oracle, nctx, ops, 64, 1, 1)
    for _ in range(3):
        rc, stats, descs, _ = produce_and_drain(lib, rings, nctx, ops, mode=1)
        assert rc == 0 and stats.descriptors == nctx * ops and lib.ofi_amd_gin_producer_status(rings) == 0
        assert np.array_equal(np.frombuffer(descs, dtype=np.uint64).reshape(nctx, ops, 8), want)
    lib.ofi_amd_gin_rings_destroy(rings)


@pytest.mark.parametrize("nctx", [2, 40])
def test_no_slot_is_taken_that_is_not_free(lib, oracle, gpu, nctx):
    """A ring that still holds 100 descriptors has room for two groups more; the third is waited for and given up on."""
    rings = make_rings(lib, nctx, 256)
    assert lib.ofi_amd_gin_produce_seeded(rings, SEED, 100, 1, 64, 1, 1, 0, _gpu.stream()) == 0
    assert lib.ofi_amd_gin_produce_seeded(rings, SEED, 1000, 1, 64, 1, 1, 50, _gpu.stream()) == 0
    _gpu.sync()
    assert lib.ofi_amd_gin_producer_status(rings) != 0
    rc, stats, got = drain_descs(lib, rings, nctx, 228)
    assert rc == 0 and stats.descriptors == nctx * 228
    want = oracle_stream(oracle, nctx, 128, 64, 1, 1)
    assert np.array_equal(got[:, :100], want[:, :100]) and np.array_equal(got[:, 100:], want)
    lib.ofi_amd_gin_rings_destroy(rings)
