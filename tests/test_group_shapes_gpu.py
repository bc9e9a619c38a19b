"""Compactions at the ends of their shapes: one tile, the last count of tiles
that takes one per block and the first that takes several, a last block with
few tiles, and runs that cross tiles and blocks."""
import numpy as np
import pytest

import oracle
from rccl_amd import thrust, workloads
from rccl_amd.device import DeviceBuffer

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("tile_order")]

# Items of a tile: u32 keys alone; u32 keys + 8-byte values; u64 keys + payloads + values.
TILE = {("u32", 0, False): 4_352, ("u32", 0, True): 3_328, ("u64", 8, True): 1_792}
# Tiles up to which a block takes one, four (then eight).
ONE, FOUR = 2_048, 8_192


def _runs(kind, n, longest, seed):
    """Runs of 1 to `longest` equal keys, neighbours always different."""
    length = workloads.hash_range(seed, n // max(1, longest // 2) + 2) % np.uint64(longest) + \
        np.uint64(1)
    first = np.cumsum(length)
    at = np.searchsorted(first, np.arange(n, dtype=np.uint64), side="right")
    return at.astype(oracle.KIND_DTYPES[kind])


@pytest.mark.parametrize("tiles,extra,kind,pay,reduce",
                         [(t, e, *shape) for shape in TILE
                          for t, e in ((1, -1), (1, 0), (1, 1), (ONE, 0), (ONE, 1))] +
                         [(FOUR, 1, "u32", 0, True)])
@pytest.mark.parametrize("longest", [5, 20_000])
def test_compaction_shapes(launch, tiles, extra, kind, pay, reduce, longest):
    n = tiles * TILE[(kind, pay, reduce)] + extra
    keys = _runs(kind, n, longest, n)
    starts = np.flatnonzero(np.concatenate([[True], keys[1:] != keys[:-1]]))
    ex = thrust.Execution(launch)
    k, ok = DeviceBuffer.from_host(keys), DeviceBuffer.zeroed(keys.dtype, n)
    count = DeviceBuffer.zeroed(np.uint64, 1)
    ins, outs = k, ok
    if pay:
        payload = np.arange(n, dtype=np.uint64)
        op = DeviceBuffer.zeroed(np.uint64, n)
        ins, outs = (k, DeviceBuffer.from_host(payload)), (ok, op)
    if reduce:
        vals = workloads.hash_range(3, n)
        ov = DeviceBuffer.zeroed(np.uint64, n)
        thrust.reduce_by_key(ex, ins, DeviceBuffer.from_host(vals), outs, ov, count,
                             thrust.equal, thrust.NaturalBagAdd)
        assert np.array_equal(ov.to_host_vec()[:starts.size], np.add.reduceat(vals, starts))
    else:
        thrust.unique_copy_by(ex, ins, outs, count)
    assert int(count.to_host_vec()[0]) == starts.size
    assert np.array_equal(ok.to_host_vec()[:starts.size], keys[starts])
    if pay:
        assert np.array_equal(op.to_host_vec()[:starts.size], payload[starts])
