"""Counted set operations (no output): one block, the ends of a look-back
group of 64 blocks, several groups, against the counts that numpy gives; each
workspace is used twice."""
import numpy as np
import pytest

from rccl_amd import cub
from rccl_amd.device import DeviceBuffer

pytestmark = pytest.mark.gpu

# Items of a small tile's block, for 4- and 8-byte keys.
TILE = 512 * 16


@pytest.mark.parametrize("dtype", [np.uint32, np.uint64])
@pytest.mark.parametrize("total", [1, TILE, TILE + 1, 63 * TILE, 64 * TILE, 64 * TILE + 1,
                                   65 * TILE, 400 * TILE + 3, 5_000_011, 40_000_003])
def test_set_counts(launch, tile_order, dtype, total):
    na = total // 3
    a = np.arange(na, dtype=dtype) * dtype(3)
    b = np.arange(total - na, dtype=dtype) * dtype(2)
    # Both hold the multiples of 6 below the smaller end.
    both = -(-min(na * 3, (total - na) * 2) // 6)
    want = {"union": total - both, "intersection": both, "difference": na - both,
            "symmetric_difference": total - 2 * both}
    da, db = DeviceBuffer.from_host(a), DeviceBuffer.from_host(b)
    for op, count in want.items():
        ws = cub.device_set_workspace(launch, op, dtype, na, total - na)
        for _ in range(2):
            ws.output_count.copy_from(DeviceBuffer.from_host(np.array([2**63], dtype=np.uint64)))
            cub.device_set_keys(launch, op, da, db, ws, None)
            launch.synchronize()
            assert ws.count() == count, op
