"""Record sort where the number of byte positions that vary reaches and passes
the launches of their own (2N), at both tile sizes, against numpy's lexsort."""
import numpy as np
import pytest

from rccl_amd import record_sort, thrust, workloads
from rccl_amd.device import DeviceBuffer

pytestmark = pytest.mark.gpu


def _rows(arity, n, varying):
    """n rows whose low `varying` byte positions (last column first) vary."""
    cols = []
    for c in range(arity):
        place = 4 * (arity - 1 - c)  # byte position of the column's low byte
        k = min(4, max(0, varying - place))
        mask = (1 << (8 * k)) - 1
        h = workloads.hash_range(101 * c + n, n) >> np.uint64(17)
        cols.append((h & np.uint64(mask)).astype(np.uint32) | np.uint32(0x01020304 & ~mask))
    return np.stack(cols, 1)


@pytest.mark.parametrize("arity", [2, 4, 6])
@pytest.mark.parametrize("extra", [-1, 0, 1, 2, "all"])
@pytest.mark.parametrize("n", [65_536, (1 << 19) - 1, 1 << 19])
@pytest.mark.parametrize("in_place", [False, True])
def test_active_passes_around_own_launches(launch, radix_ranking, arity, extra, n, in_place):
    if n > 65_536 and (arity != 4 or extra in (-1, 2)):
        pytest.skip("tile sizes are compared at one arity")
    varying = 4 * arity if extra == "all" else 2 * arity + extra
    host = _rows(arity, n, varying)
    pay = np.arange(n, dtype=np.uint64)
    order = np.lexsort(host.T[::-1])
    ex = thrust.Program.load(0).par(launch.stream())
    rows, payload = record_sort.RowBuffer.from_host(host), DeviceBuffer.from_host(pay)
    if in_place:
        record_sort.sort_rows_with_payload_lexicographic(ex, rows, payload)
        out, outp = rows, payload
    else:
        out, outp = record_sort.RowBuffer.zeroed(arity, n), DeviceBuffer.zeroed(np.uint64, n)
        record_sort.sort_rows_with_payload_lexicographic_into(ex, rows, payload, out, outp)
        assert np.array_equal(rows.to_host_vec(), host)
    assert np.array_equal(outp.to_host_vec(), pay[order])
    assert np.array_equal(out.to_host_vec(), host[order])
