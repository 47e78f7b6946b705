"""Field reads around the 64 MiB from which threads move chunks of 4 MiB instead of
1 MiB, at skews against both, and small, large and small reads in turn, between
which the pinned block grows.  The bytes are those that were put."""
import numpy as np
import pytest

from test_gpu_copy_edges import context, get_at

pytestmark = pytest.mark.gpu


# storage extents nodes + 1: 63.7 and 64.2 MiB
@pytest.mark.parametrize("nodes", [(140, 140, 139), (140, 140, 140)])
def test_reads_around_the_chunk_sizes(nodes):
    u, z = context(nodes)
    assert (z.nbytes >= 64 << 20) == (nodes[2] == 140)
    buf = np.empty(z.nbytes + (9 << 20), dtype=np.uint8)
    base = -buf.ctypes.data % (4 << 20)   # a chunk's first byte
    for off in (base, base + 8, base + (1 << 20) - 8, base + (1 << 20) + 16, base + (4 << 20) - 8):
        get_at(u, z, buf, off)
    u.close()


def test_the_block_grows_between_reads():
    sets = [context(n) for n in ((89, 87, 88), (140, 140, 140), (100, 90, 95))]
    for u, z in sets + sets[::-1]:
        assert np.array_equal(u.get("ucont"), z)
    for u, _ in sets:
        u.close()
