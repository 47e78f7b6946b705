"""Fields read back to the host: sizes below, at and past the 16 MiB from which
threads move 4 MiB chunks, host arrays at every skew against those chunks, an
address that is no multiple of 8, pinned memory, and two contexts at once.  The
bytes are those that were put, and no byte beside them changes."""
import ctypes as C
import threading

import numpy as np
import pytest

from curvib_old_amd import _lib
from curvib_old_amd.solver import UserCtx

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def context(nodes):
    u = UserCtx(nodes, (7, 7, 1, 1, 7, 7), 1, 100.0, 1e-3)
    z = np.arange(np.prod(u._shape("ucont", -1)), dtype=np.float64).reshape(u._shape("ucont", -1))
    u.put("ucont", z)
    return u, z


def get_at(u, z, buf, off):
    """ucont into buf (bytes) at off; the bytes around keep their value"""
    buf[:] = 0x5A
    rc = _lib.load().cv_get_field(u.h, _lib.FIELD_ID["ucont"], -1,
                                  C.cast(buf.ctypes.data + off, C.POINTER(C.c_double)))
    assert rc == _lib.CV_OK, _lib.last_error()
    assert bytes(buf[off:off + z.nbytes]) == z.tobytes()
    assert (buf[:off] == 0x5A).all() and (buf[off + z.nbytes:] == 0x5A).all()


# storage extents nodes + 1; 24 bytes a point: under 16 MiB, just past it, several
# chunks
@pytest.mark.parametrize("nodes", [(86, 87, 90), (89, 87, 88), (127, 99, 96)])
def test_field_reads_keep_their_bytes(nodes):
    u, z = context(nodes)
    assert (z.nbytes >= 16 << 20) == (nodes[0] != 86)
    buf = np.empty(z.nbytes + (9 << 20), dtype=np.uint8)
    base = -buf.ctypes.data % (4 << 20)   # a chunk's first byte
    for off in (base, base + 8, base + (4 << 20) - 8, base + (2 << 20) + 24, base + 4, base + 3):
        get_at(u, z, buf, off)
    pin = torch.empty(z.nbytes + 16, dtype=torch.uint8, pin_memory=True).numpy()
    get_at(u, z, pin, 8)
    u.close()


def test_two_contexts_read_at_once():
    pairs = [context((127, 99, 96)), context((99, 127, 97))]
    bad = []

    def reads(u, z):
        for _ in range(4):
            if not np.array_equal(u.get("ucont"), z):
                bad.append(z.shape)

    th = [threading.Thread(target=reads, args=p) for p in pairs]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad
    for u, _ in pairs:   # the last one gives the buffers back; the next context makes its own
        u.close()
    u, z = context((127, 99, 96))
    reads(u, z)
    u.close()
    assert not bad
