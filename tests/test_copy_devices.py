"""Field reads in a process with contexts on two GPUs.  The built library runs
on stand-ins for the HIP runtime's calls (preloaded, host memory, two devices, a
current device per thread) that refuse, as the runtime does, an event of one
device on a stream of another.  Every read returns the bytes that were put,
whichever device is current.

What a read pins: pinning takes time a single read does not win back unless the
block is small beside it, so reads below 64 MiB pin one block of 4 MiB, larger
ones one of 32 MiB, and further reads none."""
import os
import subprocess
import sys

import pytest

from conftest import ROOT
from curvib_old_amd import _lib

STUB = r"""
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#define API extern "C" __attribute__((visibility("default")))
struct D3 { unsigned x, y, z; };
struct Obj { int dev; };               // a stream or an event
static thread_local int cur = 0;
static thread_local struct { D3 g, b; size_t sh; void *s; } cfg;
static std::map<const void *, std::string> names;
static std::mutex mu;
static long events = 0, pinned = 0, pins = 0, pin_bytes = 0;
API long stub_events() { return events; }
API long stub_pinned() { return pinned; }   // blocks of 64 KiB and more alive
API long stub_pins() { return pins; }       // and ever made
API long stub_pin_bytes() { return pin_bytes; }
API int stub_device() { return cur; }
API void **__hipRegisterFatBinary(const void *) { static void *m; return &m; }
API void __hipUnregisterFatBinary(void **) {}
API void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
API void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, D3 *, D3 *, int *) {
  names[f] = name;
}
API int __hipPushCallConfiguration(D3 g, D3 b, size_t sh, void *s) { cfg.g = g; cfg.b = b; cfg.sh = sh; cfg.s = s; return 0; }
API int __hipPopCallConfiguration(D3 *g, D3 *b, size_t *sh, void **s) { *g = cfg.g; *b = cfg.b; *sh = cfg.sh; *s = cfg.s; return 0; }
API int hipLaunchKernel(const void *f, D3, D3, void **a, size_t, void *) {
  if (names[f].find("k_copy") != std::string::npos)
    memcpy(*(double **)a[0], *(double **)a[1], *(long *)a[2] * sizeof(double));
  return 0;
}
API int hipSetDevice(int d) { if (d < 0 || d > 1) return 101; cur = d; return 0; }
API int hipGetLastError() { return 0; }
API const char *hipGetErrorString(int) { return "refused by the stand-in"; }
API int hipMalloc(void **p, size_t n) { *p = calloc(n, 1); return *p ? 0 : 2; }
API int hipFree(void *p) { free(p); return 0; }
API int hipHostMalloc(void **p, size_t n, unsigned) {
  char *q = (char *)malloc(n + 64);
  *(size_t *)q = n;
  *p = q + 64;
  std::lock_guard<std::mutex> l(mu);
  if (n >= 1 << 16) { pinned++; pins++; pin_bytes += n; }
  return 0;
}
API int hipHostFree(void *p) {
  char *q = (char *)p - 64;
  std::lock_guard<std::mutex> l(mu);
  if (*(size_t *)q >= 1 << 16) pinned--;
  free(q);
  return 0;
}
API int hipMemcpyAsync(void *d, const void *s, size_t n, int, void *) { memcpy(d, s, n); return 0; }
API int hipMemsetAsync(void *, int, size_t, void *) { return 0; }   // only fresh, zeroed memory here
API int hipPointerGetAttributes(void *, const void *) { return 1; }  // pageable memory
API int hipStreamCreateWithFlags(void **s, unsigned) { *s = new Obj{cur}; return 0; }
API int hipStreamDestroy(void *s) { delete (Obj *)s; return 0; }
API int hipStreamSynchronize(void *) { return 0; }
static int make_event(void **e) { std::lock_guard<std::mutex> l(mu); events++; *e = new Obj{cur}; return 0; }
API int hipEventCreate(void **e) { return make_event(e); }
API int hipEventCreateWithFlags(void **e, unsigned) { return make_event(e); }
API int hipEventDestroy(void *e) { std::lock_guard<std::mutex> l(mu); events--; delete (Obj *)e; return 0; }
API int hipEventRecord(void *e, void *s) { return ((Obj *)e)->dev == ((Obj *)s)->dev ? 0 : 400; }
API int hipEventSynchronize(void *) { return 0; }
"""

DRIVER = r"""
import ctypes as C, sys, threading
import numpy as np
from curvib_old_amd import _lib
from curvib_old_amd.solver import UserCtx

stub = C.CDLL(sys.argv[1])
assert _lib.load() and stub.stub_device() == 0


def context(device, seed):
    u = UserCtx((NODES,) * 3, (7, 7, 1, 1, 7, 7), 1, 100.0, 1e-3, device=device)
    z = np.random.default_rng(seed).random(u._shape("p", -1))
    assert z.nbytes >= MIN_BYTES
    u.put("p", z)
    return u, z


def read(u, z):
    assert np.array_equal(u.get("p"), z)


def in_thread(f, *a):
    bad = []

    def go():
        try:
            f(*a)
        except Exception as e:
            bad.append(e)
    t = threading.Thread(target=go)
    t.start()
    t.join()
    if bad:
        raise bad[0]


MODE = sys.argv[2]
if MODE == "other device current":      # the last call went to GPU 1
    a, b = context(0, 1), context(1, 2)
    assert stub.stub_device() == 1
    read(*a), read(*a), read(*b), read(*a)
elif MODE == "fresh thread":            # its current device is GPU 0
    a = context(1, 3)
    in_thread(read, *a), read(*a), in_thread(read, *a)
    b = None
else:                                   # either order, from threads, contexts of both devices alive
    a, b = context(1, 4), context(0, 5)
    for q in (b, a, b, a):
        in_thread(read, *q)
        read(*q)
a[0].close()
if b is not None:
    b[0].close()
assert stub.stub_pinned() == 0 and stub.stub_events() == 0, (stub.stub_pinned(), stub.stub_events())
print("reads ok")
"""


PINS = r"""
import ctypes as C, sys
import numpy as np
from curvib_old_amd import _lib
from curvib_old_amd.solver import UserCtx

stub = C.CDLL(sys.argv[1])
stub.stub_pin_bytes.restype = C.c_long
u = UserCtx((NODES,) * 3, (7, 7, 1, 1, 7, 7), 1, 100.0, 1e-3)
z = np.random.default_rng(6).random(u._shape("p", -1))
u.put("p", z)
for _ in range(3):
    assert np.array_equal(u.get("p"), z)
print("pinned", stub.stub_pins(), stub.stub_pin_bytes(), z.nbytes)
u.close()
assert stub.stub_pinned() == 0 and stub.stub_events() == 0
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    d = tmp_path_factory.mktemp("hip_stub")
    (d / "stub.cpp").write_text(STUB)
    so = d / "libhip_stub.so"
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-o", str(so), str(d / "stub.cpp")], check=True)
    return so


def run_on_stub(stub, driver, *args):
    env = dict(os.environ, PYTHONPATH=ROOT, OPENBLAS_NUM_THREADS="1")
    env["LD_PRELOAD"] = " ".join(p for p in (str(stub), env.get("LD_PRELOAD", "")) if p)
    return subprocess.run([sys.executable, "-c", driver, str(stub), *args], env=env, capture_output=True, text=True,
                          timeout=300)


@pytest.mark.skipif(not os.path.exists(_lib.SO_PATH), reason="the library is not built")
@pytest.mark.parametrize("mode", ["other device current", "fresh thread", "both devices"])
@pytest.mark.parametrize("nodes", [60, 160])    # below and above the sizes that threads move
def test_reads_of_contexts_on_two_devices(stub, mode, nodes):
    driver = DRIVER.replace("NODES", str(nodes)).replace("MIN_BYTES", str(nodes ** 3 * 8))
    r = run_on_stub(stub, driver, mode)
    assert r.returncode == 0 and "reads ok" in r.stdout, (mode, r.stdout[-500:], r.stderr[-1500:])


@pytest.mark.skipif(not os.path.exists(_lib.SO_PATH), reason="the library is not built")
@pytest.mark.parametrize("nodes", [60, 160, 330])    # by the runtime; 33 and 290 MB by threads
def test_a_read_pins_one_small_block(stub, nodes):
    r = run_on_stub(stub, PINS.replace("NODES", str(nodes)))
    assert r.returncode == 0, (r.stdout[-500:], r.stderr[-1500:])
    blocks, pinned, nbytes = (int(v) for v in r.stdout.split()[-3:])
    want = 0 if nbytes < 16 << 20 else 4 << 20 if nbytes < 64 << 20 else 32 << 20
    assert blocks == (want > 0) and pinned == want, (blocks, pinned, nbytes)
