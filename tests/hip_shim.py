"""A library that stands between libonegraph and the HIP runtime in a child
process: it can refuse pinned or device allocations by size, leave a launch out
and report an error for a stream's state, and it counts what the calls did.
Nothing it does reaches the GPU: such calls end on the host, all others go to
the runtime as they are."""
import os
import subprocess
import sys
import textwrap

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#define _GNU_SOURCE
#include <dlfcn.h>
#include <pthread.h>
#include <stdatomic.h>
#include <stddef.h>
static void *real(const char *name) {
    static void *h;
    if (!h) h = dlopen("libamdhip64.so.7", RTLD_LAZY);
    if (!h) h = dlopen("/opt/rocm/lib/libamdhip64.so.7", RTLD_LAZY);
    return dlsym(h, name);
}
typedef struct { size_t lo, hi; } Range;
static Range deny_pin = {1, 0}, deny_dev = {1, 0};
static atomic_long fills_null, fills_stream, denied, live_pin, live_dev;
static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;
static struct { void *p; size_t n; int pin; } rec[1 << 14];
static void note(void *p, size_t n, int pin) {
    pthread_mutex_lock(&mu);
    for (int i = 0; i < 1 << 14; ++i)
        if (!rec[i].p) { rec[i].p = p; rec[i].n = n; rec[i].pin = pin; break; }
    pthread_mutex_unlock(&mu);
    atomic_fetch_add(pin ? &live_pin : &live_dev, (long)n);
}
static void drop(void *p) {
    pthread_mutex_lock(&mu);
    for (int i = 0; p && i < 1 << 14; ++i)
        if (rec[i].p == p) {
            rec[i].p = NULL;
            atomic_fetch_sub(rec[i].pin ? &live_pin : &live_dev, (long)rec[i].n);
            break;
        }
    pthread_mutex_unlock(&mu);
}
int hipHostMalloc(void **p, size_t n, unsigned flags) {
    if (n >= deny_pin.lo && n <= deny_pin.hi) { atomic_fetch_add(&denied, 1); *p = NULL; return 2; }
    int e = ((int (*)(void **, size_t, unsigned))real("hipHostMalloc"))(p, n, flags);
    if (!e) note(*p, n, 1);
    return e;
}
int hipHostFree(void *p) { drop(p); return ((int (*)(void *))real("hipHostFree"))(p); }
int hipMalloc(void **p, size_t n) {
    if (n >= deny_dev.lo && n <= deny_dev.hi) { atomic_fetch_add(&denied, 1); *p = NULL; return 2; }
    int e = ((int (*)(void **, size_t))real("hipMalloc"))(p, n);
    if (!e) note(*p, n, 0);
    return e;
}
int hipFree(void *p) { drop(p); return ((int (*)(void *))real("hipFree"))(p); }
int hipMemset(void *p, int v, size_t n) {
    atomic_fetch_add(&fills_null, 1);
    return ((int (*)(void *, int, size_t))real("hipMemset"))(p, v, n);
}
int hipMemsetAsync(void *p, int v, size_t n, void *s) {
    atomic_fetch_add(s ? &fills_stream : &fills_null, 1);
    return ((int (*)(void *, int, size_t, void *))real("hipMemsetAsync"))(p, v, n, s);
}
int shim_pinned_has(size_t n) {
    int has = 0;
    pthread_mutex_lock(&mu);
    for (int i = 0; i < 1 << 14; ++i) has |= rec[i].p && rec[i].pin && rec[i].n == n;
    pthread_mutex_unlock(&mu);
    return has;
}
typedef struct { unsigned x, y, z; } Dim;
static atomic_int query_error;
static unsigned skip_grid, skip_block;
int hipStreamQuery(void *s) {
    if (atomic_load(&query_error)) return 999;
    return ((int (*)(void *))real("hipStreamQuery"))(s);
}
int hipLaunchKernel(const void *f, Dim g, Dim b, void **a, size_t lds, void *s) {
    if (skip_grid && g.x == skip_grid && b.x == skip_block) return 0;
    return ((int (*)(const void *, Dim, Dim, void **, size_t, void *))real("hipLaunchKernel"))(f, g, b, a, lds, s);
}
void shim_query_error(int on) { atomic_store(&query_error, on); }
void shim_skip_launch(unsigned grid, unsigned block) { skip_grid = grid; skip_block = block; }
void shim_deny_pinned(size_t lo, size_t hi) { deny_pin.lo = lo; deny_pin.hi = hi; }
void shim_deny_device(size_t lo, size_t hi) { deny_dev.lo = lo; deny_dev.hi = hi; }
long shim_denied(void) { return atomic_load(&denied); }
long shim_fills_null(void) { return atomic_load(&fills_null); }
long shim_fills_stream(void) { return atomic_load(&fills_stream); }
long shim_live_pinned(void) { return atomic_load(&live_pin); }
long shim_live_device(void) { return atomic_load(&live_dev); }
"""

HEAD = """
import ctypes as C, sys
shim = C.CDLL({so!r}, mode=C.RTLD_GLOBAL)   # before the library is loaded: its calls come here
shim.shim_deny_pinned.argtypes = shim.shim_deny_device.argtypes = [C.c_size_t, C.c_size_t]
for name in ("denied", "fills_null", "fills_stream", "live_pinned", "live_device"):
    getattr(shim, "shim_" + name).restype = C.c_long
shim.shim_pinned_has.argtypes = [C.c_size_t]
sys.path.insert(0, {root!r})
import numpy as np
import onegraph_amd as og
import oracle
assert og.device_count() > 0
"""


def run(tmp_path, *code, timeout=100):
    """Runs the pieces of code (each with an indent of its own) in a child whose
    library calls go through the shim.  Its asserts fail the test."""
    src, so = str(tmp_path / "shim.c"), str(tmp_path / "shim.so")
    with open(src, "w") as f:
        f.write(SOURCE)
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", so, src, "-ldl", "-lpthread"], check=True)
    text = "\n".join([HEAD.format(so=so, root=ROOT)] + [textwrap.dedent(c) for c in code] + ["print('done')"])
    r = subprocess.run([sys.executable, "-u", "-c", text], capture_output=True, text=True, timeout=timeout, cwd=ROOT)
    assert r.returncode == 0 and r.stdout.endswith("done\n"), r.stdout + r.stderr
