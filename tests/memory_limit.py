"""Device memory under a limit: code run in a process of its own, in which
hipMalloc refuses what would take the live blocks past a byte budget.

The library's calls are bound to the limiter because it is loaded before the
library and for everyone; nothing is filled up to make memory short."""
import os
import subprocess
import sys

LIMITER = r"""
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
#define SLOTS 65536
static void *ptr[SLOTS];
static size_t len[SLOTS];
static long long live, peak, budget = -1;
static int pinned_off;
long long limit_live(void) { return live; }
long long limit_peak(int reset) { long long p = peak; if (reset) peak = live; return p; }
void limit_set(long long bytes) { budget = bytes; }
void limit_no_pinned(int off) { pinned_off = off; }
int hipMalloc(void **p, size_t n) {
    static int (*real)(void **, size_t);
    if (!real) real = (int (*)(void **, size_t))dlsym(RTLD_NEXT, "hipMalloc");
    if (budget >= 0 && live + (long long)n > budget) return 2; /* hipErrorOutOfMemory */
    int e = real(p, n);
    for (int i = 0; e == 0 && i < SLOTS; i++)
        if (!ptr[i]) {
            ptr[i] = *p;
            len[i] = n;
            live += (long long)n;
            if (live > peak) peak = live;
            break;
        }
    return e;
}
int hipFree(void *p) {
    static int (*real)(void *);
    if (!real) real = (int (*)(void *))dlsym(RTLD_NEXT, "hipFree");
    for (int i = 0; p && i < SLOTS; i++)
        if (ptr[i] == p) {
            ptr[i] = NULL;
            live -= (long long)len[i];
            break;
        }
    return real(p);
}
int hipHostMalloc(void **p, size_t n, unsigned flags) {
    static int (*real)(void **, size_t, unsigned);
    if (!real) real = (int (*)(void **, size_t, unsigned))dlsym(RTLD_NEXT, "hipHostMalloc");
    if (pinned_off) return 2;
    return real(p, n, flags);
}
"""

HEAD = """
import ctypes, sys
limit = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
limit.limit_live.restype = limit.limit_peak.restype = ctypes.c_longlong
limit.limit_set.argtypes = [ctypes.c_longlong]
sys.path[:0] = sys.argv[2:]
import numpy as np
import tilespgemm as ts
from tsg_check import log
"""


def run_limited(tmp_path, code, timeout=100):
    """Runs `code` after HEAD; it has `limit`, `ts`, `np` and `log`."""
    src, lib = tmp_path / "limit.c", tmp_path / "limit.so"
    src.write_text(LIMITER)
    subprocess.check_call(["gcc", "-O1", "-shared", "-fPIC", str(src), "-o", str(lib), "-L/opt/rocm/lib",
                           "-Wl,--no-as-needed", "-lamdhip64", "-Wl,-rpath,/opt/rocm/lib", "-ldl"])
    here = os.path.dirname(os.path.abspath(__file__))
    root = os.path.dirname(here)
    prog = tmp_path / "run.py"
    prog.write_text(HEAD + code)
    r = subprocess.run([sys.executable, "-u", str(prog), str(lib), os.path.join(root, "rw-spgemm_amd"), here,
                        os.path.join(root, "oracle")], timeout=timeout, capture_output=True, text=True)
    print(r.stdout[-3000:], r.stderr[-3000:], flush=True)
    assert r.returncode == 0
