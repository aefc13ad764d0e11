"""A stand-in for the HIP runtime, for tests of what the library does around
its GPU calls (allocation failures, lifetimes) on the CPU: it counts and
orders the calls and runs nothing.  Loaded ahead of the library's own runtime
(RTLD_GLOBAL) in a process of its own."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "fortrancfd_amd", "libfcfd.so")

SOURCE = r"""
#include <stddef.h>
#include <stdlib.h>
typedef struct { unsigned x, y, z; } d3;
static int calls, fail_at, live, launches;
static long seq, launched, synced;          /* order of graph launches and stream synchronisations */
static int destroyed, early;                /* graphs destroyed, of them with a launch not waited for */
static double *host[64];
static int nhost;
static int hit(void) { return ++calls == fail_at; }
void standin_reset(int n) { calls = live = launches = 0; fail_at = n; }
int standin_live(void) { return live; }
int standin_launches(void) { return launches; }
int standin_graph_launches(void) { return launched > 0; }
int standin_destroyed(void) { return destroyed; }
int standin_destroyed_early(void) { return early; }

int hipMalloc(void **p, size_t n) { (void)n; if (hit()) return 2; *p = malloc(16); ++live; return 0; }
int hipMemcpy(void *d, const void *s, size_t n, int k) { (void)d; (void)s; (void)n; (void)k; return hit() ? 1 : 0; }
int hipFree(void *p) { free(p); --live; return 0; }
int hipHostMalloc(void **p, size_t n, unsigned f) { (void)f; *p = calloc(1, n + 8); if (nhost < 64) host[nhost++] = *p; return 0; }
int hipHostFree(void *p) { (void)p; return 0; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *st) { (void)d; (void)s; (void)n; (void)k; (void)st; return 0; }
int hipMemset(void *d, int v, size_t n) { (void)d; (void)v; (void)n; return 0; }
int hipMemsetAsync(void *d, int v, size_t n, void *st) { (void)d; (void)v; (void)n; (void)st; return 0; }
int hipGetSymbolAddress(void **p, const void *s) { (void)s; *p = malloc(16); return 0; }
int hipGetDevice(int *d) { *d = 0; return 0; }
int hipSetDevice(int d) { (void)d; return 0; }
int hipDeviceGetAttribute(int *v, int a, int d) { (void)a; (void)d; *v = 256; return 0; }
int hipGetLastError(void) { return 0; }
const char *hipGetErrorString(int e) { (void)e; return "stand-in"; }
int hipStreamCreate(void **s) { *s = malloc(16); return 0; }
int hipStreamDestroy(void *s) { (void)s; return 0; }
int hipStreamSynchronize(void *s) { (void)s; synced = ++seq; return 0; }
int hipEventCreate(void **e) { *e = malloc(16); return 0; }
int hipEventCreateWithFlags(void **e, unsigned f) { (void)f; *e = malloc(16); return 0; }
int hipEventDestroy(void *e) { (void)e; return 0; }
int hipEventRecord(void *e, void *s) { (void)e; (void)s; return 0; }
int hipEventElapsedTime(float *t, void *a, void *b) { (void)a; (void)b; *t = 0; return 0; }
/* a waited-for status says that the first case has ended */
int hipEventSynchronize(void *e) { (void)e; for (int q = 0; q < nhost; ++q) host[q][0] = 1.0; return 0; }
int hipStreamBeginCapture(void *s, int m) { (void)s; (void)m; return 0; }
int hipStreamEndCapture(void *s, void **g) { (void)s; *g = malloc(16); return 0; }
int hipGraphInstantiate(void **x, void *g, void *n, char *l, size_t b) { (void)g; (void)n; (void)l; (void)b; *x = malloc(16); return 0; }
int hipGraphDestroy(void *g) { free(g); return 0; }
int hipGraphLaunch(void *x, void *s) { (void)x; (void)s; launched = ++seq; return 0; }
int hipGraphExecDestroy(void *x) { free(x); ++destroyed; early += launched > synced; return 0; }
int __hipPushCallConfiguration(d3 g, d3 b, size_t s, void *st) { (void)g; (void)b; (void)s; (void)st; return 0; }
int __hipPopCallConfiguration(d3 *g, d3 *b, size_t *s, void **st) { d3 o = {1, 1, 1}; *g = *b = o; *s = 0; *st = 0; return 0; }
int hipLaunchKernel(const void *f, d3 g, d3 b, void **a, size_t s, void *st) {
    (void)f; (void)g; (void)b; (void)a; (void)s; (void)st;
    ++launches;
    return 0;
}
"""

HEAD = r"""
import ctypes as C, sys
sys.path.insert(0, sys.argv[1])
hip = C.CDLL(sys.argv[2], mode=C.RTLD_GLOBAL)   # ahead of the library's own HIP runtime
lib = C.CDLL(sys.argv[3])
from fortrancfd_amd.types import Case
vp = C.c_void_p
"""


def run(tmp_path, body: str) -> None:
    """HEAD + body, which prints "done" at its end"""
    src, so = tmp_path / "standin.c", tmp_path / "standin.so"
    src.write_text(SOURCE)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-o", str(so), str(src)], check=True)
    r = subprocess.run([sys.executable, "-c", HEAD + body, ROOT, str(so), LIB], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "done", r.stdout + r.stderr
