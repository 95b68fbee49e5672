"""The host driver against a HIP runtime that is not there: the built library
is loaded beside a small stand-in for libamdhip64 (allocations from the heap,
copies by memcpy, launches that do nothing), in a process of its own, so that
failures can be made at chosen calls.  No GPU code runs here."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "diffeqflux.jl_amd", "diffeqflux_hip", "libnode_hip.so")

STUB = r"""
#include <stdlib.h>
#include <string.h>
long stub_mallocs, stub_live, stub_fail_at = -1, stub_attrs, stub_attr_changes;
static int last;
static const void* fn[256]; static int val[256], nfn;
#define OK(name) int name() { return 0; }
int hipMalloc(void** p, size_t n) {
  *p = 0;
  if (stub_mallocs++ == stub_fail_at) return last = 2;
  *p = calloc(1, n); ++stub_live; return 0;
}
int hipFree(void* p) { if (p) { free(p); --stub_live; } return 0; }
int hipHostMalloc(void** p, size_t n, unsigned f) { *p = calloc(1, n); return 0; }
int hipHostFree(void* p) { free(p); return 0; }
int hipMemsetAsync(void* p, int v, size_t n, void* s) { memset(p, v, n); return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int k, void* st) { memcpy(d, s, n); return 0; }
int hipGetDeviceCount(int* n) { *n = 1; return 0; }
int hipGetDevice(int* n) { *n = 0; return 0; }
int hipDeviceGetAttribute(int* v, int a, int d) { *v = 256; return 0; }
int hipGetSymbolAddress(void** p, const void* s) { static char b[64]; *p = b; return 0; }
int hipGetLastError() { int e = last; last = 0; return e; }
const char* hipGetErrorString(int e) { return e ? "stub: out of memory" : "ok"; }
int hipStreamCreateWithFlags(void** s, unsigned f) { *s = &nfn; return 0; }
int hipEventCreate(void** e) { *e = &nfn; return 0; }
int hipEventElapsedTime(float* t, void* a, void* b) { *t = 1.f; return 0; }
int hipStreamEndCapture(void* s, void** g) { *g = &nfn; return 0; }
int hipGraphInstantiate(void** e, void* g, void* a, void* b, size_t n) { *e = &nfn; return 0; }
int hipFuncSetAttribute(const void* f, int a, int v) {  /* calls that change what another set */
  ++stub_attrs;
  for (int i = 0; i < nfn; ++i) if (fn[i] == f) { if (val[i] != v) { val[i] = v; ++stub_attr_changes; } return 0; }
  fn[nfn] = f; val[nfn++] = v; return 0;
}
static void* bin;
void** __hipRegisterFatBinary(const void* d) { return &bin; }
OK(__hipRegisterFunction) OK(__hipRegisterVar) OK(__hipUnregisterFatBinary)
OK(__hipPushCallConfiguration) OK(__hipPopCallConfiguration) OK(hipLaunchKernel)
OK(hipEventDestroy) OK(hipEventRecord) OK(hipEventSynchronize) OK(hipGraphDestroy)
OK(hipGraphExecDestroy) OK(hipGraphLaunch) OK(hipMemcpy2DAsync) OK(hipMemcpyToSymbolAsync)
OK(hipStreamBeginCapture) OK(hipStreamDestroy) OK(hipStreamSynchronize)
"""

PRELUDE = f"""
import ctypes, importlib.util, os, sys
stub = ctypes.CDLL(os.environ["HIP_STUB"], mode=ctypes.RTLD_GLOBAL)
spec = importlib.util.spec_from_file_location(
    "_lib", {os.path.join(ROOT, "diffeqflux.jl_amd", "diffeqflux_hip", "_lib.py")!r})
_lib = importlib.util.module_from_spec(spec)
spec.loader.exec_module(_lib)
lib = _lib.load()
def counter(name):
    return ctypes.c_long.in_dll(stub, name)
def create(widths, batch, precision="fp32", input_map=0):
    acts = ["tanh"] * (len(widths) - 2) + ["identity"]
    d = _lib.make_desc(widths, acts, input_map, precision, batch)
    h = ctypes.c_void_p()
    return lib.node_create(ctypes.byref(d), ctypes.byref(h)), h
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    d = tmp_path_factory.mktemp("hip_stub")
    src, so = d / "stub.c", d / "libamdhip64.so.7"
    src.write_text(STUB)
    subprocess.run(["gcc", "-w", "-shared", "-fPIC", "-o", str(so), "-Wl,-soname,libamdhip64.so.7",
                    str(src)], check=True)

    def go(body):
        env = dict(os.environ, HIP_STUB=str(so), LD_LIBRARY_PATH=str(d))
        r = subprocess.run([sys.executable, "-c", PRELUDE + body], env=env, capture_output=True,
                           text=True, timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr
        return r.stdout
    return go


@pytest.mark.parametrize("widths,batch,precision", [([2, 50, 2], 1, "fp32"),
                                                    ([16, 200, 200, 16], 40, "bf16x3")])
def test_create_without_memory_for_the_fused_steps(run, widths, batch, precision):
    """Any one allocation of node_create fails.  The weight copies of the fused
    steps (two per layer) are not needed: the handle is made without them.
    Every other failure is the error it was, and nothing leaks."""
    out = run(f"""
rc, h = create({widths}, {batch}, {precision!r})
n = counter("stub_mallocs").value
assert rc == 0 and n > 0
lib.node_destroy(h)
assert counter("stub_live").value == 0
made = 0
for k in range(n):
    counter("stub_mallocs").value, counter("stub_fail_at").value = 0, k
    rc, h = create({widths}, {batch}, {precision!r})
    assert rc in (0, -2) and (rc == 0) == bool(h.value)
    made += rc == 0
    if rc == 0:
        assert lib.node_destroy(h) == 0
    assert counter("stub_live").value == 0
print("made", made)
""")
    assert out.split()[-1] == str(2 * (len(widths) - 1))


def test_lds_limits_do_not_depend_on_the_handle(run):
    """The dynamic-LDS limit of a kernel is the process's, not a launch's: handles
    of other sizes, driven by other threads, set the same one."""
    out = run("""
import numpy as np
o = _lib.SolveOpts()
o.t0, o.t1, o.abstol, o.reltol, o.adaptive, o.maxiters = 0.0, 1.0, 1e-6, 1e-6, 1, 4
keep = []
for kind in ("fwd", "ragged"):
    for hidden in (50, 20, 33):
        rc, h = create([2, hidden, 2], 3)
        assert rc == 0
        p = np.zeros(5 * hidden + 2, np.float32)
        assert lib.node_set_params(h, p.ctypes.data, p.size) == 0
        u = np.zeros((3, 2), np.float32)
        if kind == "fwd":  # (the step counter never moves here)
            st = _lib.Stats()
            assert lib.node_forward(h, ctypes.byref(o), u.ctypes.data, None, 0, None, 0,
                                    ctypes.byref(st)) == -3
        else:
            t1, off, ts = np.ones(3), np.arange(4), np.ones(3)
            res = [np.zeros(s, d) for s, d in (((3, 2), np.float32), (3, np.int32), ((3, 4), np.int32))]
            rs = _lib.RaggedStats()
            rc = lib.node_ragged_forward(h, ctypes.byref(o), 3, t1.ctypes.data, u.ctypes.data,
                                         off.ctypes.data, ts.ctypes.data, *[x.ctypes.data for x in res],
                                         ctypes.byref(rs))
            print(kind, rc, lib.node_last_error(h))
print("sets", counter("stub_attrs").value, "changes", counter("stub_attr_changes").value)
""")
    print(out)
    words = out.split()
    assert int(words[words.index("sets") + 1]) > 0
    assert words[-1] == "0"
