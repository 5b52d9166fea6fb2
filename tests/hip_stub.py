"""Host code of libptv3_hip.so over a runtime that launches nothing.

Which calls the library makes, in which order, and what it does where one fails or where the part is another one, cannot be
seen on a GPU. Here a small library answers the HIP calls in its place: it keeps a record of them, lets a chosen one fail and
claims any number of CUs. Kernels are never run, so the addresses a test hands over need not be memory. Each test's code runs
in a process of its own, which loads the stand-in in front of the runtime."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

_STUB = r"""
#include <stddef.h>
#include <string.h>
typedef struct { unsigned x, y, z; } dim3;
typedef struct { char op[24]; void *a, *b; long failed; } call;
call hip_calls[65536];
int hip_n_calls, hip_cus = 256, hip_fail_nth;
char hip_fail_op[24];
static long events;
static int note(const char* op, void* a, void* b) {
    call* c = &hip_calls[hip_n_calls++ & 65535];
    strncpy(c->op, op, 23);
    c->a = a;
    c->b = b;
    return c->failed = !strcmp(op, hip_fail_op) && hip_fail_nth-- == 0;
}
int hipLaunchKernel(const void* f, dim3 g, dim3 b, void** args, size_t lds, void* stream) { return note("launch", stream, (void*)f); }
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, void* stream) { (void)g; (void)b; (void)lds; return hip_calls[65535].b = stream, 0; }
int __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, void** stream) {
    *g = *b = (dim3){1, 1, 1};
    *lds = 0;
    *stream = hip_calls[65535].b;
    return 0;
}
int hipGetLastError(void) { return 0; }
int hipPeekAtLastError(void) { return 0; }
int hipGetDevice(int* d) { *d = hip_cus / 8 % 64; return 0; }   /* one device a number of CUs: the library asks each once */
int hipDeviceGetAttribute(int* v, int attr, int d) { *v = hip_cus; return 0; }
int hipFuncSetAttribute(const void* f, int attr, int v) { return 0; }
int hipEventCreateWithFlags(void** e, unsigned flags) {
    void* made = (void*)(0x1000 + 16 * events++);
    const int failed = note("create", made, 0);
    if (!failed) *e = made;
    return failed;
}
int hipEventDestroy(void* e) { return note("destroy", e, 0); }
int hipEventRecord(void* e, void* stream) { return note("record", stream, e); }
int hipStreamWaitEvent(void* stream, void* e, unsigned flags) { return note("wait", stream, e); }
int hipStreamSynchronize(void* stream) { return note("synchronize", stream, 0); }
"""

_PRELUDE = r"""
import ctypes, sys
hip = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
class Call(ctypes.Structure):
    _fields_ = [("op", ctypes.c_char * 24), ("a", ctypes.c_void_p), ("b", ctypes.c_void_p), ("failed", ctypes.c_long)]
_calls = (Call * 65536).in_dll(hip, "hip_calls")
_n = ctypes.c_int.in_dll(hip, "hip_n_calls")
def calls():
    assert _n.value < 65535
    return [(c.op.decode(), c.a or 0, c.b or 0, bool(c.failed)) for c in _calls[:_n.value]]
def clear(fail=None, nth=0, cus=256):
    _n.value = 0
    ctypes.c_int.in_dll(hip, "hip_fail_nth").value = nth
    ctypes.c_int.in_dll(hip, "hip_cus").value = cus
    (ctypes.c_char * 24).in_dll(hip, "hip_fail_op").value = (fail or "").encode()
from pointtransformerv3_amd import _lib
lib = _lib.load()
"""


def run(code, tmp_path):
    """Runs `code` behind the prelude above; a failed assertion in it is the test's."""
    src, so = tmp_path / "hip_stub.c", tmp_path / "hip_stub.so"
    src.write_text(_STUB)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-w", "-o", str(so), str(src)], check=True)
    env = dict(os.environ, PYTHONPATH=os.pathsep.join([ROOT, os.path.join(ROOT, "tests")]))
    got = subprocess.run([sys.executable, "-c", _PRELUDE + code, str(so)], cwd=ROOT, env=env, capture_output=True, text=True, timeout=300)
    assert got.returncode == 0, got.stdout + got.stderr
    return got.stdout
