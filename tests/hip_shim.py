"""A child process in which some HIP calls of the library go through functions of this file's
own: they count and log them, and can refuse a cooperative launch, report that a kernel gave
up a wait (its word on the host reads 1) or fail an allocation (the real hipMalloc is then
asked for more than any card has, so that HIP's last error is what a full card leaves).  The functions come before HIP's in the process's symbol order, because
they are loaded first and globally."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>

int coop_calls = 0, coop_refuse = 0;            /* refuse the next `coop_refuse` cooperative launches */
int gave_up = 0;                                /* the next `gave_up` abort words read 1 */
int flow_gave_up = 0, *flow_word = NULL;        /* the next `flow_gave_up` waits for an event set the sweeps' word */
int launches = 0;
int malloc_calls = 0, malloc_fail_at = -1, malloc_fail_n = 1; /* fail calls malloc_fail_at ... */
int attr_n = 0, attr_value[256];
const void* attr_func[256];

static void* real(const char* name) {
  void* h = dlopen("libamdhip64.so.7", RTLD_NOLOAD | RTLD_LAZY);
  return h ? dlsym(h, name) : NULL;
}
int hipMalloc(void** p, size_t n) {
  int (*f)(void**, size_t) = (int (*)(void**, size_t))real("hipMalloc");
  const int k = malloc_calls++;
  if (malloc_fail_at >= 0 && k >= malloc_fail_at && k < malloc_fail_at + malloc_fail_n) n = (size_t)1 << 50;
  return f(p, n);
}
int hipFuncSetAttribute(const void* func, int attr, int value) {
  int (*f)(const void*, int, int) = (int (*)(const void*, int, int))real("hipFuncSetAttribute");
  if (attr_n < 256) attr_func[attr_n] = func, attr_value[attr_n++] = value;
  return f(func, attr, value);
}
int hipMemcpyAsync(void* dst, const void* src, size_t n, int kind, void* s) {
  int (*f)(void*, const void*, size_t, int, void*) = (int (*)(void*, const void*, size_t, int, void*))real("hipMemcpyAsync");
  const int e = f(dst, src, n, kind, s);
  if (e == 0 && n == 4 && kind == 2 && gave_up > 0) {
    int (*sync)(void*) = (int (*)(void*))real("hipStreamSynchronize");
    gave_up--;
    sync(s);
    *(int*)dst = 1;
  }
  return e;
}
int hipHostMalloc(void** p, size_t n, unsigned flags) {
  int (*f)(void**, size_t, unsigned) = (int (*)(void**, size_t, unsigned))real("hipHostMalloc");
  const int e = f(p, n, flags);
  if (e == 0 && n == 4) flow_word = *p;
  return e;
}
int hipEventSynchronize(void* ev) {
  int (*f)(void*) = (int (*)(void*))real("hipEventSynchronize");
  const int e = f(ev);
  if (flow_gave_up > 0 && flow_word) {
    flow_gave_up--;
    *flow_word = 1;
  }
  return e;
}
typedef struct { unsigned x, y, z; } dim3_t;
int hipLaunchKernel(const void* func, dim3_t g, dim3_t b, void** args, size_t lds, void* s) {
  int (*f)(const void*, dim3_t, dim3_t, void**, size_t, void*) =
      (int (*)(const void*, dim3_t, dim3_t, void**, size_t, void*))real("hipLaunchKernel");
  launches++;
  return f(func, g, b, args, lds, s);
}
int hipLaunchCooperativeKernel(const void* func, dim3_t g, dim3_t b, void** args, unsigned lds, void* s) {
  int (*f)(const void*, dim3_t, dim3_t, void**, unsigned, void*) =
      (int (*)(const void*, dim3_t, dim3_t, void**, unsigned, void*))real("hipLaunchCooperativeKernel");
  coop_calls++;
  if (coop_refuse > 0) {
    coop_refuse--;
    return 720; /* hipErrorCooperativeLaunchTooLarge */
  }
  return f(func, g, b, args, lds, s);
}
"""

HEAD = """
import ctypes, sys
sys.path.insert(0, %r)
shim = ctypes.CDLL(%r, ctypes.RTLD_GLOBAL)
def val(name):
    return ctypes.c_int.in_dll(shim, name)
import numpy as np
import frontistr_amd as fa
from oracle import restate
"""


def run(tmp_path, script, timeout=100):
    """The printed lines of `script` in a child (its names: shim, val, np, fa, restate)."""
    src, lib, prog = (str(tmp_path / n) for n in ("shim.c", "shim.so", "prog.py"))
    with open(src, "w") as f:
        f.write(SOURCE)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-w", src, "-o", lib, "-ldl"], check=True)
    with open(prog, "w") as f:
        f.write(HEAD % (ROOT, lib) + script)
    p = subprocess.run([sys.executable, prog], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True,
                       timeout=timeout, cwd=ROOT)
    assert p.returncode == 0, p.stdout[-3000:]
    return p.stdout.splitlines()
