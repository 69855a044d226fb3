"""A hipMalloc that refuses chosen sizes, in front of the one libovl.so calls: for tests of what a call does without
room for a buffer.  Used in a process of its own: install() must run before the library is loaded."""
import ctypes as C
import os
import subprocess

SOURCE = r"""
#include <stddef.h>
typedef int (*fn)(void **, size_t);
static fn real;
static size_t refused[8];
static int refusals;
void shim_real(void *f) { real = (fn)f; }
void shim_refuse(int slot, size_t bytes) { refused[slot] = bytes; }
int shim_refusals(void) { return refusals; }
int hipMalloc(void **p, size_t n)
{
    for (int k = 0; k < 8; ++k)
        if (n && n == refused[k]) { ++refusals; return 2; } /* hipErrorOutOfMemory */
    return real(p, n);
}
"""


def install(folder):
    src, so = os.path.join(folder, "shim.c"), os.path.join(folder, "shim.so")
    with open(src, "w") as f:
        f.write(SOURCE)
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", src, "-o", so], check=True)
    hip = C.CDLL("libamdhip64.so.7")
    shim = C.CDLL(so, mode=C.RTLD_GLOBAL)
    shim.shim_real(C.cast(hip.hipMalloc, C.c_void_p))
    shim.shim_refuse.argtypes = [C.c_int, C.c_size_t]
    return shim
