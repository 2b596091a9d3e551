"""aih_init when device memory runs out, without a device: the HIP calls it makes
are answered by a small library loaded ahead of the HIP runtime."""
import os
import subprocess
import sys

import pytest

from aihost_amd import _native as nat
from aihost_amd import build

STUB = r"""
#include <hip/hip_runtime_api.h>
#include <cstdlib>
#include <cstring>
#include <cstdint>
// objects handed out and not given back; allocations of device memory; the
// number of them that succeed
extern "C" {
int live = 0, mallocs = 0, allowed = 0;
size_t asked = 0;
static hipError_t give(void **p) { *p = malloc(1); ++live; return hipSuccess; }
static hipError_t take(void *p) { free(p); --live; return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int)   // a macro: the versioned name
{
    memset(p, 0, sizeof *p);
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) { static char at[256]; *p = at; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return give((void **)s); }
hipError_t hipStreamDestroy(hipStream_t s) { return take(s); }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *c) { *c = hipStreamCaptureStatusNone; return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t, unsigned) { return give(p); }
hipError_t hipHostFree(void *p) { return take(p); }
hipError_t hipEventCreate(hipEvent_t *e) { return give((void **)e); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return give((void **)e); }
hipError_t hipEventDestroy(hipEvent_t e) { return take(e); }
hipError_t hipMalloc(void **p, size_t bytes)
{
    asked = bytes;
    return mallocs++ < allowed ? give(p) : hipErrorOutOfMemory;
}
hipError_t hipFree(void *p) { return take(p); }
hipError_t hipGetLastError(void) { return hipSuccess; }
}
"""

RUN = r"""
import ctypes, sys
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL(sys.argv[2])
n = lambda name: ctypes.c_int.in_dll(stub, name)
ctx = ctypes.c_void_p(1)
n("allowed").value = int(sys.argv[3])
rc = lib.aih_init(0, ctypes.byref(ctx))
held, asked = n("live").value, ctypes.c_size_t.in_dll(stub, "asked").value
if ctx.value:
    assert lib.aih_destroy(ctx) == 0
print(rc, ctx.value is not None, held, n("live").value, n("mallocs").value, asked)
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    d = tmp_path_factory.mktemp("stub")
    src, so = d / "stub.cpp", d / "libstub.so"
    src.write_text(STUB)
    subprocess.run(["g++", "-shared", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(build.ROCM, "include"),
                    str(src), "-o", str(so)], check=True)
    return str(so)


def _init(stub, allowed):
    out = subprocess.run([sys.executable, "-c", RUN, stub, nat.LIB_PATH, str(allowed)], check=True, capture_output=True,
                         text=True, timeout=120).stdout.split()
    return int(out[0]), out[1] == "True", *map(int, out[2:])


def test_init_sets_the_partial_sums_aside(stub):
    rc, made, held, left, mallocs, asked = _init(stub, 1)
    assert (rc, made, mallocs) == (nat.AIH_OK, True, 1)
    assert held > 0 and left == 0 and asked >= nat.NOALLOC_SCRATCH_BYTES


def test_init_without_room_for_the_partial_sums_fails(stub):
    # a context without them would sum the splits of a product in another
    # order than the allocation-free entry point, or not split it
    rc, made, held, left, mallocs, _ = _init(stub, 0)
    assert (rc, made, mallocs) == (nat.HIP_ERROR_OUT_OF_MEMORY, False, 1)
    assert held == 0 and left == 0
