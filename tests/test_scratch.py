"""The handle's scratch against a scripted allocator, on the CPU: handle.cpp
built with stubs for the HIP calls it makes.  A request that can do without
memory must leave the stream's buffer alone when it is refused, must not ask
for the refused size at every call, and must never take another stream's
buffer."""
import ctypes
import os
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(REPO, "teco-ops_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

STUB = r"""
#include "common.h"
#include <cstdlib>
#include <set>
static size_t limit;            // bytes that may be allocated in all
static size_t held;
static int mallocs, frees, captured;
static std::set<void *> live;
static size_t size_of(void *p) { return static_cast<size_t *>(p)[0]; }
extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
    ++mallocs;
    if (held + n > limit) return hipErrorOutOfMemory;
    *p = std::malloc(sizeof(size_t));
    static_cast<size_t *>(*p)[0] = n;
    held += n;
    live.insert(*p);
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    ++frees;
    if (!live.erase(p)) return hipErrorInvalidValue;
    held -= size_of(p);  // (the address stays taken, so that no later buffer has it)
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s) {
    *s = captured ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
void t_limit(size_t n) { limit = n; }
void t_capture(int on) { captured = on; }
int t_mallocs() { return mallocs; }
int t_frees() { return frees; }
size_t t_held() { return held; }
int t_live(void *p) { return live.count(p); }
void *t_need(tecoopsHandle_t h, size_t n) {
    void *p = nullptr;
    return tecoops::handle_scratch(h, n, &p) == TECOOPS_STATUS_SUCCESS ? p : nullptr;
}
void *t_try(tecoopsHandle_t h, size_t n) { return tecoops::handle_scratch_if_any(h, n); }
int t_retry() { return static_cast<int>(kScratchRetry); }
}
"""


@pytest.fixture(scope="module")
def stubbed(tmp_path_factory):
    d = tmp_path_factory.mktemp("scratch")
    src, out = d / "stub.cpp", d / "libscratch.so"
    src.write_text(STUB)
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1",
                    "-I", os.path.join(REPO, "include"), "-I", CSRC, "-I", os.path.join(ROCM, "include"),
                    os.path.join(CSRC, "handle.cpp"), str(src), "-o", str(out)], check=True)
    lib = ctypes.CDLL(str(out))
    lib.t_held.restype = ctypes.c_size_t
    for f in (lib.t_need, lib.t_try):
        f.restype, f.argtypes = ctypes.c_void_p, [ctypes.c_void_p, ctypes.c_size_t]
    lib.t_limit.argtypes = [ctypes.c_size_t]
    lib.t_live.argtypes = [ctypes.c_void_p]
    lib.tecoopsSetStream.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    lib.tecoopsDestroy.argtypes = [ctypes.c_void_p]
    return lib


@pytest.fixture
def handle(stubbed):
    h = ctypes.c_void_p()
    assert stubbed.tecoopsCreate(ctypes.byref(h)) == 0
    stubbed.t_limit(1 << 40)
    stubbed.t_capture(0)
    yield h
    stubbed.tecoopsDestroy(h)
    assert stubbed.t_held() == 0


def test_refused_request_keeps_the_buffer(stubbed, handle):
    decode = stubbed.t_need(handle, 1000)
    stubbed.t_limit(5000)  # the rest of the memory is taken
    frees = stubbed.t_frees()
    assert stubbed.t_try(handle, 100000) is None
    assert stubbed.t_live(decode) and stubbed.t_frees() == frees
    mallocs = stubbed.t_mallocs()
    assert stubbed.t_need(handle, 1000) == decode and stubbed.t_mallocs() == mallocs


def test_refused_size_is_not_tried_at_every_call(stubbed, handle):
    stubbed.t_limit(5000)
    n0 = stubbed.t_mallocs()
    for _ in range(stubbed.t_retry() // 2):
        assert stubbed.t_try(handle, 100000) is None
        assert stubbed.t_try(handle, 200000) is None
    assert stubbed.t_mallocs() - n0 <= 2
    # a smaller size is asked for at once, and memory that came back is found
    assert stubbed.t_try(handle, 4000) is not None
    stubbed.t_limit(1 << 40)
    got = None
    for _ in range(stubbed.t_retry() + 1):
        got = got or stubbed.t_try(handle, 100000)
    assert got is not None


def test_granted_request_replaces_the_buffer(stubbed, handle):
    decode = stubbed.t_need(handle, 1000)
    big = stubbed.t_try(handle, 100000)
    assert big is not None and not stubbed.t_live(decode)
    assert stubbed.t_need(handle, 1000) == big and stubbed.t_try(handle, 99999) == big


def test_optional_request_takes_nothing_over(stubbed, handle):
    first = []
    for s in range(1, 9):
        stubbed.tecoopsSetStream(handle, s)
        first.append(stubbed.t_need(handle, 1000))
    stubbed.tecoopsSetStream(handle, 99)
    assert stubbed.t_try(handle, 500) is None
    assert all(stubbed.t_live(p) for p in first)
    assert stubbed.t_need(handle, 1000) is not None  # an op that needs it takes one over
    assert not stubbed.t_live(first[0]) and all(stubbed.t_live(p) for p in first[1:])


def test_nothing_under_capture(stubbed, handle):
    stubbed.t_need(handle, 1000)
    stubbed.t_capture(1)
    assert stubbed.t_try(handle, 500) is None and stubbed.t_need(handle, 500) is None
