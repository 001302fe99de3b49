"""The copies between the caller's arrays and the device, no GPU: hostcopy.hip
compiled for the host against a stand-in for the HIP calls it makes, whose
copies run only when something waits for them, and fail where told to."""
import ctypes
import mmap
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
INC = "/opt/rocm/include"

HARNESS = r"""
#include <cstring>
#include <map>
#include <mutex>
#include <vector>
#include "SRC"

namespace {
struct Op { void* d; const void* s; size_t n; };
std::mutex mu;
std::vector<Op> q;           // the stream: what is enqueued, and how far it has run
size_t ran = 0;
std::map<hipEvent_t, size_t> at;
int calls[3], fail_at[3];    // copies, records, waits; the call from which they fail (0: none)
int kind;                    // of the caller's array, -1: not known to the runtime
bool fails(int k) { return ++calls[k] >= fail_at[k] && fail_at[k]; }
void run_to(size_t n) {
  for (; ran < n; ran++) std::memcpy(q[ran].d, q[ran].s, q[ran].n);
}
}  // namespace
extern "C" {
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  const std::lock_guard<std::mutex> l(mu);
  if (fails(0)) return hipErrorUnknown;
  q.push_back({d, s, n});
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  const std::lock_guard<std::mutex> l(mu);
  if (fails(1)) return hipErrorUnknown;
  at[e] = q.size();
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  const std::lock_guard<std::mutex> l(mu);
  if (fails(2)) return hipErrorUnknown;
  run_to(at[e]);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  const std::lock_guard<std::mutex> l(mu);
  run_to(q.size());
  return hipSuccess;
}
hipError_t hipMemcpyWithStream(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  const std::lock_guard<std::mutex> l(mu);
  if (fails(0)) return hipErrorUnknown;
  q.push_back({d, s, n});
  run_to(q.size());
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*) {
  std::memset(a, 0, sizeof(*a));
  if (kind < 0) return hipErrorInvalidValue;
  a->type = (hipMemoryType)kind;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = new char[n]; return hipSuccess; }
hipError_t hipHostFree(void* p) { delete[] (char*)p; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  static size_t k = 0;
  *e = (hipEvent_t)(++k);
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
}
namespace amps {
int hip_fail(hipError_t, const char*) { return AMPS_E_HIP; }
}
// the status; *pending: copies still to run when the call returned, *copies:
// the number made
extern "C" int copy_case(char* dst, const char* src, size_t n, int to_host, int slots, int memory, int fc, int fr,
                         int fw, size_t* pending, size_t* copies) {
  amps_ctx c;
  kind = memory;
  if (slots) host_copy_init(&c);
  q.clear(), at.clear(), ran = 0;
  std::memset(calls, 0, sizeof(calls));
  fail_at[0] = fc, fail_at[1] = fr, fail_at[2] = fw;
  const int r = to_host ? copy_to_host(&c, dst, src, n) : copy_to_device(&c, dst, src, n);
  *pending = q.size() - ran;
  *copies = q.size();
  hipStreamSynchronize(nullptr);
  host_copy_free(&c);
  return r;
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    if not (shutil.which("g++") and os.path.exists(os.path.join(INC, "hip", "hip_runtime.h"))):
        pytest.skip("needs g++ and the HIP headers")
    d = tmp_path_factory.mktemp("hostcopy")
    src = d / "harness.cpp"
    src.write_text(HARNESS.replace("SRC", os.path.join(ROOT, "amps_amd", "csrc", "hostcopy.hip")))
    so = d / "harness.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I", INC,
                    str(src), "-o", str(so)], check=True, capture_output=True, text=True)
    f = ctypes.CDLL(str(so)).copy_case
    f.argtypes = [ctypes.c_void_p, ctypes.c_char_p, ctypes.c_size_t] + [ctypes.c_int] * 6 + \
        [ctypes.POINTER(ctypes.c_size_t)] * 2

    def run(n, to_host, slots=1, fail=(0, 0, 0), memory=0, fresh=False):
        src = bytes(bytearray((i * 2654435761 >> 13) & 255 for i in range(4099))) * (n // 4099 + 1)
        dst = mmap.mmap(-1, n, flags=mmap.MAP_PRIVATE | mmap.MAP_ANONYMOUS)
        if not fresh:
            dst[:] = bytes(n)
        pending, copies = ctypes.c_size_t(), ctypes.c_size_t()
        at = (ctypes.c_char * n).from_buffer(dst)
        r = f(ctypes.addressof(at), src, n, to_host, slots, memory, *fail, ctypes.byref(pending), ctypes.byref(copies))
        return r, pending.value, copies.value, bytes(at) == src[:n]

    return run


@pytest.mark.parametrize("to_host", [0, 1])
@pytest.mark.parametrize("slots", [1, 0])
@pytest.mark.parametrize("n", [1, 4096, (1 << 20) - 1, 1 << 20, (4 << 20) - 1, 4 << 20, (16 << 20) - 1,
                               16 << 20, (16 << 20) + 4097, 45 << 20])
def test_copy_is_whole(lib, n, slots, to_host):
    """Both sides of the sizes from which the slots are used, ragged last chunks
    and more chunks than slots: every byte, and nothing left to run where the
    copy went through the slots or to the host."""
    r, pending, copies, same = lib(n, to_host, slots)
    assert r == 0 and same
    through = slots and n >= (4 << 20 if to_host else 16 << 20)
    assert copies > 1 if through else copies == 1
    assert pending == 0 or (not to_host and not through)


def test_pages_not_there_yet_take_the_slots_earlier(lib):
    """A fresh destination takes its page faults in the copy: from 1 MiB on by
    several threads."""
    for n, through in (((1 << 20) - 1, False), (1 << 20, True), (3 << 20, True)):
        r, pending, copies, same = lib(n, 1, fresh=True)
        assert r == 0 and same and pending == 0 and (copies > 1) == through


@pytest.mark.parametrize("to_host", [0, 1])
@pytest.mark.parametrize("memory,through", [(0, True), (-1, True), (1, False), (2, False), (3, False)])
def test_only_pageable_memory_takes_the_slots(lib, to_host, memory, through):
    """Arrays that the caller pinned (1), or that are device (2) or managed (3)
    memory, go in one copy; ordinary ones, by either way the runtime says so,
    through the slots."""
    r, _, copies, same = lib(45 << 20, to_host, memory=memory)
    assert r == 0 and same and (copies > 1) == through


@pytest.mark.parametrize("to_host", [0, 1])
@pytest.mark.parametrize("call", [0, 1, 2])
@pytest.mark.parametrize("when", [1, 4, 9])
def test_failed_copy_leaves_the_slots_idle(lib, to_host, call, when):
    """A copy, an event's record or its wait that fails is reported, and no
    copy that reads or writes the slots is still to run: the next call on the
    context uses them."""
    fail = [0, 0, 0]
    fail[call] = when
    r, pending, _, _ = lib(45 << 20, to_host, 1, tuple(fail))
    assert r != 0 and pending == 0
