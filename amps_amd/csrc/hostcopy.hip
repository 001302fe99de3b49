// hostcopy.hip — large copies between the caller's (pageable) arrays and the device.
//
// A pageable hipMemcpy stages through the runtime's pinned buffers with one
// host thread, which on a fresh array also takes its page faults: 17 GB/s to
// the host (4 on a fresh array) and 26 to 35 from it, where the bus moves 57.  Here a
// few threads that live for the call copy between the array and a context's own
// pinned slots, two per thread, while the other slots are on the bus: 40 GB/s
// (12 on a fresh array), less some 130 us to start and join them.
#include <hip/hip_runtime.h>
#include <sys/mman.h>
#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <functional>
#include <mutex>
#include <thread>

#include "amps_common.h"

using namespace amps;

namespace {
constexpr int THREADS = 4, SLOTS = 2 * THREADS;
constexpr size_t SLOT_BYTES = PIN_BYTES / SLOTS;
// Sizes from which the slots are ahead (us, a plain copy and the slots): to the
// host, 2 MiB 125 and 183, 4 MiB 248 and 237, 16 MiB 926 and 527, but where
// the pages are not there yet 512 KiB 95 and 165, 1 MiB 259 and 200, 4 MiB 1,063 and
// 487; to the device, of an array that the caches hold 16 MiB 458 and 483, 32 MiB
// 904 and 900, of one that they don't 8 MiB 323 and 343, 16 MiB 630 and 532.
constexpr size_t MIN_TO_HOST = (size_t)4 << 20, MIN_TO_FRESH = (size_t)1 << 20, MIN_TO_DEVICE = (size_t)16 << 20;

struct Job {
  amps_ctx* c;
  char* dst;
  const char* src;
  size_t bytes, chunk;
  bool to_host;
  std::atomic<size_t> next{0};
  std::atomic<int> err{0};
};

// one thread's share: chunks taken in turn until none is left.  A slot is
// used again only after its event, and every event is waited for before the
// return, so the slots are idle between calls.
void work(Job& j, int t) {
  amps_ctx* c = j.c;
  hipError_t e = hipSetDevice(c->device);
  const size_t n = (j.bytes + j.chunk - 1) / j.chunk;
  size_t at[2] = {n, n};  // the chunk in each of the two slots, n: none
  auto size = [&](size_t i) { return std::min(j.chunk, j.bytes - i * j.chunk); };
  auto slot = [&](int s) { return c->h_pin + (size_t)(2 * t + s) * SLOT_BYTES; };
  auto retire = [&](int s) {
    if (at[s] == n) return;
    const hipError_t q = hipEventSynchronize(c->pin_ev[2 * t + s]);
    if (q == hipSuccess && j.to_host) std::memcpy(j.dst + at[s] * j.chunk, slot(s), size(at[s]));
    if (e == hipSuccess) e = q;
    at[s] = n;
  };
  int s = 0;
  while (e == hipSuccess && !j.err.load()) {
    const size_t i = j.next.fetch_add(1);
    if (i >= n) break;
    retire(s);
    if (e != hipSuccess) break;
    if (j.to_host) {
      e = hipMemcpyAsync(slot(s), j.src + i * j.chunk, size(i), hipMemcpyDeviceToHost, c->stream);
    } else {
      std::memcpy(slot(s), j.src + i * j.chunk, size(i));
      e = hipMemcpyAsync(j.dst + i * j.chunk, slot(s), size(i), hipMemcpyHostToDevice, c->stream);
    }
    if (e == hipSuccess) e = hipEventRecord(c->pin_ev[2 * t + s], c->stream);
    if (e == hipSuccess) at[s] = i;
    s ^= 1;
    if (e == hipSuccess && j.to_host) retire(s);  // the earlier chunk, while this one is on the bus
  }
  retire(s);
  retire(s ^ 1);
  if (e != hipSuccess) j.err.store((int)e);
}

// the array's first, middle and last page are in memory
bool resident(const void* p, size_t bytes) {
  const uintptr_t page = (uintptr_t)sysconf(_SC_PAGESIZE), a = (uintptr_t)p;
  for (const uintptr_t q : {a, a + bytes / 2, a + bytes - 1}) {
    unsigned char in = 0;
    if (mincore((void*)(q / page * page), 1, &in) != 0 || !(in & 1)) return false;
  }
  return true;
}

bool through_slots(const amps_ctx* c, const void* host, size_t bytes, bool to_host) {
  if (!c->h_pin || bytes < (to_host ? MIN_TO_FRESH : MIN_TO_DEVICE)) return false;
  // pinned memory takes the bus's rate by itself (32 MiB 597 us, through the
  // slots 915); what is no host memory at all is the runtime's to resolve
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, host) != hipSuccess)
    (void)hipGetLastError();  // a pointer that the runtime does not know
  else if (a.type != hipMemoryTypeUnregistered)
    return false;
  return !to_host || bytes >= MIN_TO_HOST || !resident(host, bytes);
}

int copy(amps_ctx* c, void* dst, const void* src, size_t bytes, bool to_host) {
  if (!through_slots(c, to_host ? dst : src, bytes, to_host)) {
    // complete on return (12 us for a few bytes, an asynchronous copy and a wait 20)
    if (to_host) HIP_TRY(hipMemcpyWithStream(dst, src, bytes, hipMemcpyDeviceToHost, c->stream));
    // a pageable source is read before the return
    else HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, c->stream));
    return 0;
  }
  const std::lock_guard<std::mutex> lock(c->pin_mutex);  // one call at a time on the slots
  Job j{c, (char*)dst, (const char*)src, bytes, 0, to_host};
  // at least two chunks a thread, whole pages
  j.chunk = std::min(SLOT_BYTES, ((bytes + SLOTS - 1) / SLOTS + 4095) / 4096 * 4096);
  std::thread th[THREADS - 1];
  for (int t = 1; t < THREADS; t++) {
    try {
      th[t - 1] = std::thread(work, std::ref(j), t);
    } catch (const std::exception&) {
      break;  // no more threads: the ones there are take all chunks
    }
  }
  work(j, 0);
  for (auto& t : th)
    if (t.joinable()) t.join();
  const hipError_t e = (hipError_t)j.err.load();
  // a copy whose event could not be recorded or waited for may still run
  if (e != hipSuccess) (void)hipStreamSynchronize(c->stream);
  HIP_TRY(e);
  return 0;
}
}  // namespace

namespace amps {
// pinned slots and their events; without them the copies are plain ones
void host_copy_init(amps_ctx* c) {
  void* p = nullptr;
  if (hipHostMalloc(&p, PIN_BYTES, hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();
    return;
  }
  for (int i = 0; i < SLOTS; i++)
    if (hipEventCreateWithFlags(&c->pin_ev[i], hipEventDisableTiming) != hipSuccess) {
      (void)hipGetLastError();
      c->pin_ev[i] = nullptr;
      c->h_pin = (char*)p;
      host_copy_free(c);
      return;
    }
  c->h_pin = (char*)p;
}
void host_copy_free(amps_ctx* c) {
  for (hipEvent_t& e : c->pin_ev) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
  if (c->h_pin) (void)hipHostFree(c->h_pin);
  c->h_pin = nullptr;
}
// after the stream's work, complete on return
int copy_to_host(amps_ctx* c, void* dst, const void* src, size_t bytes) { return copy(c, dst, src, bytes, true); }
int copy_to_device(amps_ctx* c, void* dst, const void* src, size_t bytes) { return copy(c, dst, src, bytes, false); }
}  // namespace amps
