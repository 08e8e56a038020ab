"""The copies of large states to the host (hostcopy.cpp) without a GPU: compiled here with the
host compiler against a stand-in for the few runtime calls it makes, whose events complete after a
set time."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "magudi_amd", "csrc")

RUNTIME = r"""
#pragma once
#include <atomic>
#include <chrono>
#include <cstdlib>
#include <cstring>
#include <thread>
enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorInvalidResource = 400 };
enum { hipMemcpyDeviceToHost = 2, hipEventDisableTiming = 2, hipHostMallocDefault = 0 };
struct Stream { int device; };
struct Event { int device; int waits_ms; };
typedef Stream* hipStream_t;
typedef Event* hipEvent_t;
inline volatile int g_wait_ms = 0;      // of the next event; below 0: until g_release
inline volatile bool g_release = false;
inline std::atomic<int> g_copies{0};
inline int g_fail_copy = -1, g_events = 0, g_pinned = 0;
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1 };
struct hipPointerAttribute_t { hipMemoryType type; };
inline const void* g_registered = nullptr;
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  a->type = p == g_registered ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
  return p == g_registered ? hipSuccess : hipErrorInvalidValue;
}
typedef int hipDevice_t;
inline int g_device = 0;
inline hipError_t hipGetDevice(int* d) { *d = g_device; return hipSuccess; }
inline hipError_t hipSetDevice(int d) { g_device = d; return hipSuccess; }
inline hipError_t hipStreamGetDevice(hipStream_t st, hipDevice_t* d) { *d = st->device; return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned = 0) { *p = std::malloc(n); ++g_pinned; return hipSuccess; }
inline hipError_t hipHostFree(void* p) { std::free(p); --g_pinned; return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = static_cast<Event*>(std::malloc(sizeof(Event)));
  **e = {g_device, 0};
  ++g_events;
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) { std::free(e); --g_events; return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, hipStream_t) {
  if (g_copies++ == g_fail_copy) return hipErrorInvalidValue;
  std::memcpy(d, s, n);
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t st) {
  if (e->device != st->device) return hipErrorInvalidResource;
  e->waits_ms = g_wait_ms;     // the first event after other work on the stream
  g_wait_ms = 0;
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
  while (e->waits_ms < 0 && !g_release) std::this_thread::sleep_for(std::chrono::milliseconds(1));
  if (e->waits_ms > 0) std::this_thread::sleep_for(std::chrono::milliseconds(e->waits_ms));
  e->waits_ms = 0;
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
"""

MAIN = r"""
#include <algorithm>
#include <cstdio>
#include <ctime>
#include <new>
#include <vector>
#include "hostcopy.h"
static double cpu() {
  timespec t;
  clock_gettime(CLOCK_PROCESS_CPUTIME_ID, &t);
  return t.tv_sec + 1e-9 * t.tv_nsec;
}
// this thread's allocations fail from the g_left-th on (a thread start makes one)
static std::atomic<long> g_left{-1};
static thread_local bool g_watched = false;
void* operator new(std::size_t n) {
  if (g_watched && g_left >= 0 && g_left-- <= 0) throw std::bad_alloc();
  if (void* p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }
int main(int argc, char** argv) {
  const size_t n = (size_t)atol(argv[2]), off = (size_t)atol(argv[3]);
  std::vector<unsigned char> src(std::max(n, size_t(40) << 20)), room(n + off + 64, 0xcc);
  for (size_t i = 0; i < src.size(); ++i) src[i] = (unsigned char)(i * 2654435761u >> 13);
  Stream st{0};
  mgd::HostCopy hc;
  const auto good = [&] {
    for (size_t i = 0; i < off; ++i) if (room[i] != 0xcc) return 0;
    for (size_t i = 0; i < 64; ++i) if (room[off + n + i] != 0xcc) return 0;
    return std::memcmp(room.data() + off, src.data(), n) == 0 ? 1 : 0;
  };
  if (!std::strcmp(argv[1], "copy")) {
    g_fail_copy = atoi(argv[4]);
    const int rc = hc.to_host(room.data() + off, src.data(), n, &st);
    std::printf("%d %d %d\n", rc, rc == 0 ? good() : 0, g_copies.load());
    g_fail_copy = -1;
    const int rc2 = hc.to_host(room.data() + off, src.data(), n, &st);
    std::printf("%d %d\n", rc2, good());
  } else if (!std::strcmp(argv[1], "wait")) {
    (void)hc.to_host(room.data() + off, src.data(), n, &st);
    g_wait_ms = 400;
    const double t0 = cpu();
    const int rc = hc.to_host(room.data() + off, src.data(), n, &st);
    std::printf("%d %d %.6f\n", rc, good(), cpu() - t0);
  } else if (!std::strcmp(argv[1], "memory")) {
    g_watched = true;
    g_left = atoi(argv[4]);
    int rc = -1;
    try {
      rc = hc.to_host(room.data() + off, src.data(), n, &st);
    } catch (...) {                        // nothing may pass the C entry points
    }
    g_left = -1;
    std::printf("%d %d\n", rc, good());
  } else if (!std::strcmp(argv[1], "device")) {
    g_device = 1;
    const int rc = hc.to_host(room.data() + off, src.data(), n, &st);
    std::printf("%d %d %d\n", rc, good(), g_device);
  } else if (!std::strcmp(argv[1], "registered")) {
    g_registered = room.data() + off;
    const int rc = hc.to_host(room.data() + off, src.data(), n, &st);
    std::printf("%d %d %d\n", rc, good(), g_copies.load());
  } else if (!std::strcmp(argv[1], "beside")) {
    // `others` copies that wait for their streams, then one more: the runtime copies it makes
    const int others = atoi(argv[4]);
    const size_t no = (size_t)atol(argv[5]);
    std::vector<std::thread> busy;
    for (int k = 0; k < others; ++k) {
      g_wait_ms = -1;
      busy.emplace_back([&] {
        std::vector<unsigned char> room2(no);
        mgd::HostCopy hc2;
        Stream st2{0};
        (void)hc2.to_host(room2.data(), src.data(), no, &st2);   // 33 MiB: 16 slots and more
      });
      while (g_copies < 16 * (k + 1)) std::this_thread::yield();   // it has filled its ring
    }
    std::this_thread::sleep_for(std::chrono::milliseconds(20));
    const int before = g_copies;
    const int rc = hc.to_host(room.data() + off, src.data(), n, &st);
    const int made = g_copies - before;
    g_release = true;
    for (std::thread& t : busy) t.join();
    std::printf("%d %d %d\n", rc, good(), made);
  }
  return 0;
}
"""


@pytest.fixture(scope="module")
def tool(tmp_path_factory):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("no host compiler")
    if len(os.sched_getaffinity(0)) < 4:
        pytest.skip("copies take several threads on 4 CPUs or more")
    d = tmp_path_factory.mktemp("hostcopy")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(RUNTIME)
    (d / "main.cpp").write_text(MAIN)
    exe = str(d / "t")
    subprocess.check_call([cxx, "-std=c++17", "-O1", "-Wall", "-I", str(d), "-I", CSRC, "-o", exe,
                           str(d / "main.cpp"), os.path.join(CSRC, "hostcopy.cpp"), "-pthread"])

    def run(*args):
        out = subprocess.run([exe, *map(str, args)], capture_output=True, text=True, timeout=60)
        assert out.returncode == 0, (args, out.returncode, out.stderr)
        return [line.split() for line in out.stdout.splitlines()]
    return run


MIB = 1 << 20


@pytest.mark.parametrize("n,off", [(4 * MIB - 1, 0), (4 * MIB, 8), (5 * MIB + 13, 4096), (33 * MIB, 24),
                                   (71 * MIB + 5, 3)])
def test_copies(tool, n, off):
    for fail in (-1, 0, 1, 2):
        first, second = tool("copy", n, off, fail)
        failed = 0 <= fail < int(first[2])
        assert (int(first[0]) != 0) == failed and int(first[1]) == (0 if failed else 1), fail
        assert second == ["0", "1"], fail


def test_threads_sleep_while_the_stream_is_busy(tool):
    """A copy behind 0.4 s of other work on its stream: the process spends next to no CPU time."""
    (rc, good, cpu), = tool("wait", 12 * MIB, 0)
    assert rc == "0" and good == "1"
    assert float(cpu) < 0.1, cpu


@pytest.mark.parametrize("n,others,threads", [(5 * MIB, 0, True), (5 * MIB, 1, False), (40 * MIB, 1, True),
                                              (40 * MIB, 4, True)])
def test_copies_beside_others(tool, n, others, threads):
    """A small copy beside another one is one plain copy, a large one is not."""
    (rc, good, made), = tool("beside", n, 0, others, 33 * MIB)
    assert rc == "0" and good == "1"
    assert (int(made) > 1) == threads


@pytest.mark.parametrize("n", [5 * MIB, 40 * MIB])
def test_registered_memory_is_copied_to_directly(tool, n):
    assert tool("registered", n, 8) == [["0", "1", "1"]]


@pytest.mark.parametrize("left", range(9))
def test_without_memory_for_threads(tool, left):
    """Memory runs out at the first, second, .. allocation of a copy: fewer threads or a plain copy,
    the same bytes, no exception."""
    assert tool("memory", 20 * MIB, 16, left) == [["0", "1"]]


def test_another_current_device(tool):
    """The region is on device 0, the caller's current device is 1, and stays so."""
    assert tool("device", 12 * MIB, 0) == [["0", "1", "1"]]
