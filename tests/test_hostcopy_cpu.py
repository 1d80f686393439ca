"""The copy of device results to pageable memory (splat.js_amd/csrc/
gs_hostcopy.h) on the CPU, over stand-ins for the HIP calls (tests/host/
hip_stub.h): every block arrives, with worker threads and where none can be
started; a fill that fails ends the call with its
error, after which the ring works again; so does pinned memory that cannot be
had."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROBE = r"""
#include <stdio.h>
#include <sys/resource.h>
#include <unistd.h>
#include <atomic>
#include <set>
#include "gs_hostcopy.h"
using namespace gs;

static std::mutex gm;
static std::set<std::thread::id> takers;
static hipError_t plain = hipSuccess;   // why the call was the caller's own

// `count` blocks of `bytes`: block k holds bytes (k + i) & 0xff; failAt: that fill fails
static int copy(HostRing& ring, int count, size_t bytes, int failAt, hipError_t* err) {
  std::vector<unsigned char> out((size_t)(count > 0 ? count : 0) * bytes, 0xee);
  Stream st;
  std::atomic<int> taken{0};
  takers.clear();
  plain = hipSuccess;
  *err = ring_copy(
      ring, &st, count, bytes,
      [&](int k, char* slot) {
        if (k == failAt) return hipErrorUnknown;
        for (size_t i = 0; i < bytes; i++) slot[i] = (char)((size_t)k + i);
        return hipSuccess;
      },
      [&](int k, const char* slot) {
        { std::lock_guard<std::mutex> l(gm); takers.insert(std::this_thread::get_id()); }
        taken++;
        memcpy(out.data() + (size_t)k * bytes, slot, bytes);
      },
      [&](hipError_t why) {   // the caller's own copy
        plain = why;
        return hipSuccess;
      });
  if (plain != hipSuccess) return 0;
  if (*err != hipSuccess) return st.syncs == 1 && taken <= failAt ? 0 : 1;
  for (int k = 0; k < count; k++)
    for (size_t i = 0; i < bytes; i++)
      if (out[(size_t)k * bytes + i] != (unsigned char)((size_t)k + i)) return 1;
  return taken == (count > 0 ? count : 0) ? 0 : 1;
}

int main(int argc, char** argv) {
  const std::string mode = argv[1];
  if (mode == "nomem") {   // pinned memory or an event that cannot be had: the caller's copy, no error left behind
    HostRing r;
    hipError_t e;
    int bad = 0;
    mallocsLeft = 0;
    copy(r, 4, 1000, 0, &e);
    bad |= e != hipSuccess || plain != hipErrorOutOfMemory || lastErrors != 1 || r.have != 0 || r.buf != nullptr;
    mallocsLeft = 1 << 30;
    eventsLeft = 2;
    copy(r, 4, 1000, 0, &e);
    bad |= e != hipSuccess || plain != hipErrorUnknown || lastErrors != 2;
    eventsLeft = 1 << 30;
    bad |= copy(r, 4, 1000, -1, &e) || e != hipSuccess || plain != hipSuccess;
    r.release();
    printf("%d %d\n", bad, pinned);
    return 0;
  }
  HostRing ring;
  hipError_t e;
  int bad = 0;
  size_t most = 0;
  if (mode == "nothreads") {   // no room for a thread's stack
    if (ring.ensure(HostRing::kSlots, 1 << 17) != hipSuccess) return 2;
    void* room = malloc(20 << 20);   // for the copies below
    memset(room, 1, 20 << 20);
    free(room);
    long pages = 0;
    FILE* f = fopen("/proc/self/statm", "r");
    if (!f || fscanf(f, "%ld", &pages) != 1) return 2;
    fclose(f);
    rlimit lim;
    getrlimit(RLIMIT_AS, &lim);
    lim.rlim_cur = (rlim_t)pages * sysconf(_SC_PAGESIZE) + (rlim_t(6) << 20);
    if (setrlimit(RLIMIT_AS, &lim)) return 2;
  }
  const int counts[] = {0, 1, 2, 3, 5, 8, 9, 17, 40, 100};
  const size_t sizes[] = {1, 4095, 4096, 4097, 100000};
  for (int rep = 0; rep < (mode == "nothreads" ? 1 : 5); rep++)
    for (int c : counts)
      for (size_t b : sizes) {
        if (mode == "nothreads" && (size_t)c * b > 2000000) continue;
        bad |= copy(ring, c, b, -1, &e) || e != hipSuccess;
        most = std::max(most, takers.size());
        for (int at : {0, 1, c / 2, c - 1}) {
          if (at < 0 || at >= c || rep) continue;
          bad |= copy(ring, c, b, at, &e) || e != hipErrorUnknown;
        }
      }
  ring.release();
  printf("%d %zu %d %d\n", bad, most, pinnedMost <= (int)(HostRing::kSlots * HostRing::kSlotBytes), pinned);
  return 0;
}
"""


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    d = tmp_path_factory.mktemp("hostcopy")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text('#include "hip_stub.h"\n')
    (d / "probe.cpp").write_text("#include <string>\n" + PROBE)
    exe = d / "probe"
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-pthread", "-I", str(d), "-I", os.path.join(ROOT, "tests", "host"),
                           "-I", os.path.join(ROOT, "splat.js_amd", "csrc"), "-o", str(exe), str(d / "probe.cpp")])
    return lambda mode: subprocess.run([str(exe), mode], stdout=subprocess.PIPE, text=True, timeout=100, check=True).stdout.split()


def test_every_block_arrives(probe):
    bad, most, bounded, left = map(int, probe("threads"))
    assert not bad and bounded and left == 0
    # four threads and the caller's: the stacks that the C library keeps
    assert most <= 5


def test_where_threads_cannot_be_started(probe):
    bad, most, bounded, left = map(int, probe("nothreads"))
    assert not bad and most == 1 and bounded and left == 0


def test_pinned_memory_that_cannot_be_had(probe):
    assert probe("nomem") == ["0", "0"]
