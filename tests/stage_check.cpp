// CPU check of the host transfers (lbgpu-prime-dev_amd/csrc/lbm_stage.hpp).
// The HIP calls that the header makes are defined here: memory is ordinary,
// device work runs where it is launched, and what the header asked for is
// recorded.  Argument: the check to run; prints "ok" or what was wrong.
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <thread>

#include "lbm_stage.hpp"

using namespace lbm;

static std::atomic<unsigned> g_host_flags{0}, g_event_flags{0};
static std::atomic<int> g_allocs{0}, g_frees{0}, g_events{0};
static std::atomic<size_t> g_most{SIZE_MAX};  // bytes of the largest pinned allocation granted

extern "C" {
hipError_t hipHostMalloc(void **p, size_t n, unsigned flags) {
  g_host_flags = flags;
  if (n > g_most) return hipErrorOutOfMemory;
  g_allocs++;
  *p = malloc(n);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p) {
  g_frees++;
  free(p);
  return hipSuccess;
}
hipError_t hipGetDevice(int *d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned flags) {
  g_event_flags = flags;
  *e = reinterpret_cast<hipEvent_t>(static_cast<uintptr_t>(++g_events));
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipMemcpyAsync(void *to, const void *from, size_t n, hipMemcpyKind, hipStream_t) {
  memcpy(to, from, n);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
}

#define CHECK(x)                                          \
  do {                                                    \
    if (!(x)) {                                           \
      printf("line %d: %s\n", __LINE__, #x);              \
      exit(1);                                            \
    }                                                     \
  } while (0)

// one array of comps components of N nodes, as a handle would move it
struct Array {
  long N;
  int comps;
  std::vector<double> gpu, host;
  hipEvent_t ev[kStageSlots] = {};
  bool pinned = true;
  Array(long N_, int comps_) : N(N_), comps(comps_), gpu((size_t)N_ * comps_), host((size_t)N_ * comps_) {}
  template <typename Wait>
  hipError_t move(bool up, Wait &&wait) {
    auto device = [&](const Piece &p, double *slot) {
      for (int c = 0; c < p.nc; c++) {
        double *g = gpu.data() + (p.c0 + c) * N + p.n0, *s = slot + (size_t)c * p.nn;
        if (up) memcpy(g, s, (size_t)p.nn * sizeof(double));
        else memcpy(s, g, (size_t)p.nn * sizeof(double));
      }
      return hipSuccess;
    };
    auto copy = [&](const Piece &p, double *slot) {
      wait();
      for (int c = 0; c < p.nc; c++) {
        double *h = host.data() + (p.c0 + c) * N + p.n0, *s = slot + (size_t)c * p.nn;
        if (up) memcpy(s, h, (size_t)p.nn * sizeof(double));
        else memcpy(h, s, (size_t)p.nn * sizeof(double));
      }
    };
    const hipError_t e = staged(pieces_of(comps, N), up, nullptr, ev, device, copy, pinned);
    if (pinned) return e;
    constexpr long room = 777;  // values of the handle's buffer
    double dev[room];
    return unpinned(pieces_of(comps, N, room), up, nullptr, dev, room, device, copy);
  }
  hipError_t move(bool up) {
    return move(up, [] {});
  }
  bool round_trip(double seed) {
    for (size_t q = 0; q < host.size(); q++) host[q] = seed + (double)q;
    if (move(true) != hipSuccess || gpu != host) return false;
    std::fill(host.begin(), host.end(), -1.0);
    return move(false) == hipSuccess && gpu == host;
  }
};

// what kernels and host threads read and write in turn has to be coherent,
// and the events behind which the host reads have to release to the system
static void coherent() {
  stage_join();
  CHECK(Array(1000, 3).round_trip(1.0));
  CHECK(g_host_flags & hipHostMallocCoherent);
  CHECK(!(g_host_flags & hipHostMallocNonCoherent));
  CHECK(g_event_flags & hipEventReleaseToSystem);
  CHECK(Array(700001, 5).round_trip(2.0));
  CHECK(g_host_flags & hipHostMallocCoherent);
  stage_leave();
  CHECK(g_allocs == g_frees);
}

// a system that pins no more memory, or none of the size wanted: the transfer
// goes without, and with again once there is some
static void refused() {
  stage_join();
  for (long N : {1L, 500L, 777L, 778L, 300000L}) {
    Array a(N, 4), b(N, 19);
    g_most = 0;
    CHECK(a.round_trip(1.0) && !a.pinned);
    CHECK(b.round_trip(2.0) && !b.pinned);
    g_most = SIZE_MAX;
    CHECK(a.round_trip(3.0) && a.pinned);
    CHECK(b.round_trip(4.0) && b.pinned);
    stage_leave();  // gives everything back
    stage_join();
  }
  stage_leave();
  CHECK(g_allocs == g_frees);
}

// a transfer that begins while another one runs does not wait for its end: it
// gets slots when the other is between two pieces, and memory that no one
// else uses meanwhile
static void beside() {
  stage_join();
  constexpr long N = kStageSlot / sizeof(double);
  Array large(N, 100), small(1000, 3);
  std::atomic<int> pieces{0}, done{0};
  std::thread t([&] {
    const hipError_t e = large.move(false, [&] {
      pieces++;
      std::this_thread::sleep_for(std::chrono::milliseconds(10));
    });
    CHECK(e == hipSuccess);
    done++;
  });
  while (pieces < 20) std::this_thread::yield();
  CHECK(small.round_trip(1.0));
  CHECK(done == 0 && pieces < 90);
  t.join();
  CHECK(pieces == 100);
  stage_leave();
  CHECK(g_allocs == g_frees);
}

// many transfers at once, more than there are slots, some refused memory;
// handles come and go beside them
static void crowd() {
  std::atomic<int> rounds{0};
  std::vector<std::thread> t;
  for (int q = 0; q < 12; q++)
    t.emplace_back([&, q] {
      for (int r = 0; r < 6; r++) {
        stage_join();
        Array a(q % 3 ? 1000 + 131 * q : 400000 + 7777 * q, 1 + (q + r) % 7);
        CHECK(a.round_trip(1000.0 * q + r));
        if (q == 0) g_most = r & 1 ? SIZE_MAX : kStageSlot - 1;
        stage_leave();
        rounds++;
      }
    });
  for (auto &x : t) x.join();
  CHECK(rounds == 72 && g_allocs == g_frees);
}

int main(int argc, char **argv) {
  const char *what = argc > 1 ? argv[1] : "";
  if (!strcmp(what, "coherent")) coherent();
  else if (!strcmp(what, "refused")) refused();
  else if (!strcmp(what, "beside")) beside();
  else if (!strcmp(what, "crowd")) crowd();
  else return 2;
  printf("ok\n");
  return 0;
}
