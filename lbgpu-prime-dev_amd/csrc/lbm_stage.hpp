// Host arrays to and from the GPU through pinned memory.
//
// Fields and populations cross the C ABI as dense FP64 arrays in the
// caller's ordinary memory.  The GPU expands or compacts them (k_dense_*)
// while it writes or reads pinned slots directly, and a few host threads copy
// between the slots and the caller's array, each with a slot of its own, so
// that the bus and the copies (for a fresh array mostly the cost of its first
// touch) run together.
//
// Without pinned memory (the system refuses to pin more) transfers go through a
// small device buffer of the handle and ordinary copies instead.
//
// Slots and threads are one set per process, made on first use, at most
// kStageSlots * kStageSlot bytes and kStageSlots - 1 threads, released with the
// last handle.  A transfer holds them from start to end; transfers of other
// threads wait.
#pragma once

#include <hip/hip_runtime_api.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <functional>
#include <mutex>
#include <thread>
#include <vector>

namespace lbm {

constexpr int kStageSlots = 8;              // slots, and host threads at most
constexpr size_t kStageSlot = 2u << 20;     // bytes of a slot
// One thread (the caller's first) for each MiB: a thread moves a MiB in 60 us
// (fields of 1.3 MB: 0.062 ms alone; 2.9 MB: 0.109 ms with two, 0.13 alone).
// 1 GB of fields: 20 GB/s with two threads, 33 with four, 44 with six, 47 with
// eight.
constexpr size_t kStageAlone = 1u << 20;

struct Stage {
  std::mutex mu;   // held for a whole transfer
  int users = 0;
  char *buf = nullptr;
  size_t bytes = 0;

  // Helper threads, started by the first transfer that wants them, asleep
  // between transfers, ended with the last handle.  The caller works too and
  // waits only for helpers that have begun: on a machine whose cores are all
  // busy (a BLAS pool still spinning after the caller's last product) a
  // thread that has to be started or joined costs a scheduler tick, 4 ms a
  // transfer where 18 MB take 0.7.
  std::mutex jm;
  std::condition_variable wake, idle;
  std::vector<std::thread> threads;
  const std::function<void(int)> *job = nullptr;
  int next = 0, most = 0, begun = 0;  // slots given out and to give, helpers at work
  bool stop = false;

  void helper() {
    std::unique_lock<std::mutex> lock(jm);
    for (;;) {
      wake.wait(lock, [&] { return stop || (job && next < most); });
      if (stop) return;
      const std::function<void(int)> *const mine = job;
      const int slot = next++;
      begun++;
      lock.unlock();
      (*mine)(slot);
      lock.lock();
      if (--begun == 0) idle.notify_all();
    }
  }
  // fn(0) here, fn(1) .. fn(workers - 1) on helpers that come in time
  void run(const std::function<void(int)> &fn, int workers) {
    if (workers > 1) {
      std::lock_guard<std::mutex> lock(jm);
      try {
        while ((int)threads.size() < workers - 1) threads.emplace_back([this] { helper(); });
      } catch (const std::exception &) {
        // fewer helpers: the others take their share
      }
      job = &fn;
      next = 1;
      most = workers;
    }
    if (workers > 1) wake.notify_all();
    fn(0);
    if (workers > 1) {
      std::unique_lock<std::mutex> lock(jm);
      job = nullptr;
      idle.wait(lock, [&] { return begun == 0; });
    }
  }
  void end_threads() {
    {
      std::lock_guard<std::mutex> lock(jm);
      stop = true;
    }
    wake.notify_all();
    for (auto &t : threads) t.join();
    threads.clear();
    stop = false;
  }
};
// never destroyed: a process may end with handles open
inline Stage &stage() {
  static Stage *const s = new Stage;
  return *s;
}
inline void stage_join() {
  std::lock_guard<std::mutex> lock(stage().mu);
  stage().users++;
}
inline void stage_leave() {
  Stage &s = stage();
  std::lock_guard<std::mutex> lock(s.mu);
  if (--s.users > 0) return;
  s.end_threads();
  if (s.buf) (void)hipHostFree(s.buf);
  s.buf = nullptr;
  s.bytes = 0;
}

// at least `bytes` (up to all slots) of pinned memory; false when the system
// gives none; s.mu is held
inline bool stage_hold(Stage &s, size_t bytes) {
  if (s.bytes >= bytes) return true;
  if (s.buf) (void)hipHostFree(s.buf);
  s.buf = nullptr;
  s.bytes = 0;
  // small transfers share one slot, others get all of them
  const size_t want = bytes <= kStageSlot ? kStageSlot : kStageSlot * kStageSlots;
  // coherent, whatever HIP_HOST_COHERENT says: kernels and host threads read
  // and write a slot in turn while the process runs on
  const hipError_t e = hipHostMalloc((void **)&s.buf, want, hipHostMallocPortable | hipHostMallocCoherent);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    s.buf = nullptr;
    return false;
  }
  s.bytes = want;
  return true;
}

// One piece of a transfer: nc components of nn nodes from node n0, at most a
// slot's worth; host moves it between the slot and the caller's memory,
// device (when there is device work) launches the kernel on the slot.
struct Piece {
  int c0, nc;
  long n0, nn;
};

// the pieces of comps components of N nodes each, at most `most` values in one
inline std::vector<Piece> pieces_of(int comps, long N, long most = (long)(kStageSlot / sizeof(double))) {
  std::vector<Piece> v;
  if (N <= most) {
    const int group = (int)std::min<long>(comps, std::max<long>(1, most / N));
    for (int c = 0; c < comps; c += group) v.push_back({c, std::min(group, comps - c), 0, N});
  } else {
    for (int c = 0; c < comps; c++)
      for (long n = 0; n < N; n += most) v.push_back({c, 1, n, std::min(most, N - n)});
  }
  return v;
}

// Moves all pieces: device(piece, slot) launches on `stream` and returns a
// hipError_t, host(piece, slot) copies; up: host memory to the GPU.  events:
// kStageSlots events of the caller, created here when null.  pinned: false
// when there was no pinned memory and nothing has been moved.
template <typename Device, typename Host>
hipError_t staged(const std::vector<Piece> &pieces, bool up, hipStream_t stream, hipEvent_t *events, Device &&device,
                  Host &&host, bool &pinned) {
  pinned = true;
  size_t total = 0, largest = 0;
  for (const Piece &p : pieces) {
    const size_t b = (size_t)p.nc * p.nn * sizeof(double);
    total += b;
    largest = std::max(largest, b);
  }
  if (!total) return hipSuccess;
  const int n = (int)pieces.size();
  const int workers = (int)std::max<size_t>(1, std::min<size_t>(std::min(kStageSlots, n), total / kStageAlone));
  const size_t slot = (largest + 255) & ~(size_t)255;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  Stage &s = stage();
  std::lock_guard<std::mutex> lock(s.mu);
  if (!stage_hold(s, slot * workers)) {
    pinned = false;
    return hipSuccess;
  }
  for (int w = 0; w < workers; w++)
    // the host reads the slot behind the event: its writes are released to the system
    if (!events[w] &&
        (e = hipEventCreateWithFlags(&events[w], hipEventDisableTiming | hipEventReleaseToSystem)) != hipSuccess)
      return e;
  std::atomic<int> next{0}, bad{(int)hipSuccess};
  auto work = [&](int w) {
    hipError_t r = hipSetDevice(dev);
    char *const at = s.buf + w * slot;
    bool busy = false;
    for (int c; r == hipSuccess && bad.load() == (int)hipSuccess && (c = next.fetch_add(1)) < n;) {
      const Piece &p = pieces[c];
      if (up) {
        if (busy) r = hipEventSynchronize(events[w]);
        if (r == hipSuccess) host(p, (double *)at);
      }
      if (r == hipSuccess) r = device(p, (double *)at);
      if (r == hipSuccess) r = hipEventRecord(events[w], stream);
      busy = r == hipSuccess;
      if (!up) {
        if (r == hipSuccess) r = hipEventSynchronize(events[w]);
        busy = false;
        if (r == hipSuccess) host(p, (double *)at);
      }
    }
    if (r != hipSuccess) bad.store((int)r);
  };
  s.run(work, workers);
  // the slots are free again once the GPU has read them
  e = hipStreamSynchronize(stream);
  return bad.load() != (int)hipSuccess ? (hipError_t)bad.load() : e;
}

// The same without pinned memory, one piece after the other: dev is device
// memory of `values` doubles that holds any of the pieces, and the host's side
// of a piece is ordinary memory.
template <typename Device, typename Host>
hipError_t unpinned(const std::vector<Piece> &pieces, bool up, hipStream_t stream, double *dev, long values,
                    Device &&device, Host &&host) {
  std::vector<double> buf((size_t)values);
  for (const Piece &p : pieces) {
    const size_t bytes = (size_t)p.nc * p.nn * sizeof(double);
    hipError_t e;
    if (up) {
      host(p, buf.data());
      if ((e = hipMemcpyAsync(dev, buf.data(), bytes, hipMemcpyHostToDevice, stream)) != hipSuccess) return e;
      if ((e = device(p, dev)) != hipSuccess) return e;
      if ((e = hipStreamSynchronize(stream)) != hipSuccess) return e;
    } else {
      if ((e = device(p, dev)) != hipSuccess) return e;
      if ((e = hipMemcpyAsync(buf.data(), dev, bytes, hipMemcpyDeviceToHost, stream)) != hipSuccess) return e;
      if ((e = hipStreamSynchronize(stream)) != hipSuccess) return e;
      host(p, buf.data());
    }
  }
  return hipSuccess;
}

}  // namespace lbm
