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
// kStageSlots slots of kStageSlot bytes and kStageSlots - 1 threads, released
// with the last handle.  Transfers of several threads share them: each has a
// slot at least from its start to its end (the ninth at once waits for one),
// and takes up to its share of the others; a transfer that has more than its
// share gives slots back between pieces when another has less.  (2 MB of
// fields from two threads 0.15 ms each, from four 0.20, where whole transfers
// one after the other took 0.21 and 0.43; a sample beside another handle's
// 131 MB 0.08 ms against 2.8.)
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
  // one transfer: fn(slot) moves pieces through a slot until there are none
  // left or the slot is wanted elsewhere
  struct Job {
    const std::function<void(int)> *fn = nullptr;
    int want = 1;   // slots it can use
    int held = 0;   // slots it has
    int begun = 0;  // helpers at work on it
  };
  struct Task {
    Job *job;
    int slot;
  };

  std::mutex life;  // handles come and go: users, and the release with the last
  int users = 0;

  std::mutex mu;  // everything below but the memory, which belongs to the slot's holder
  std::condition_variable freed, wake, idle;
  char *buf[kStageSlots] = {};
  bool out[kStageSlots] = {};
  std::vector<Job *> jobs;
  // Helper threads, started by the first transfer that wants them, asleep
  // between transfers, ended with the last handle.  The caller works too and
  // waits only for helpers that have begun: on a machine whose cores are all
  // busy (a BLAS pool still spinning after the caller's last product) a
  // thread that has to be started or joined costs a scheduler tick, 4 ms a
  // transfer where 18 MB take 0.7.
  std::vector<std::thread> threads;
  std::vector<Task> tasks;  // slots given to a job whose helper has not come yet
  bool stop = false;

  int share() const { return std::max(1, kStageSlots / (int)std::max<size_t>(1, jobs.size())); }
  int take() {
    for (int s = 0; s < kStageSlots; s++)
      if (!out[s]) {
        out[s] = true;
        return s;
      }
    return -1;
  }
  void give(Job &j, int slot) {
    out[slot] = false;
    j.held--;
    freed.notify_one();
  }
  // slots and helpers up to the job's share
  void grow(Job &j) {
    while (j.held < std::min(j.want, share())) {
      const int slot = take();
      if (slot < 0) return;
      j.held++;
      try {
        // a slot for the caller of each job, the others for helpers
        if (threads.size() < (size_t)kStageSlots - 1 && threads.size() < busy() + 1)
          threads.emplace_back([this] { helper(); });
        tasks.push_back({&j, slot});
      } catch (const std::exception &) {
        give(j, slot);  // fewer helpers: the others take their share
        return;
      }
      wake.notify_one();
    }
  }
  // helpers that have or will have work
  size_t busy() const {
    size_t n = tasks.size();
    for (const Job *j : jobs) n += (size_t)j->begun;
    return n;
  }
  void helper() {
    std::unique_lock<std::mutex> lock(mu);
    for (;;) {
      wake.wait(lock, [&] { return stop || !tasks.empty(); });
      if (stop) return;
      const Task t = tasks.back();
      tasks.pop_back();
      t.job->begun++;
      lock.unlock();
      (*t.job->fn)(t.slot);
      lock.lock();
      give(*t.job, t.slot);
      if (--t.job->begun == 0) idle.notify_all();
    }
  }
  // Between two pieces: whether the holder of one of the job's slots goes on.
  // The caller always does, and takes what it lacks of its share.
  bool stay(Job &j, bool caller) {
    std::lock_guard<std::mutex> lock(mu);
    if (caller) {
      grow(j);
      return true;
    }
    if (j.held <= share()) return true;
    for (const Job *o : jobs)
      if (o->held < std::min(o->want, share())) return false;
    return true;
  }
  // no memory for a slot: the others take its share
  void less(Job &j) {
    std::lock_guard<std::mutex> lock(mu);
    j.want = std::max(1, j.want - 1);
  }
  // the memory of a slot that the caller of this holds
  char *memory(int slot) {
    if (buf[slot]) return buf[slot];
    // coherent, whatever HIP_HOST_COHERENT says: kernels and host threads read
    // and write a slot in turn while the process runs on
    void *p = nullptr;
    if (hipHostMalloc(&p, kStageSlot, hipHostMallocPortable | hipHostMallocCoherent) != hipSuccess) {
      (void)hipGetLastError();
      return nullptr;
    }
    return buf[slot] = (char *)p;
  }
};
// never destroyed: a process may end with handles open
inline Stage &stage() {
  static Stage *const s = new Stage;
  return *s;
}
inline void stage_join() {
  Stage &s = stage();
  std::lock_guard<std::mutex> lock(s.life);
  s.users++;
}
inline void stage_leave() {
  Stage &s = stage();
  std::lock_guard<std::mutex> lock(s.life);
  if (--s.users > 0) return;
  {
    std::lock_guard<std::mutex> l(s.mu);
    s.stop = true;
  }
  s.wake.notify_all();
  for (auto &t : s.threads) t.join();
  s.threads.clear();
  s.stop = false;
  for (char *&b : s.buf) {
    if (b) (void)hipHostFree(b);
    b = nullptr;
  }
}

// A transfer's first slot, from its start to its end
struct StageLease {
  Stage &s;
  Stage::Job &job;
  int slot = -1;
  StageLease(Stage &s_, Stage::Job &j) : s(s_), job(j) {
    std::unique_lock<std::mutex> lock(s.mu);
    s.jobs.push_back(&job);
    s.freed.wait(lock, [&] { return (slot = s.take()) >= 0; });
    job.held++;
  }
  StageLease(const StageLease &) = delete;
  ~StageLease() {
    std::unique_lock<std::mutex> lock(s.mu);
    // slots whose helper has not come, and helpers that have begun
    for (size_t q = 0; q < s.tasks.size();)
      if (s.tasks[q].job == &job) {
        s.give(job, s.tasks[q].slot);
        s.tasks.erase(s.tasks.begin() + (long)q);
      } else {
        q++;
      }
    s.idle.wait(lock, [&] { return job.begun == 0; });
    s.give(job, slot);
    s.jobs.erase(std::find(s.jobs.begin(), s.jobs.end(), &job));
  }
};

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
  if (largest > kStageSlot) return hipErrorInvalidValue;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  Stage &s = stage();
  std::atomic<int> next{0}, bad{(int)hipSuccess};
  Stage::Job job;
  job.want = (int)std::max<size_t>(1, std::min<size_t>(std::min(kStageSlots, n), total / kStageAlone));
  int first = -1;
  const std::function<void(int)> work = [&](int w) {
    const bool caller = w == first;
    char *const at = s.memory(w);
    if (!at) {
      s.less(job);
      return;
    }
    hipError_t r = hipSetDevice(dev);
    // the host reads the slot behind the event: its writes are released to the system
    if (r == hipSuccess && !events[w])
      r = hipEventCreateWithFlags(&events[w], hipEventDisableTiming | hipEventReleaseToSystem);
    bool busy = false;  // the GPU may still read the slot
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
      if (r == hipSuccess && !s.stay(job, caller)) break;
    }
    // a slot is given back free; the caller waits for the whole stream below
    if (!caller) {
      if (r != hipSuccess) (void)hipStreamSynchronize(stream);
      else if (busy) r = hipEventSynchronize(events[w]);
    }
    if (r != hipSuccess) bad.store((int)r);
  };
  {
    job.fn = &work;
    StageLease lease(s, job);
    first = lease.slot;
    if (!s.memory(first)) {
      pinned = false;
      return hipSuccess;
    }
    s.stay(job, true);
    work(first);
    e = hipStreamSynchronize(stream);
  }
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
