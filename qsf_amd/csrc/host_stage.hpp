// host_stage.hpp — large states between the device and caller memory, through pinned slots.
//
// A plain copy to pageable memory ran at 10 GB/s (512^3 FP64, 2 GiB: 210 ms beside 561 ms for 150
// steps): one thread takes the destination's page faults and the copy out of the runtime's own
// staging. Here the device writes pieces into a ring of pinned slots and several host threads copy
// (or, for an FP32 state, widen) them out, so the faults and copies run side by side with the
// transfer, and an FP32 state crosses the bus in its own four bytes a value. The way up is the same
// with the roles exchanged.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace qsf {

// Owned by one context; 24 MiB of pinned memory from the first large state on, given back with it.
class HostStage {
  static constexpr size_t kSlotBytes = size_t(2) << 20;
  static constexpr int kSlots = 12, kThreads = 8;
  std::mutex use_;   // one state at a time
  char* mem_ = nullptr;
  hipEvent_t ev_[kSlots] = {};
  int events_ = 0;

  hipError_t prepare() {
    if (!mem_) {
      void* p = nullptr;
      if (hipError_t e = hipHostMalloc(&p, kSlotBytes * kSlots, hipHostMallocDefault); e != hipSuccess) return e;
      mem_ = static_cast<char*>(p);
    }
    for (; events_ < kSlots; ++events_)
      if (hipError_t e = hipEventCreateWithFlags(&ev_[events_], hipEventDisableTiming); e != hipSuccess) return e;
    return hipSuccess;
  }

 public:
  // Below this the plain copy is as fast (its pages are few), and the slots are not needed.
  static constexpr int64_t kLeastBytes = int64_t(16) << 20;

  HostStage() = default;
  HostStage(const HostStage&) = delete;
  HostStage& operator=(const HostStage&) = delete;
  ~HostStage() {
    for (int k = 0; k < events_; ++k) (void)hipEventDestroy(ev_[k]);
    if (mem_) (void)hipHostFree(mem_);
  }

  // `count` reals at device address `src` (float where `widen`, else double) to dst as doubles, after
  // what the stream holds; complete on return.
  hipError_t read(double* dst, const void* src, int64_t count, bool widen, hipStream_t s) {
    std::lock_guard<std::mutex> one(use_);
    if (hipError_t e = prepare(); e != hipSuccess) return e;
    const int64_t unit = widen ? 4 : 8, per = (int64_t)kSlotBytes / unit;
    const int64_t chunks = (count + per - 1) / per;
    std::mutex mu;
    std::condition_variable cv;
    std::vector<char> done((size_t)chunks, 0);
    int64_t next = 0, landed = 0;   // chunks taken by the threads; chunks that are in their slots
    bool stop = false;
    auto out = [&](int64_t c) {   // chunk c from its slot to its place
      const char* from = mem_ + (size_t)(c % kSlots) * kSlotBytes;
      const int64_t k = std::min(per, count - c * per);
      double* to = dst + c * per;
      if (widen) {
        const float* f = reinterpret_cast<const float*>(from);
        for (int64_t i = 0; i < k; ++i) to[i] = (double)f[i];
      } else {
        std::memcpy(to, from, (size_t)k * 8);
      }
    };
    auto fetch = [&](int64_t c) {
      return hipMemcpyAsync(mem_ + (size_t)(c % kSlots) * kSlotBytes, static_cast<const char*>(src) + c * per * unit,
                            (size_t)(std::min(per, count - c * per) * unit), hipMemcpyDeviceToHost, s);
    };
    auto work = [&] {
      std::unique_lock<std::mutex> lk(mu);
      while (next < chunks) {
        const int64_t c = next++;
        cv.wait(lk, [&] { return landed > c || stop; });
        if (stop) return;
        lk.unlock();
        out(c);
        lk.lock();
        done[(size_t)c] = 1;
        cv.notify_all();
      }
    };
    std::vector<std::thread> threads;
    hipError_t err = hipSuccess;
    try {
      threads.reserve(kThreads);
      const int most = (int)std::min<int64_t>(kThreads, chunks);
      while ((int)threads.size() < most) threads.emplace_back(work);
    } catch (const std::exception&) {   // as many as could be started
    }
    int64_t issued = 0;
    if (threads.empty()) {   // none: chunk by chunk here
      for (int64_t c = 0; c < chunks; ++c) {
        err = fetch(c);
        if (hipError_t e = hipStreamSynchronize(s); err == hipSuccess) err = e;
        if (err != hipSuccess) return err;
        out(c);
      }
      return hipSuccess;
    }
    for (int64_t ready = 0; ready < chunks && err == hipSuccess;) {
      while (issued < chunks && err == hipSuccess) {
        if (issued >= kSlots) {
          std::unique_lock<std::mutex> lk(mu);
          if (!done[(size_t)(issued - kSlots)]) {
            if (issued > ready) break;   // a piece on its way is waited for first
            cv.wait(lk, [&] { return done[(size_t)(issued - kSlots)] != 0; });
          }
        }
        err = fetch(issued);
        if (err == hipSuccess) err = hipEventRecord(ev_[issued % kSlots], s);
        if (err == hipSuccess) ++issued;
      }
      if (err != hipSuccess) break;
      err = hipEventSynchronize(ev_[ready % kSlots]);
      if (err != hipSuccess) break;
      ++ready;
      std::lock_guard<std::mutex> lk(mu);
      landed = ready;
      cv.notify_all();
    }
    {
      std::lock_guard<std::mutex> lk(mu);
      if (err != hipSuccess) stop = true;
      cv.notify_all();
    }
    for (auto& t : threads) t.join();
    if (err != hipSuccess) (void)hipStreamSynchronize(s);   // no copy into a slot is left behind
    return err;
  }

  // `count` doubles at src to device address `dst` (rounded to float where `narrow`); complete on return.
  hipError_t write(void* dst, const double* src, int64_t count, bool narrow, hipStream_t s) {
    std::lock_guard<std::mutex> one(use_);
    if (hipError_t e = prepare(); e != hipSuccess) return e;
    const int64_t unit = narrow ? 4 : 8, per = (int64_t)kSlotBytes / unit;
    const int64_t chunks = (count + per - 1) / per;
    std::mutex mu;
    std::condition_variable cv;
    std::vector<char> filled((size_t)chunks, 0);
    int64_t next = 0, freed = 0;   // chunks taken by the threads; chunks whose slots are free again
    bool stop = false;
    auto in = [&](int64_t c) {   // chunk c into its slot
      char* to = mem_ + (size_t)(c % kSlots) * kSlotBytes;
      const int64_t k = std::min(per, count - c * per);
      const double* from = src + c * per;
      if (narrow) {
        float* f = reinterpret_cast<float*>(to);
        for (int64_t i = 0; i < k; ++i) f[i] = (float)from[i];
      } else {
        std::memcpy(to, from, (size_t)k * 8);
      }
    };
    auto work = [&] {
      std::unique_lock<std::mutex> lk(mu);
      while (next < chunks) {
        const int64_t c = next++;
        cv.wait(lk, [&] { return c < freed + kSlots || stop; });
        if (stop) return;
        lk.unlock();
        in(c);
        lk.lock();
        filled[(size_t)c] = 1;
        cv.notify_all();
      }
    };
    std::vector<std::thread> threads;
    try {
      threads.reserve(kThreads);
      const int most = (int)std::min<int64_t>(kThreads, chunks);
      while ((int)threads.size() < most) threads.emplace_back(work);
    } catch (const std::exception&) {   // as many as could be started
    }
    const bool alone = threads.empty();
    hipError_t err = hipSuccess;
    for (int64_t c = 0; c < chunks && err == hipSuccess; ++c) {
      // the threads may run up to kThreads chunks ahead: the transfers before those are waited for
      const int64_t over = alone ? c - kSlots : c - (kSlots - kThreads);
      if (over >= 0) {
        err = hipEventSynchronize(ev_[over % kSlots]);
        if (err != hipSuccess) break;
        std::lock_guard<std::mutex> lk(mu);
        freed = over + 1;
        cv.notify_all();
      }
      if (alone) {
        in(c);
      } else {
        std::unique_lock<std::mutex> lk(mu);
        cv.wait(lk, [&] { return filled[(size_t)c] != 0; });
      }
      err = hipMemcpyAsync(static_cast<char*>(dst) + c * per * unit, mem_ + (size_t)(c % kSlots) * kSlotBytes,
                           (size_t)(std::min(per, count - c * per) * unit), hipMemcpyHostToDevice, s);
      if (err == hipSuccess) err = hipEventRecord(ev_[c % kSlots], s);
    }
    {
      std::lock_guard<std::mutex> lk(mu);
      if (err != hipSuccess) stop = true;
      cv.notify_all();
    }
    for (auto& t : threads) t.join();
    const hipError_t e = hipStreamSynchronize(s);   // the slots are free again
    return err != hipSuccess ? err : e;
  }
};

}  // namespace qsf
