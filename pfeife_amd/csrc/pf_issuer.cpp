// Issues a step's jobs (captured graphs, with the events between their streams) from a thread of its own.
//
// A hipGraphLaunch costs the host some 24 us and an event record or wait 3-10 us; a step of a small model makes
// hundreds of them, in between runs of user code (loss, backward hooks) that hold the Python interpreter.  Both take
// about the same time, and neither needs the other to be finished: the caller hands jobs over in the order they are
// to be issued, goes on with user code, and waits only for the job whose result that code reads.
#include <atomic>
#include <condition_variable>
#include <deque>
#include <exception>
#include <mutex>
#include <string>
#include <thread>

#include "pf_common.h"

namespace {

struct Span {
  const pf_job* jobs;
  int n;
};

struct Issuer {
  explicit Issuer(int device) : device_(device), thread_([this] { run(); }) {}
  ~Issuer() {
    {
      std::lock_guard<std::mutex> lock(mutex_);
      stop_ = true;
    }
    work_.notify_one();
    thread_.join();
  }
  int64_t push(const pf_job* jobs, int n) {
    int64_t ticket;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      queue_.push_back(Span{jobs, n});
      ticket = handed_.load(std::memory_order_relaxed) + n;
      handed_.store(ticket, std::memory_order_release);
    }
    work_.notify_one();
    return ticket;
  }
  void wait(int64_t ticket) {
    for (int i = 0; i < SPIN; ++i) {
      if (issued_.load(std::memory_order_acquire) >= ticket) return;
      __builtin_ia32_pause();
    }
    std::unique_lock<std::mutex> lock(mutex_);
    done_.wait(lock, [&] { return issued_.load(std::memory_order_acquire) >= ticket; });
  }
  // the first failure since the last call ("" if none); later jobs are issued all the same
  std::string take_error() {
    std::lock_guard<std::mutex> lock(mutex_);
    std::string e;
    e.swap(error_);
    return e;
  }

 private:
  static constexpr int SPIN = 2000;   // (some 50 us: a sleeping thread takes about as long to wake)

  void fail(const char* what, hipError_t e) {
    std::lock_guard<std::mutex> lock(mutex_);
    if (error_.empty()) error_ = std::string(what) + ": " + hipGetErrorString(e);
  }
  void issue(const pf_job& j) {
    hipStream_t st = (hipStream_t)j.stream;
    hipError_t e;
    for (int i = 0; i < j.n_waits; ++i)
      if ((e = hipStreamWaitEvent(st, (hipEvent_t)j.waits[i], 0)) != hipSuccess) fail("wait", e);
    if (j.graph && (e = hipGraphLaunch((hipGraphExec_t)j.graph, st)) != hipSuccess) fail("graph launch", e);
    if (j.record && (e = hipEventRecord((hipEvent_t)j.record, st)) != hipSuccess) fail("record", e);
  }
  void run() {
    hipError_t e = hipSetDevice(device_);
    if (e != hipSuccess) fail("hipSetDevice", e);
    int64_t taken = 0;
    for (;;) {
      for (int i = 0; i < SPIN && handed_.load(std::memory_order_acquire) == taken; ++i) __builtin_ia32_pause();
      Span s;
      {
        std::unique_lock<std::mutex> lock(mutex_);
        work_.wait(lock, [&] { return stop_ || !queue_.empty(); });
        if (queue_.empty()) return;
        s = queue_.front();
        queue_.pop_front();
      }
      for (int i = 0; i < s.n; ++i) {
        issue(s.jobs[i]);
        issued_.store(++taken, std::memory_order_release);
      }
      {
        std::lock_guard<std::mutex> lock(mutex_);   // (a waiter is either before its check or asleep)
      }
      done_.notify_all();
    }
  }

  const int device_;
  std::mutex mutex_;
  std::condition_variable work_, done_;
  std::deque<Span> queue_;
  std::atomic<int64_t> handed_{0}, issued_{0};
  std::string error_;
  bool stop_ = false;
  std::thread thread_;   // (last: it runs as soon as it is constructed)
};

}  // namespace

extern "C" int pf_issuer_create(int device, void** out) {
  PF_REQUIRE(out != nullptr, "pf_issuer_create: null result pointer");
  try {
    *out = new Issuer(device);
  } catch (const std::exception& e) {   // no memory, or no thread to be had
    *out = nullptr;
    pf_set_error("pf_issuer_create: %s", e.what());
    return PF_ERR_HIP;
  }
  return PF_OK;
}

extern "C" int pf_issuer_push(void* issuer, const pf_job* jobs, int n, int64_t* ticket) {
  PF_REQUIRE(issuer && ticket && n >= 0 && (jobs || n == 0), "pf_issuer_push: bad arguments");
  for (int i = 0; i < n; ++i)
    PF_REQUIRE(jobs[i].stream && jobs[i].n_waits >= 0 && (jobs[i].waits || jobs[i].n_waits == 0), "pf_issuer_push: bad job %d", i);
  try {
    *ticket = ((Issuer*)issuer)->push(jobs, n);
  } catch (const std::exception& e) {
    pf_set_error("pf_issuer_push: %s", e.what());
    return PF_ERR_HIP;
  }
  return PF_OK;
}

extern "C" int pf_issuer_wait(void* issuer, int64_t ticket) {
  PF_REQUIRE(issuer != nullptr, "pf_issuer_wait: null issuer");
  ((Issuer*)issuer)->wait(ticket);
  const std::string e = ((Issuer*)issuer)->take_error();
  if (!e.empty()) {
    pf_set_error("pf_issuer_wait: %s", e.c_str());
    return PF_ERR_HIP;
  }
  return PF_OK;
}

extern "C" int pf_issuer_destroy(void* issuer) {
  delete (Issuer*)issuer;
  return PF_OK;
}

extern "C" int pf_event_create(void** out) {
  PF_REQUIRE(out != nullptr, "pf_event_create: null result pointer");
  hipEvent_t ev = nullptr;
  const hipError_t e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
  if (e != hipSuccess) {
    pf_set_error("pf_event_create: %s", hipGetErrorString(e));
    return PF_ERR_HIP;
  }
  *out = (void*)ev;
  return PF_OK;
}

extern "C" int pf_event_destroy(void* event) {
  if (event) (void)hipEventDestroy((hipEvent_t)event);
  return PF_OK;
}
