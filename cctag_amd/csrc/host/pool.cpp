// TaskPool (see pool.hpp).
#include "pool.hpp"

#include <algorithm>
#include <chrono>
#include <climits>
#include <cstdlib>
#include <map>
#include <memory>

namespace cctagx {
namespace {

inline void cpu_relax() {
#if defined(__x86_64__) || defined(__i386__)
  __builtin_ia32_pause();
#endif
}

// Spins (pause only: an idle sibling hardware thread should cost the busy
// one as little as possible) until done() or `micros` have passed.
// Returns done().
template <class F>
bool spin_until(F&& done, int micros) {
  using Clock = std::chrono::steady_clock;
  const auto t0 = Clock::now();
  for (int i = 0;; ++i) {
    if (done()) return true;
    if ((i & 255) == 255 &&
        std::chrono::duration_cast<std::chrono::microseconds>(Clock::now() - t0).count() >= micros)
      return done();
    cpu_relax();
  }
}

}  // namespace

TaskPool::TaskPool(int threads) {
  try {
    for (int i = 1; i < threads; ++i) workers_.emplace_back([this] { worker(); });
  } catch (...) {  // those started end before the exception goes on
    end();
    throw;
  }
}

TaskPool::~TaskPool() { end(); }

void TaskPool::end() {
  {
    std::lock_guard<std::mutex> lk(m_);
    stop_.store(true);
  }
  wake_.notify_all();
  for (std::thread& t : workers_) t.join();
}

int TaskPool::default_threads() {
  if (const char* s = std::getenv("CCTAGX_HOST_THREADS")) {
    const int v = std::atoi(s);
    if (v >= 1) return std::min(v, 256);
  }
  const int hw = (int)std::thread::hardware_concurrency();
  return std::max(1, std::min(hw, 16));
}

void TaskPool::drain(const std::function<void(int)>& fn, int n) {
  for (;;) {
    const int i = next_.fetch_add(1, std::memory_order_relaxed);
    if (i >= n) return;
    try {
      fn(i);
    } catch (...) {
      std::lock_guard<std::mutex> lk(m_);
      if (!error_) error_ = std::current_exception();
    }
  }
}

void TaskPool::worker() {
  uint64_t seen = 0;
  for (;;) {
    if (!spin_until([&] { return stop_.load() || gen_.load() != seen; }, kIdleSpinMicros)) {
      std::unique_lock<std::mutex> lk(m_);
      wake_.wait(lk, [&] { return stop_.load() || gen_.load() != seen; });
    }
    if (stop_.load()) return;
    seen = gen_.load();
    busy_.fetch_add(1);
    const std::function<void(int)>* fn = fn_.load();
    if (fn) drain(*fn, n_.load());
    busy_.fetch_sub(1);
    if (caller_waits_.load()) {
      { std::lock_guard<std::mutex> lk(m_); }
      done_.notify_all();
    }
  }
}

void TaskPool::run(int n, const std::function<void(int)>& fn) {
  if (n <= 0) return;
  if (workers_.empty() || n == 1) {
    for (int i = 0; i < n; ++i) fn(i);
    return;
  }
  // a worker still leaving the previous job must not see this one's fields
  // half written
  spin_until([&] { return busy_.load() == 0; }, kWaitSpinMicros);
  while (busy_.load() != 0) std::this_thread::yield();
  n_.store(n);
  next_.store(0);
  error_ = nullptr;
  fn_.store(&fn);
  {
    std::lock_guard<std::mutex> lk(m_);
    gen_.fetch_add(1);
  }
  wake_.notify_all();
  drain(fn, n);
  // every index is handed out; wait for the workers still inside the job
  if (!spin_until([&] { return busy_.load() == 0; }, kWaitSpinMicros)) {
    std::unique_lock<std::mutex> lk(m_);
    caller_waits_.store(true);
    done_.wait(lk, [&] { return busy_.load() == 0; });
    caller_waits_.store(false);
  }
  fn_.store(nullptr);
  std::exception_ptr err;
  {
    std::lock_guard<std::mutex> lk(m_);
    err = error_;
    error_ = nullptr;
  }
  if (err) std::rethrow_exception(err);
}

namespace {
struct PoolShelf {
  int places = 0, pools = 0;          // pools: leased and idle
  int most = INT_MAX;                 // pools that could be started when it was last tried
  std::vector<std::unique_ptr<TaskPool>> idle;  // the last one was used last
};
struct PoolShelves {
  std::mutex m;
  std::map<int, PoolShelf> of;  // by thread count
};
// (never destroyed: handles may outlive static destruction)
PoolShelves& shelves() {
  static PoolShelves* s = new PoolShelves;
  return *s;
}

// Threads may have become free, or scarce: starting one is worth a try again.
void try_again(PoolShelves& all) {
  for (auto& s : all.of) s.second.most = INT_MAX;
}

// A place more for pools of `threads`, and its first pool when there is none.
// Throws, with nothing changed, when the pool's threads cannot be started.
void enter(int threads) {
  PoolShelves& all = shelves();
  std::unique_lock<std::mutex> lk(all.m);
  PoolShelf& s = all.of[threads];
  s.idle.reserve(s.places + 1);  // a lease's end allocates nothing
  ++s.places;
  try_again(all);
  if (s.pools > 0) return;
  ++s.pools;
  lk.unlock();
  std::unique_ptr<TaskPool> pool;
  try {
    pool = std::make_unique<TaskPool>(threads);
  } catch (...) {
    lk.lock();
    --s.pools;
    --s.places;
    throw;
  }
  lk.lock();
  s.idle.push_back(std::move(pool));
}

void leave(int threads) {
  std::unique_ptr<TaskPool> ended;  // joined outside the lock
  PoolShelves& all = shelves();
  std::lock_guard<std::mutex> lk(all.m);
  PoolShelf& s = all.of[threads];
  --s.places;
  if (s.pools > s.places && !s.idle.empty()) {
    ended = std::move(s.idle.front());
    s.idle.erase(s.idle.begin());
    --s.pools;
  }
  try_again(all);
}
}  // namespace

void PoolPlace::set(int threads) {
  if (threads < 1) threads = 1;
  if (threads == threads_) return;
  if (threads > 1) enter(threads);
  if (threads_ > 1) leave(threads_);
  threads_ = threads;
}

PoolLease::PoolLease(const PoolPlace& place) {
  const int threads = place.threads();
  if (threads <= 1) return;
  PoolShelves& all = shelves();
  std::unique_lock<std::mutex> lk(all.m);
  PoolShelf& s = all.of[threads];
  if (!s.idle.empty()) {
    pool_ = s.idle.back().release();
    s.idle.pop_back();
    return;
  }
  if (s.pools >= s.most) return;
  ++s.pools;
  lk.unlock();
  try {
    pool_ = new TaskPool(threads);
  } catch (const std::exception&) {
    lk.lock();
    s.most = --s.pools;
  }
}

PoolLease::~PoolLease() {
  if (!pool_) return;
  std::unique_ptr<TaskPool> pool(pool_);  // (joined outside the lock when its place has gone)
  PoolShelves& all = shelves();
  std::lock_guard<std::mutex> lk(all.m);
  PoolShelf& s = all.of[pool->threads()];
  if (s.pools > s.places) --s.pools;
  else s.idle.push_back(std::move(pool));
}

int pools_alive(int threads) {
  PoolShelves& all = shelves();
  std::lock_guard<std::mutex> lk(all.m);
  return all.of[threads].pools;
}

void parallel_for(TaskPool* pool, int n, const std::function<void(int)>& fn) {
  if (pool) {
    pool->run(n, fn);
  } else {
    for (int i = 0; i < n; ++i) fn(i);
  }
}

}  // namespace cctagx
