// Iterations on bitmaps (run_step_dense) on the host: the dense_* launches run
// in order on a thread that stands in for the device, so the host side polls,
// grows and ends as it does on a GPU.  The tests script what only happens by
// chance there: a report that is half published when the host looks, a failed
// launch, a failed allocation, a write into memory already given back.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <thread>

#include "tc_pipes_cpu.cpp"

#include "srd_devloop.h"
#include "srd_runtime.h"

namespace {

struct Device {
  std::mutex mu;
  std::condition_variable cv;
  std::deque<std::function<void()>> q;
  bool busy = false, stop = false, paused = false;
  std::thread th;
  Device() : th([this] { loop(); }) {}
  ~Device() {
    {
      std::lock_guard<std::mutex> g(mu);
      stop = true;
      paused = false;
    }
    cv.notify_all();
    th.join();
  }
  void loop() {
    std::unique_lock<std::mutex> g(mu);
    for (;;) {
      cv.wait(g, [this] { return stop || (!q.empty() && !paused); });
      if (q.empty()) return;
      std::function<void()> f = std::move(q.front());
      q.pop_front();
      busy = true;
      g.unlock();
      f();
      g.lock();
      busy = false;
      cv.notify_all();
    }
  }
  void put(std::function<void()> f) {
    std::lock_guard<std::mutex> g(mu);
    q.push_back(std::move(f));
    cv.notify_all();
  }
  bool idle() { return q.empty() && !busy; }  // under mu
};
Device* g_dev = nullptr;  // one per test run (sim_reset), so that a run's rest cannot reach the next

// ---- what a test scripts (sim_reset clears it)
std::atomic<uint64_t> g_split_tick{0};   // book that is half published when the host looks (0: none)
std::atomic<bool> g_half{false};         // it stored its overflow flag, its tick not yet
std::atomic<bool> g_drained{false};      // the host has waited for the stream since
std::atomic<bool> g_hold{false};         // iterations wait for the host to wait for them
std::atomic<bool> g_tail{false};         // and has enqueued launches since
std::atomic<uint64_t> g_plans{0}, g_books{0}, g_fail_book{0}, g_queries{0};
std::atomic<uint64_t> g_limit{0}, g_used{0}, g_late_writes{0};
// the nth allocation fails (0: none) of those once iterations run, or of those of g_fail_bytes
std::atomic<uint64_t> g_fail_alloc{0}, g_fail_bytes{0};
std::atomic<bool> g_running{false};      // a run has enqueued its first iteration
std::atomic<int> g_upload_fails{0};
std::mutex g_pin_mu;
std::map<const char*, uint64_t> g_pins;   // pinned blocks handed out

void wait_for(const std::function<bool()>& f) {
  for (int i = 0; i < 4000 && !f(); ++i) std::this_thread::sleep_for(std::chrono::milliseconds(1));
}

bool pinned_alive(const void* p) {
  std::lock_guard<std::mutex> g(g_pin_mu);
  auto it = g_pins.upper_bound(static_cast<const char*>(p));
  return it != g_pins.begin() && std::prev(it)->first + std::prev(it)->second > p;
}

void enqueue(std::function<void()> f) { g_dev->put(std::move(f)); }

}  // namespace

extern "C" int sim_stream_op(int op) {
  if (!g_dev) return 1;
  std::unique_lock<std::mutex> g(g_dev->mu);
  if (op == 1) {
    if (g_dev->paused && ++g_queries >= 3) {
      g_dev->paused = false;
      g_dev->cv.notify_all();
    }
    return g_dev->idle();
  }
  g_drained = true;
  const bool hold = g_dev->paused && !g_tail;  // until launches follow the host's answer
  g_dev->paused = false;
  g_dev->cv.notify_all();
  g_dev->cv.wait(g, [] { return g_dev->idle(); });
  g_dev->paused = g_dev->paused || hold;
  return 1;
}

extern "C" void sim_reset() {
  delete g_dev;
  g_dev = new Device();
  g_split_tick = g_plans = g_books = g_fail_book = g_queries = g_limit = g_late_writes = 0;
  g_half = g_drained = g_tail = g_running = g_hold = false;
  g_fail_alloc = g_fail_bytes = 0;
  g_upload_fails = 0;
}
extern "C" int sim_upload_fails() { return g_upload_fails; }
extern "C" void sim_set_upload_fails(int on) { g_upload_fails = on; }
extern "C" void sim_split_report(uint64_t tick) { g_split_tick = tick; }
// The device starts on what is enqueued only when the host waits for it (or
// asks three times).
extern "C" void sim_hold() {
  std::lock_guard<std::mutex> g(g_dev->mu);
  g_hold = true;
}
extern "C" void sim_fail_book(uint64_t nth) { g_books = 0, g_fail_book = nth; }
extern "C" void sim_fail_alloc(uint64_t nth, uint64_t bytes) { g_fail_alloc = nth, g_fail_bytes = bytes; }
extern "C" uint64_t sim_allocs_to_failure() { return g_fail_alloc; }
extern "C" void sim_pool_limit(uint64_t bytes) { g_limit = bytes; }
extern "C" uint64_t sim_pool_used() { return g_used; }
extern "C" uint64_t sim_late_writes() { return g_late_writes; }
// Size of a buffer whose growth failed.
extern "C" uint64_t sim_size_after_failure() {
  srd::DevBuf<uint32_t> b(64, nullptr);
  g_limit = g_used + 1024;
  try {
    b.reserve(1 << 20, nullptr);
  } catch (const std::exception&) {
  }
  g_limit = 0;
  return b.p ? ~uint64_t(0) : b.n;
}
extern "C" uint64_t sim_dense_iterations() { return g_plans; }

namespace srd {

void* pool_alloc(uint64_t bytes, hipStream_t) {
  const bool chosen = (g_fail_bytes ? bytes == g_fail_bytes : g_running.load()) && g_fail_alloc && --g_fail_alloc == 0;
  if (chosen || (g_limit && g_used + bytes > g_limit))
    fail("simulated pool: no memory for " + std::to_string(bytes) + " bytes");
  g_used += bytes;
  return std::calloc(1, bytes ? bytes : 1);
}
void pool_free(void* p, uint64_t bytes, hipStream_t) {
  if (!p) return;
  g_used -= bytes;
  if (g_dev) enqueue([p] { std::free(p); });  // stream order
  else std::free(p);
}
void* pinned_acquire(uint64_t bytes, uint64_t* got) {
  *got = bytes;
  char* p = static_cast<char*>(std::calloc(1, bytes ? bytes : 1));
  std::lock_guard<std::mutex> g(g_pin_mu);
  g_pins[p] = bytes;
  return p;
}
void pinned_release(void* p, uint64_t) {
  std::lock_guard<std::mutex> g(g_pin_mu);
  g_pins.erase(static_cast<char*>(p));  // kept allocated: a late write is counted, not a crash
}

static uint64_t words_of(const DenseRel& r) { return uint64_t(r.nblocks) * (kDenseBlockWords / 2); }

// Rows and roots in key order of the bits of NEW (& ~FULL) in the blocks `on`.
static uint64_t each_row(const DenseRel& r, const uint8_t* on, const std::function<void(uint64_t, bool)>& f) {
  uint64_t n = 0, last = ~uint64_t(0);
  const uint32_t rs = r.shift * (r.k - 1);
  for (uint64_t w = 0; w < words_of(r); ++w) {
    if (!on[w >> 12]) continue;
    for (uint64_t x = r.nw[w] & ~(r.fl ? r.fl[w] : 0); x; x &= x - 1) {
      const uint64_t key = (w << 6) | uint64_t(__builtin_ctzll(x));
      f(key, (key >> rs) != last);
      last = key >> rs;
      ++n;
    }
  }
  return n;
}
static void count(const DenseRel& r, const uint8_t* on) {  // one total, in block 0
  uint64_t roots = 0;
  const uint64_t n = each_row(r, on, [&](uint64_t, bool first) { roots += first && r.k > 1; });
  std::fill(r.blk, r.blk + r.nblocks, uint64_t(0));
  r.blk[0] = n | roots << kDenseRowBits;
}
static void emit(const DenseRel& r, const uint8_t* on) {
  uint64_t n = 0, g = 0;
  const uint64_t mask = (uint64_t(1) << r.shift) - 1;
  each_row(r, on, [&](uint64_t key, bool first) {
    for (uint32_t c = 0; c < r.k; ++c)
      r.delta[uint64_t(c) * r.stride + n] = uint32_t((key >> (r.shift * (r.k - 1 - c))) & mask);
    if (first) r.root_v[g] = uint32_t(key >> (r.shift * (r.k - 1))), r.root_o[g] = uint32_t(n), ++g;
    ++n;
  });
}

void dense_set_rows(const uint32_t* cols, uint64_t stride, uint64_t n, uint32_t k, uint32_t shift,
                    uint64_t* bits, uint8_t* sum, hipStream_t) {
  enqueue([=] {
    for (uint64_t i = 0; i < n; ++i) {
      uint64_t key = 0;
      for (uint32_t c = 0; c < k; ++c) key = (key << shift) | cols[uint64_t(c) * stride + i];
      bits[key >> 6] |= uint64_t(1) << (key & 63);
      sum[key >> 18] = 1;
    }
  });
}

void dense_plan(DenseCtl*, SrdDyn* d, uint32_t, const uint64_t* key_work, uint64_t* work_start, uint64_t,
                uint64_t*, uint32_t*, uint32_t grain, uint32_t least, hipStream_t) {
  ++g_plans;
  g_running = true;
  if (g_hold.exchange(false)) {
    std::lock_guard<std::mutex> g(g_dev->mu);
    g_dev->paused = true;
    g_queries = 0;
  }
  // the third iteration is enqueued late: the device is already in the second
  if (g_split_tick && g_plans == g_split_tick + 1) wait_for([] { return g_half.load(); });
  enqueue([=] {
    if (d->skip) return;
    uint64_t t = 0;
    for (uint64_t i = 0; i < d->n_root; ++i) work_start[i] = t, t += key_work[i];
    work_start[d->n_root] = t;
    d->total_work = t;
    d->grain = least ? srd_grain(t, grain, least) : grain;
    d->n_slices = (t + d->grain - 1) / d->grain;
  });
}

void dense_count(const DenseCtl* c, const DenseRel& r, hipStream_t) {
  if (g_drained) g_tail = true;
  enqueue([=] {
    if (c->skip) return;
    std::copy(r.nsum, r.nsum + r.nblocks, r.live);
    count(r, r.live);
  });
}

static void book(const DenseBook& B) {
  DenseCtl* c = B.ctl;
  if (c->skip) {
    c->emit = 0;
    return;
  }
  uint64_t need = 0, sum = 0, n[kDevRels];
  for (uint32_t r = 0; r < B.nrels; ++r) {
    n[r] = B.rel[r].blk[0] & kDenseRowMask;
    if (n[r] > B.rel[r].stride) need = std::max(need, n[r]);
    sum += n[r];
  }
  uint32_t ovf = need ? uint32_t(kOvfNew) : 0u;
  if (c->iter >= c->iter_cap) ovf |= uint32_t(kOvfIters);
  if (ovf) {
    c->overflow = ovf;
    c->skip = 1;
    c->emit = 0;
    for (uint32_t p = 0; p < B.npipes; ++p) B.pipe[p].dyn->skip = 1;
  } else {
    for (uint32_t r = 0; r < B.nrels; ++r) {
      const uint64_t g = B.rel[r].k > 1 ? B.rel[r].blk[0] >> kDenseRowBits : n[r];
      std::fill(B.rel[r].nsum, B.rel[r].nsum + B.rel[r].nblocks, uint8_t(0));
      B.rel[r].rec[c->iter] = n[r];
      c->delta_n[r] = n[r];
      c->delta_r[r] = g;
      c->full_n[r] += n[r];
      if (n[r]) B.rel[r].root_o[g] = uint32_t(n[r]);
    }
    c->iter += 1;
    c->done = sum == 0;
    c->emit = 1;
    c->skip = c->done || c->iter >= c->max_iter;
    for (uint32_t p = 0; p < B.npipes; ++p) {
      SrdDyn* d = B.pipe[p].dyn;
      const DlBind& bd = B.pipe[p].bind;
      for (uint32_t v = 0; v < bd.n_views; ++v) {
        const int r = bd.vrel[v];
        if (r < 0) continue;
        IndexView& iv = d->views.v[v];
        iv.cols = B.rel[r].delta;
        iv.root_vals = B.rel[r].root_v;
        iv.root_offs = B.rel[r].root_o;
        iv.stride = B.rel[r].stride;
        iv.n = uint32_t(c->delta_n[r]);
        iv.r = uint32_t(c->delta_r[r]);
      }
      uint32_t drv = bd.root_view[0];
      for (uint32_t i = 0; i < bd.n_root_src; ++i)
        if (d->views.v[bd.root_view[i]].r < d->views.v[drv].r) drv = bd.root_view[i];
      d->skip = c->skip;
      d->drv_view = drv;
      d->n_root = d->views.v[drv].r;
    }
  }
  c->tick += 1;
  volatile DenseSeen* h = B.seen;
  if (!pinned_alive(B.seen)) ++g_late_writes;
  h->iter = c->iter;
  h->need = need;
  h->done = c->done;
  h->overflow = ovf;
  if (ovf && c->tick == g_split_tick) {
    // the host looks now, and the launches after its answer wait for it to look again
    g_half = true;
    g_drained = g_tail = false;
    wait_for([] { return g_drained.load(); });
    std::lock_guard<std::mutex> g(g_dev->mu);
    g_dev->paused = true;
    g_queries = 0;
    __atomic_store_n(const_cast<uint64_t*>(&h->tick), c->tick, __ATOMIC_RELEASE);
    // the wait for the stream in progress ends with this launch's successors
    // that were enqueued before it
    while (!g_dev->q.empty()) {
      auto f = std::move(g_dev->q.front());
      g_dev->q.pop_front();
      f();
    }
    return;
  }
  __atomic_store_n(const_cast<uint64_t*>(&h->tick), c->tick, __ATOMIC_RELEASE);
}

void dense_book(const DenseBook& B, hipStream_t) {
  if (++g_books == g_fail_book) fail("simulated launch failure");
  enqueue([B] { book(B); });
}

void dense_emit(const DenseCtl* c, const DenseRel& r, hipStream_t) {
  enqueue([=] {
    if (!c->emit) return;
    emit(r, r.live);
    for (uint64_t w = 0; w < words_of(r); ++w) r.fl[w] |= r.nw[w], r.nw[w] = 0;
    for (uint32_t b = 0; b < r.nblocks; ++b) r.fsum[b] |= r.live[b];
  });
}

void dense_inst(const DenseCtl* c, uint32_t rel, const uint32_t* col0, const uint32_t* bounds,
                uint32_t n_inst, uint64_t* out, hipStream_t s) {
  enqueue([=] {
    if (c->emit) instance_counts(col0, c->delta_n[rel], bounds, n_inst, out + (c->iter - 1) * n_inst, s);
  });
}

void dense_index_count(const DenseRel& r, hipStream_t) {
  enqueue([=] {
    count(r, r.nsum);
    r.blk[r.nblocks] = r.blk[0];
  });
}
void dense_index_emit(const DenseRel& r, hipStream_t) {
  enqueue([=] { emit(r, r.nsum); });
}

}  // namespace srd

namespace {

void rec_mark(const SrdLaunchArgs* a, hipStream_t) {
  uint64_t rows = 0;
  for (uint64_t it = 0; it < a->total_work; ++it, ++rows) {
    const uint32_t k = uint32_t(std::upper_bound(a->work_start, a->work_start + a->n_root + 1, it) -
                                a->work_start) - 1;
    const uint64_t li = it - a->work_start[k];
    const uint32_t b1 = a->key_rng[k * 4 + 2], d1 = a->key_rng[k * 4 + 3] - b1;
    const uint64_t x = colp(a->views.v[0], 1)[a->key_rng[k * 4] + li / d1];
    const uint64_t z = colp(a->views.v[1], 1)[b1 + li % d1];
    const uint64_t key = z << a->mark_shift | x;
    a->mark_bits[key >> 5] |= 1u << (key & 31);
    a->mark_sum[key >> 18] = 1;
  }
  if (a->mark_rows) *a->mark_rows += rows;
}

template <SrdLaunchFn F>
void queued(const SrdLaunchArgs* a, hipStream_t s) {
  if (!a->mark_bits) return dyn_launch<F>(a, s);  // iterations of rows: run at once
  const SrdLaunchArgs b = *a;
  enqueue([b, s] { dyn_launch<F>(&b, s); });
}

// TCRec_D0's device-sized launches in the bitmap loop are queued; the other
// two rules run outside it.  On the host loop it marks too.
SrdPipelineDesc* dense_pipes() {
  static SrdPipelineDesc p[3] = {k_pipes[0], k_pipes[1], k_pipes[2]};
  p[2].root_dyn = &queued<&rec_root>;
  p[2].mark = &rec_mark;
  return p;
}

const SrdPipelineExt k_exts[] = {
  {"EdgeLoad", 0, nullptr, nullptr, 0, 0, 0, -1, 0},
  {"TCBase", 0, nullptr, nullptr, 0, 0, 0, -1, 0},
  {"TCRec_D0", 0, &queued<&rec_mark>, nullptr, 0, 0, 0, -1, 0},
};

}  // namespace

// The recursive rule as one with a union pipeline.  That one is not simulated
// (union_products fails); the rule itself marks.
extern "C" srd_engine* cpu_union_engine(const char* program_text) {
  static const SrdPipelineExt exts[] = {k_exts[0], k_exts[1],
                                        {"TCRec_D0", 2, nullptr, &dense_pipes()[2], 1, 0, 0, -1, 0}};
  return srd_engine_create_ext(program_text, dense_pipes(), 3, exts, 3);
}

extern "C" srd_engine* cpu_dense_engine(const char* program_text) {
  return srd_engine_create_ext(program_text, dense_pipes(), 3, k_exts, 3);
}
