// Context, device memory, kernel timing and the Wigner tables.
#include "psx_internal.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <exception>
#include <thread>
#include <vector>

namespace psx {

void* ctx_alloc(Ctx* c, size_t bytes) {
  if (bytes == 0) bytes = 8;
  // the idle cached buffers are caches: give them back before failing
  for (CachedSlot* sl : {&c->xfer, &c->work}) {
    if (c->in_use + bytes <= c->budget) break;
    if (sl->p && !sl->busy) {
      PSX_HIP(hipStreamSynchronize(c->stream));
      void* p = sl->p;
      sl->p = nullptr;
      sl->bytes = 0;
      ctx_free(c, p);
    }
  }
  PSX_REQUIRE(c->in_use + bytes <= c->budget, PSX_ERR_BUDGET,
              "allocation of " + std::to_string(bytes) +
                  " bytes exceeds the context HBM budget");
  void* p = nullptr;
  PSX_HIP(hipMalloc(&p, bytes));
  c->allocations[p] = bytes;
  c->in_use += bytes;
  return p;
}

void ctx_free(Ctx* c, void* p) {
  if (!p) return;
  auto it = c->allocations.find(p);
  PSX_REQUIRE(it != c->allocations.end(), PSX_ERR_ARGUMENT,
              "pointer not owned by this context");
  c->in_use -= it->second;
  c->allocations.erase(it);
  PSX_HIP(hipFree(p));
}

void* ctx_scratch(Ctx* c, size_t bytes) {
  if (bytes <= c->scratch_bytes) return c->scratch;
  if (c->scratch) {
    PSX_HIP(hipStreamSynchronize(c->stream));
    ctx_free(c, c->scratch);
    c->scratch = nullptr;
    c->scratch_bytes = 0;
  }
  size_t want = bytes + bytes / 4;
  c->scratch = ctx_alloc(c, want);
  c->scratch_bytes = want;
  return c->scratch;
}

HeldBuf::HeldBuf(Ctx* cc, CachedSlot& s, size_t bytes) : c(cc), slot(&s) {
  PSX_REQUIRE(!s.busy, PSX_ERR_ARGUMENT, "cached device buffer already in use");
  if (bytes > s.bytes) {
    if (s.p) {
      PSX_HIP(hipStreamSynchronize(c->stream));
      void* p = s.p;
      s.p = nullptr;
      s.bytes = 0;
      ctx_free(c, p);
    }
    s.p = ctx_alloc(c, bytes);
    s.bytes = bytes;
  }
  s.busy = true;
  cap = bytes;
}

HeldBuf::~HeldBuf() {
  // after an error nothing may still be queued on the buffer, the next call's, or
  // on host memory that the failed call was given
  if (std::uncaught_exceptions() > errors) {
    (void)hipStreamSynchronize(c->stream);
    if (c->xstream) (void)hipStreamSynchronize(c->xstream);
  }
  slot->busy = false;
}

double* HeldBuf::take(size_t bytes) {
  const size_t at = (used + 255) & ~size_t(255);
  PSX_REQUIRE(at + bytes <= cap, PSX_ERR_ARGUMENT, "cached buffer carve overflow");
  used = at + bytes;
  return reinterpret_cast<double*>(static_cast<char*>(slot->p) + at);
}

TimedLaunch::TimedLaunch(Ctx* ctx, const char* kname) : c(ctx), name(kname) {
  if (c->timing) {
    PSX_HIP(hipEventCreate(&e0));
    PSX_HIP(hipEventCreate(&e1));
    PSX_HIP(hipEventRecord(e0, c->stream));
  }
}

TimedLaunch::~TimedLaunch() noexcept(false) {
  hipError_t le = hipGetLastError();
  if (e0) {
    (void)hipEventRecord(e1, c->stream);
    c->timers[name].pending.emplace_back(e0, e1);
  }
  // while another error unwinds the stack (a failed call inside the timed
  // scope), that error is the one reported: a second throw would terminate
  if (le != hipSuccess && std::uncaught_exceptions() == 0)
    throw Error{PSX_ERR_DEVICE, std::string("launch of ") + name + ": " +
                                    hipGetErrorString(le)};
}

// Wait for the recorded launches and fold their durations into the totals.
void resolve_timers(Ctx* c) {
  for (auto& kv : c->timers) {
    for (auto& ev : kv.second.pending) {
      PSX_HIP(hipEventSynchronize(ev.second));
      float ms = 0;
      PSX_HIP(hipEventElapsedTime(&ms, ev.first, ev.second));
      kv.second.total_ms += ms;
      kv.second.launches += 1;
      (void)hipEventDestroy(ev.first);
      (void)hipEventDestroy(ev.second);
    }
    kv.second.pending.clear();
  }
}

// gamma_m = prod_{k<=m} (2k-1)/(2k) accumulated in long double (64-bit
// mantissa); the rounding to double of each entry is then the dominant error.
int table_entries(int nmax_index) { return (nmax_index + 2 * kTabOff + 1023) & ~1023; }

void build_tables_host(int n, double* G, double* Z, double* D, double* IG) {
  for (int i = 0; i < n; ++i) G[i] = Z[i] = D[i] = IG[i] = 0.0;
  long double g = 1.0L;
  for (int m = 0; m + kTabOff < n; ++m) {
    if (m > 0) g = g * (long double)(2 * m - 1) / (long double)(2 * m);
    int i = m + kTabOff;
    G[i] = (double)g;
    Z[i] = (double)((long double)(2 * m + 1) * g);
    D[i] = (double)(1.0L / ((long double)(2 * m + 1) * g));
    IG[i] = (double)(1.0L / g);
  }
}

void ensure_tables(Ctx* c, int nmax_index) {
  Tables& t = c->tables;
  if (t.n >= nmax_index + 2 * kTabOff) return;
  const int n = table_entries(nmax_index);
  std::vector<double> G(n), Z(n), D(n), IG(n);
  build_tables_host(n, G.data(), Z.data(), D.data(), IG.data());
  // other streams (a server's slots) may read the old tables
  PSX_HIP(hipDeviceSynchronize());
  if (t.dG) {
    ctx_free(c, t.dG);
    ctx_free(c, t.dZ);
    ctx_free(c, t.dD);
    ctx_free(c, t.dIG);
  }
  size_t b = sizeof(double) * n;
  t.dG = (double*)ctx_alloc(c, b);
  t.dZ = (double*)ctx_alloc(c, b);
  t.dD = (double*)ctx_alloc(c, b);
  t.dIG = (double*)ctx_alloc(c, b);
  PSX_HIP(hipMemcpy(t.dG, G.data(), b, hipMemcpyHostToDevice));
  PSX_HIP(hipMemcpy(t.dZ, Z.data(), b, hipMemcpyHostToDevice));
  PSX_HIP(hipMemcpy(t.dD, D.data(), b, hipMemcpyHostToDevice));
  PSX_HIP(hipMemcpy(t.dIG, IG.data(), b, hipMemcpyHostToDevice));
  t.n = n;
}

}  // namespace psx

using namespace psx;

extern "C" {

int psx_ctx_create(int device, size_t hbm_budget, psx_ctx** out) {
  if (!out) return PSX_ERR_ARGUMENT;
  *out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return PSX_ERR_DEVICE;
  if (device < 0 || device >= ndev) return PSX_ERR_ARGUMENT;
  if (hipSetDevice(device) != hipSuccess) return PSX_ERR_DEVICE;
  Ctx* c = new Ctx();
  c->device = device;
  size_t freeb = 0, total = 0;
  if (hipMemGetInfo(&freeb, &total) != hipSuccess) {
    delete c;
    return PSX_ERR_DEVICE;
  }
  c->budget = hbm_budget ? hbm_budget : (size_t)(0.9 * (double)freeb);
  if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
    delete c;
    return PSX_ERR_DEVICE;
  }
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, device) == hipSuccess)
    c->cu_count = prop.multiProcessorCount;
  try {
    noalloc_init_device(device);
  } catch (const Error&) {
    (void)hipStreamDestroy(c->stream);
    delete c;
    return PSX_ERR_DEVICE;
  }
  *out = reinterpret_cast<psx_ctx*>(c);
  return PSX_OK;
}

int psx_ctx_destroy(psx_ctx* h) {
  Ctx* c = reinterpret_cast<Ctx*>(h);
  if (!c) return PSX_ERR_ARGUMENT;
  {
    std::lock_guard<std::recursive_mutex> lk(c->mu);
    if (c->live_servers > 0) {
      c->last_error = "context still has " + std::to_string(c->live_servers) +
                      " live server(s): destroy them first (psx_server_destroy)";
      return PSX_ERR_ARGUMENT;
    }
    (void)hipSetDevice(c->device);
    (void)hipStreamSynchronize(c->stream);
    try {
      resolve_timers(c);
    } catch (...) {
    }
    // library handles first, while their stream and the memory they may
    // still reference exist; then the plans, the memory and the streams
    release_blas(c);
    release_tile_cache(c);
    release_mix_tiles(c);
    release_sht_plans(c);
    for (auto& kv : c->allocations) (void)hipFree(kv.first);
    c->allocations.clear();
    release_stage(c);
    (void)hipStreamDestroy(c->stream);
  }
  delete c;
  return PSX_OK;
}

int psx_ctx_synchronize(psx_ctx* h) {
  Ctx* c = reinterpret_cast<Ctx*>(h);
  return guarded(c, [&] {
    PSX_HIP(hipSetDevice(c->device));
    PSX_HIP(hipStreamSynchronize(c->stream));
  });
}

const char* psx_ctx_last_error(psx_ctx* h) {
  Ctx* c = reinterpret_cast<Ctx*>(h);
  if (!c) return "null context";
  return c->last_error.c_str();
}

size_t psx_ctx_bytes_in_use(psx_ctx* h) {
  Ctx* c = reinterpret_cast<Ctx*>(h);
  return c ? c->in_use : 0;
}

int psx_ctx_set_timing(psx_ctx* h, int enable) {
  Ctx* c = reinterpret_cast<Ctx*>(h);
  return guarded(c, [&] { c->timing = enable != 0; });
}

int psx_ctx_kernel_time(psx_ctx* h, const char* name, int reset,
                        double* total_ms, int64_t* launches) {
  Ctx* c = reinterpret_cast<Ctx*>(h);
  return guarded(c, [&] {
    PSX_REQUIRE(name != nullptr, PSX_ERR_ARGUMENT, "null kernel name");
    resolve_timers(c);
    auto it = c->timers.find(name);
    double ms = 0;
    int64_t n = 0;
    if (it != c->timers.end()) {
      ms = it->second.total_ms;
      n = it->second.launches;
      if (reset) c->timers.erase(it);
    }
    if (total_ms) *total_ms = ms;
    if (launches) *launches = n;
  });
}

int psx_dev_alloc(psx_ctx* h, size_t bytes, void** dptr) {
  Ctx* c = reinterpret_cast<Ctx*>(h);
  return guarded(c, [&] {
    PSX_REQUIRE(dptr != nullptr, PSX_ERR_ARGUMENT, "null output pointer");
    PSX_HIP(hipSetDevice(c->device));
    *dptr = ctx_alloc(c, bytes);
  });
}

int psx_dev_free(psx_ctx* h, void* dptr) {
  Ctx* c = reinterpret_cast<Ctx*>(h);
  return guarded(c, [&] {
    PSX_HIP(hipSetDevice(c->device));
    PSX_HIP(hipStreamSynchronize(c->stream));
    ctx_free(c, dptr);
  });
}

int psx_memcpy_h2d(psx_ctx* h, void* dst, const void* src, size_t bytes) {
  Ctx* c = reinterpret_cast<Ctx*>(h);
  return guarded(c, [&] {
    PSX_HIP(hipSetDevice(c->device));
    PSX_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, c->stream));
    PSX_HIP(hipStreamSynchronize(c->stream));
  });
}

int psx_memcpy_d2h(psx_ctx* h, void* dst, const void* src, size_t bytes) {
  Ctx* c = reinterpret_cast<Ctx*>(h);
  return guarded(c, [&] {
    PSX_HIP(hipSetDevice(c->device));
    PSX_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, c->stream));
    PSX_HIP(hipStreamSynchronize(c->stream));
  });
}

}  // extern "C"

// ---- staged host copies ---------------------------------------------------
// Copies between device memory and pageable host memory run far below PCIe
// speed (a 2-D one goes row by row: 660 us for a 96 x 96 block), so all but short
// ranges go through a ring of pinned slots: the DMA runs ahead in some while host threads
// copy others, a chunk split between several threads, which also fault in a
// fresh destination's pages.  Chunks are an eighth of the transfer, at most a
// slot (12 MB, 220 us at 57 GB/s: 2 MB chunks lost 20 % of that rate between
// DMAs on 400 MB, 8 MB ones 3 % where a transfer comes in 25 pieces) and at least
// kChunkBytes, so that short ones overlap too.
namespace psx {

namespace {
constexpr int kCopyThreads = 11;                    // and the calling thread
constexpr size_t kChunkBytes = size_t(1) << 20;
constexpr int kParts = 8;                           // chunks of a transfer, where they fit
constexpr size_t kTaskBytes = size_t(768) << 10;    // of a chunk, per task
constexpr size_t kInlineBytes = size_t(256) << 10;  // copied by the caller itself
// One range up to kDirectBytes goes to the runtime as it is, out of the device from
// kDirectOutBytes on: a slot, its event and the pinned copy take 10 us more in (the
// alms of alm2map and alm2cl, 160 bytes to 730 KB: 58 -> 40, 111 -> 86, 152 -> 118 and
// 211 -> 160 us a call) and a pool thread's wake-up and copy up to 40 out (maps of 98
// and 393 KB: 77 -> 62, 133 -> 93 us).  Smaller results measure alike or better from a
// slot; above 1 MB the slots' copies overlap their DMAs.
constexpr size_t kDirectBytes = size_t(1) << 20;
constexpr size_t kDirectOutBytes = size_t(64) << 10;
}  // namespace

CopyPool::CopyPool(int threads) {
  try {
    for (int i = 0; i < threads; ++i) threads_.emplace_back([this] { work(); });
  } catch (const std::exception&) {
    // (as many as the process or its memory allow; with none, submit runs the tasks)
  }
}

CopyPool::~CopyPool() {
  {
    std::lock_guard<std::mutex> lk(mu_);
    stop_ = true;
  }
  cv_.notify_all();
  for (auto& t : threads_) t.join();
}

void CopyPool::submit(const std::function<void()>& task) {
  if (threads_.empty()) return task();
  {
    std::lock_guard<std::mutex> lk(mu_);
    tasks_.push_back(task);
  }
  cv_.notify_one();
}

void CopyPool::work() {
  for (;;) {
    std::function<void()> t;
    {
      std::unique_lock<std::mutex> lk(mu_);
      cv_.wait(lk, [&] { return stop_ || !tasks_.empty(); });
      if (tasks_.empty()) return;   // stopping
      t = std::move(tasks_.front());
      tasks_.pop_front();
    }
    t();
  }
}

void Stage::grow(int n) {
  n = std::min(n, kSlots);
  while (have < n) {
    Slot& sl = slot[have];
    if (!sl.ev) PSX_HIP(hipEventCreateWithFlags(&sl.ev, hipEventDisableTiming));
    void* p = nullptr;
    PSX_HIP(hipHostMalloc(&p, kSlotBytes, hipHostMallocDefault));
    sl.p = (char*)p;
    ++have;
  }
}

void Stage::release() {
  for (Slot& sl : slot) {
    if (sl.ev) (void)hipEventDestroy(sl.ev);
    if (sl.p) (void)hipHostFree(sl.p);
    sl.ev = nullptr;
    sl.p = nullptr;
  }
  have = next = 0;
}

void ensure_stage(Ctx* c) {
  if (c->xstream) return;
  if (!c->pool) {
    const int hw = (int)std::max(2u, std::thread::hardware_concurrency());
    c->pool = std::make_unique<CopyPool>(std::min(kCopyThreads, hw - 1));
  }
  if (!c->flag) PSX_HIP(hipHostMalloc((void**)&c->flag, kFlags * sizeof(int), hipHostMallocDefault));
  PSX_HIP(hipStreamCreateWithFlags(&c->xstream, hipStreamNonBlocking));
}

void release_stage(Ctx* c) {
  if (c->xstream) (void)hipStreamSynchronize(c->xstream);
  c->pool.reset();
  c->stage.release();
  if (c->flag) (void)hipHostFree(c->flag);
  c->flag = nullptr;
  if (c->xstream) (void)hipStreamDestroy(c->xstream);
  c->xstream = nullptr;
  for (hipEvent_t& e : c->band_ev) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
}

void ensure_band_events(Ctx* c) {
  for (hipEvent_t& e : c->band_ev)
    if (!e) PSX_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
}

namespace {
// one piece of a staged copy: nc columns of `rows` doubles, at most a slot
struct Chunk {
  double* host;
  int64_t ldh;
  double* dev;
  int64_t ldd;
  int64_t rows, nc;
  hipEvent_t after;
  size_t bytes() const { return sizeof(double) * (size_t)rows * (size_t)nc; }
};

// Cut a matrix into chunks of at most `most` doubles; packed ranges and columns
// longer than that are cut along the rows.
void cut(std::vector<Chunk>& ch, int64_t most, double* host, int64_t ldh, double* dev,
         int64_t ldd, int64_t rows, int64_t cols, hipEvent_t after) {
  if (rows <= 0 || cols <= 0) return;
  if (cols > 1 && ldh == rows && ldd == rows) {
    rows *= cols;
    cols = 1;
  }
  if (cols == 1 || rows > most) {
    for (int64_t j = 0; j < cols; ++j)
      for (int64_t i = 0; i < rows; i += most) {
        const int64_t m = std::min(most, rows - i);
        ch.push_back({host + j * ldh + i, m, dev + j * ldd + i, m, m, 1, after});
      }
    return;
  }
  const int64_t cpc = most / rows;
  for (int64_t j = 0; j < cols; j += cpc)
    ch.push_back({host + j * ldh, ldh, dev + j * ldd, ldd, rows, std::min(cpc, cols - j), after});
}

// doubles a chunk holds in a transfer of `total` in about `parts` chunks
int64_t chunk_doubles(int64_t total, int parts = kParts) {
  const int64_t lo = kChunkBytes / sizeof(double), hi = Stage::kSlotBytes / sizeof(double);
  return std::min(hi, std::max(lo, (total / parts + 511) & ~int64_t(511)));
}

void copy_cols(double* dst, int64_t ldd, const double* src, int64_t lds, int64_t rows,
               int64_t cols) {
  if (ldd == rows && lds == rows) {
    std::memcpy(dst, src, sizeof(double) * rows * cols);
    return;
  }
  for (int64_t j = 0; j < cols; ++j)
    std::memcpy(dst + j * ldd, src + j * lds, sizeof(double) * rows);
}

// (the waiting thread takes no task itself: it has the next DMA to issue)
void wait_copied(const Stage::Slot& sl) {
  while (sl.copying.load(std::memory_order_acquire)) std::this_thread::yield();
}

// waits for every host copy of the stage, also when an error unwinds: they use
// the caller's memory.  An error leaves nothing in flight on the stream either,
// since the device side may be the next call's.
struct CopiesDone {
  Stage& st;
  hipStream_t s;
  const int errors = std::uncaught_exceptions();
  ~CopiesDone() {
    for (int i = 0; i < st.have; ++i) wait_copied(st.slot[i]);
    if (std::uncaught_exceptions() > errors) (void)hipStreamSynchronize(s);
  }
};

// Copy chunk x between its host range and slot sl (to the host, or from it),
// split between pool tasks, or by the caller when the whole transfer is small.
void start_copy(Stage::Slot& sl, CopyPool& pool, bool inlined, const Chunk& x, bool to_host) {
  auto part = [&sl, to_host](const Chunk& y, int64_t at) {
    double* p = (double*)sl.p + at;
    if (to_host) copy_cols(y.host, y.ldh, p, y.rows, y.rows, y.nc);
    else copy_cols(p, y.rows, y.host, y.ldh, y.rows, y.nc);
  };
  if (inlined) {
    part(x, 0);
    return;
  }
  const bool by_rows = x.nc == 1;
  const int64_t len = by_rows ? x.rows : x.nc;
  const int64_t n = std::max<int64_t>(1, std::min<int64_t>(len, x.bytes() / kTaskBytes));
  sl.copying.store((int)n, std::memory_order_relaxed);
  for (int64_t i = 0; i < n; ++i) {
    const int64_t a = len * i / n, b = len * (i + 1) / n;
    Chunk y = x;
    if (by_rows) {
      y.host += a;
      y.rows = y.ldh = b - a;
    } else {
      y.host += a * x.ldh;
      y.nc = b - a;
    }
    const int64_t at = by_rows ? a : a * x.rows;
    auto task = [&sl, part, y, at] {
      part(y, at);
      sl.copying.fetch_sub(1, std::memory_order_release);
    };
    try {
      pool.submit(task);
    } catch (const std::bad_alloc&) {   // (not queued: the count has to come down)
      task();
    }
  }
}

bool small(const std::vector<Chunk>& ch) {
  return ch.size() == 1 && ch[0].bytes() <= kInlineBytes;
}

void d2h_chunks(hipStream_t s, Stage& st, CopyPool& pool, const std::vector<Chunk>& ch,
                const std::function<void()>* landed) {
  const size_t n = ch.size();
  if (n == 0) return;
  st.grow((int)std::min<size_t>(n, Stage::kSlots));
  CopiesDone done{st, s};
  const int ring = st.have, base = st.next;
  const bool inlined = small(ch);
  auto at = [&](size_t k) -> Stage::Slot& { return st.slot[(base + k) % ring]; };
  size_t i = 0;
  for (size_t k = 0; k < n; ++k) {
    // DMAs into every slot whose last host copy is over
    for (; i < n && i < k + ring; ++i) {
      Stage::Slot& sl = at(i);
      if (i > k && sl.copying.load(std::memory_order_acquire)) break;
      wait_copied(sl);
      const Chunk& x = ch[i];
      if (x.after) PSX_HIP(hipStreamWaitEvent(s, x.after, 0));
      const size_t colb = sizeof(double) * (size_t)x.rows;
      // (an upload still reading the slot, perhaps on another stream)
      if (hipEventQuery(sl.ev) != hipSuccess) {
        (void)hipGetLastError();
        PSX_HIP(hipStreamWaitEvent(s, sl.ev, 0));
      }
      if (x.ldd == x.rows)
        PSX_HIP(hipMemcpyAsync(sl.p, x.dev, x.bytes(), hipMemcpyDeviceToHost, s));
      else
        PSX_HIP(hipMemcpy2DAsync(sl.p, colb, x.dev, x.ldd * sizeof(double), colb, (size_t)x.nc,
                                 hipMemcpyDeviceToHost, s));
      PSX_HIP(hipEventRecord(sl.ev, s));
    }
    Stage::Slot& sl = at(k);
    PSX_HIP(hipEventSynchronize(sl.ev));
    if (k == 0 && landed) (*landed)();
    const Chunk& x = ch[k];
    start_copy(sl, pool, inlined, x, true);
  }
  st.next = (int)((base + n) % ring);
}

void h2d_chunks(hipStream_t s, Stage& st, CopyPool& pool, const std::vector<Chunk>& ch) {
  const size_t n = ch.size();
  if (n == 0) return;
  st.grow((int)std::min<size_t>(n, Stage::kSlots));
  CopiesDone done{st, s};
  const int ring = st.have, base = st.next;
  const bool inlined = small(ch);
  auto at = [&](size_t k) -> Stage::Slot& { return st.slot[(base + k) % ring]; };
  size_t i = 0;
  for (size_t k = 0; k < n; ++k) {
    // host copies into every slot whose last DMA is over
    for (; i < n && i < k + ring; ++i) {
      Stage::Slot& sl = at(i);
      if (i > k && hipEventQuery(sl.ev) != hipSuccess) {
        (void)hipGetLastError();
        break;
      }
      PSX_HIP(hipEventSynchronize(sl.ev));
      const Chunk& x = ch[i];
      start_copy(sl, pool, inlined, x, false);
    }
    Stage::Slot& sl = at(k);
    wait_copied(sl);
    const Chunk& x = ch[k];
    const size_t colb = sizeof(double) * (size_t)x.rows;
    if (x.ldd == x.rows)
      PSX_HIP(hipMemcpyAsync(x.dev, sl.p, x.bytes(), hipMemcpyHostToDevice, s));
    else
      PSX_HIP(hipMemcpy2DAsync(x.dev, x.ldd * sizeof(double), sl.p, colb, colb, (size_t)x.nc,
                               hipMemcpyHostToDevice, s));
    PSX_HIP(hipEventRecord(sl.ev, s));
  }
  st.next = (int)((base + n) % ring);
}
}  // namespace

void d2h_matrices_on(hipStream_t s, Stage& stage, CopyPool& pool, const D2HMatrix* m, int nm,
                     int parts, const std::function<void()>* landed) {
  std::vector<Chunk> ch;
  int64_t total = 0;
  for (int i = 0; i < nm; ++i)
    total += std::max<int64_t>(m[i].rows, 0) * std::max<int64_t>(m[i].cols, 0);
  const int64_t most = chunk_doubles(total, parts);
  for (int i = 0; i < nm; ++i)
    cut(ch, most, m[i].host, m[i].ldh, const_cast<double*>(m[i].dev), m[i].ldd, m[i].rows, m[i].cols,
        m[i].after);
  if (ch.size() == 1 && ch[0].nc == 1 && !ch[0].after && !landed &&
      ch[0].bytes() > kDirectOutBytes && ch[0].bytes() <= kDirectBytes) {
    PSX_HIP(hipMemcpyAsync(ch[0].host, ch[0].dev, ch[0].bytes(), hipMemcpyDeviceToHost, s));
    PSX_HIP(hipStreamSynchronize(s));
    return;
  }
  d2h_chunks(s, stage, pool, ch, landed);
}

void d2h_matrices(Ctx* c, const D2HMatrix* m, int nm, const std::function<void()>* landed) {
  ensure_stage(c);
  d2h_matrices_on(c->stream, c->stage, *c->pool, m, nm, kParts, landed);
}

void d2h_matrix(Ctx* c, double* host, int64_t ldh, const double* dev, int64_t ldd,
                int64_t rows, int64_t cols) {
  const D2HMatrix m{host, ldh, dev, ldd, rows, cols};
  d2h_matrices(c, &m, 1);
}

void d2h_matrices_overlapped(Ctx* c, const D2HMatrix* m, int nm) {
  ensure_stage(c);
  d2h_matrices_on(c->xstream, c->stage, *c->pool, m, nm, kParts);
}

namespace {
void h2d_matrix_on(Ctx* c, hipStream_t s, double* dev, int64_t ldd, const double* host,
                   int64_t ldh, int64_t rows, int64_t cols) {
  std::vector<Chunk> ch;
  cut(ch, chunk_doubles(std::max<int64_t>(rows, 0) * std::max<int64_t>(cols, 0)),
      const_cast<double*>(host), ldh, dev, ldd, rows, cols, nullptr);
  if (ch.size() == 1 && ch[0].nc == 1 && ch[0].bytes() <= kDirectBytes) {
    PSX_HIP(hipMemcpyAsync(dev, host, ch[0].bytes(), hipMemcpyHostToDevice, s));
    return;
  }
  h2d_chunks(s, c->stage, *c->pool, ch);
}
}  // namespace

void h2d_matrix(Ctx* c, double* dev, int64_t ldd, const double* host, int64_t ldh,
                int64_t rows, int64_t cols) {
  ensure_stage(c);
  h2d_matrix_on(c, c->stream, dev, ldd, host, ldh, rows, cols);
}

void h2d_matrix_x(Ctx* c, double* dev, int64_t ldd, const double* host, int64_t ldh,
                  int64_t rows, int64_t cols) {
  ensure_stage(c);
  // behind the uploads of the context stream: side by side the earlier one, for
  // which kernels wait, would share the link (1 ms on two 100 MB maps)
  if (const int have = c->stage.have)
    PSX_HIP(hipStreamWaitEvent(c->xstream, c->stage.slot[(c->stage.next + have - 1) % have].ev, 0));
  h2d_matrix_on(c, c->xstream, dev, ldd, host, ldh, rows, cols);
  PSX_HIP(hipStreamSynchronize(c->xstream));
}

void h2d_pieces(Ctx* c, void* dev, const std::vector<HostPiece>& pieces) {
  ensure_stage(c);
  if (pieces.size() == 1 && pieces[0].bytes <= kDirectBytes) {
    PSX_HIP(hipMemcpyAsync((char*)dev + pieces[0].offset, pieces[0].host, pieces[0].bytes,
                           hipMemcpyHostToDevice, c->stream));
    return;
  }
  size_t end = 0;
  for (const HostPiece& p : pieces) end = std::max(end, p.offset + p.bytes);
  if (end <= Stage::kSlotBytes) {
    c->stage.grow(1);
    Stage::Slot& sl = c->stage.slot[c->stage.next];
    PSX_HIP(hipEventSynchronize(sl.ev));
    for (const HostPiece& p : pieces) std::memcpy(sl.p + p.offset, p.host, p.bytes);
    PSX_HIP(hipMemcpyAsync(dev, sl.p, end, hipMemcpyHostToDevice, c->stream));
    PSX_HIP(hipEventRecord(sl.ev, c->stream));
    c->stage.next = (c->stage.next + 1) % c->stage.have;
    return;
  }
  for (const HostPiece& p : pieces)
    h2d_matrix(c, (double*)((char*)dev + p.offset), (int64_t)(p.bytes / sizeof(double)),
               (const double*)p.host, (int64_t)(p.bytes / sizeof(double)),
               (int64_t)(p.bytes / sizeof(double)), 1);
}

}  // namespace psx
