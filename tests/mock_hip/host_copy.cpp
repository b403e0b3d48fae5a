// The staged host copies of csrc/ctx.hip on the stand-in runtime: the case
// named by the first argument; 0 if it holds.
#include "../../powerspectra.jl_amd/csrc/psx_internal.h"

#include <new>

static thread_local int new_fails_at = -1;   // the n-th allocation from now fails
void* operator new(size_t n) {
  if (new_fails_at >= 0 && new_fails_at-- == 0) throw std::bad_alloc();
  if (void* p = std::malloc(n)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

namespace psx {
void release_blas(Ctx*) {}
void release_tile_cache(Ctx*) {}
void release_mix_tiles(Ctx*) {}
void release_sht_plans(Ctx*) {}
void noalloc_init_device(int) {}
}  // namespace psx
using namespace psx;

static Ctx* context() {
  psx_ctx* h = nullptr;
  if (psx_ctx_create(0, 0, &h) != PSX_OK) std::abort();
  return reinterpret_cast<Ctx*>(h);
}

static std::vector<double> numbers(size_t n, double first) {
  std::vector<double> v(n);
  for (size_t i = 0; i < n; ++i) v[i] = first + (double)i;
  return v;
}

// a matrix there and back, through each pair of streams, with columns apart
static bool round_trips() {
  Ctx* c = context();
  bool ok = true;
  const int64_t shapes[][3] = {{1, 1, 1}, {7, 5, 9}, {300, 300, 300}, {1000, 900, 1001},
                               {8192, 1, 8192}, {8193, 1, 8193}, {512, 256, 512}, {131073, 1, 131073},
                               {5000000, 1, 5000000}, {2000000, 4, 2000003}};
  for (auto& s : shapes)
    for (int x = 0; x < 4; ++x) {
      const int64_t rows = s[0], cols = s[1], ld = s[2];
      const std::vector<double> a = numbers(ld * cols, 1.0);
      std::vector<double> b(ld * cols, -1.0);
      double* d = (double*)ctx_alloc(c, sizeof(double) * rows * cols);
      if (x & 1) h2d_matrix_x(c, d, rows, a.data(), ld, rows, cols);
      else h2d_matrix(c, d, rows, a.data(), ld, rows, cols);
      const D2HMatrix m{b.data(), ld, d, rows, rows, cols};
      if (!(x & 1) && (x & 2)) (void)hipStreamSynchronize(c->stream);
      if (x & 2) d2h_matrices_overlapped(c, &m, 1);
      else d2h_matrices(c, &m, 1);
      for (int64_t j = 0; j < cols; ++j)
        for (int64_t i = 0; i < ld; ++i)
          ok = ok && b[j * ld + i] == (i < rows ? a[j * ld + i] : -1.0);
      ctx_free(c, d);
    }
  return psx_ctx_destroy((psx_ctx*)c) == PSX_OK && ok;
}

// a copy that fails part way leaves nothing in flight on its stream: the buffers
// on either side are the next call's
static bool nothing_in_flight_after_an_error() {
  bool ok = true;
  for (int kind = 0; kind < 4; ++kind)
    for (int at = 0; at < 8; ++at) {
      Ctx* c = context();
      const int64_t n = 4000000;
      std::vector<double> a = numbers(n, 1.0);
      double* d = (double*)ctx_alloc(c, sizeof(double) * n);
      ensure_stage(c);
      const D2HMatrix m{a.data(), n, d, n, n, 1};
      mock::fail_copy = at;
      bool threw = false;
      try {
        if (kind == 0) h2d_matrix(c, d, n, a.data(), n, n, 1);
        if (kind == 1) h2d_matrix_x(c, d, n, a.data(), n, n, 1);
        if (kind == 2) d2h_matrices(c, &m, 1);
        if (kind == 3) d2h_matrices_overlapped(c, &m, 1);
      } catch (const Error&) {
        threw = true;
      }
      mock::fail_copy = -1;
      ok = ok && threw && c->stream->ops.empty() && c->xstream->ops.empty();
      ctx_free(c, d);
      ok = ok && psx_ctx_destroy((psx_ctx*)c) == PSX_OK;
    }
  return ok;
}

// nor does an error in a call that has its device buffer filled: what is queued
// reads the caller's memory and writes the buffer
static bool nothing_in_flight_when_a_buffer_is_given_back() {
  bool ok = true;
  for (int x = 0; x < 2; ++x) {
    Ctx* c = context();
    ensure_stage(c);
    const std::vector<double> a = numbers(1000, 1.0);
    try {
      XferBuf buf(c, sizeof(double) * a.size());
      double* d = buf.take(sizeof(double) * a.size());
      PSX_HIP(hipMemcpyAsync(d, a.data(), sizeof(double) * a.size(), hipMemcpyHostToDevice,
                             x ? c->xstream : c->stream));
      PSX_REQUIRE(false, PSX_ERR_ARGUMENT, "an error");
    } catch (const Error&) {
    }
    ok = ok && c->stream->ops.empty() && c->xstream->ops.empty();
    ok = ok && psx_ctx_destroy((psx_ctx*)c) == PSX_OK;
  }
  return ok;
}

// a pool that cannot have all its threads works with those it has; one that
// cannot be made at all is an error, not the end of the process
static bool pool_without_memory() {
  int made = 0;
  for (int at = 0; at < 40; ++at) {
    std::unique_ptr<CopyPool> p;
    try {
      new_fails_at = at;
      p = std::make_unique<CopyPool>(8);
    } catch (const std::bad_alloc&) {
    }
    new_fails_at = -1;
    if (!p) continue;
    ++made;
    std::atomic<int> done{0};
    for (int i = 0; i < 20; ++i) p->submit([&] { ++done; });
    while (done < 20) std::this_thread::yield();
  }
  return made > 30;
}

int main(int argc, char** argv) {
  const std::string which = argc > 1 ? argv[1] : "";
  if (which == "round_trips") return round_trips() ? 0 : 1;
  if (which == "nothing_in_flight_after_an_error")
    return nothing_in_flight_after_an_error() ? 0 : 1;
  if (which == "nothing_in_flight_when_a_buffer_is_given_back")
    return nothing_in_flight_when_a_buffer_is_given_back() ? 0 : 1;
  if (which == "pool_without_memory") return pool_without_memory() ? 0 : 1;
  return 2;
}
