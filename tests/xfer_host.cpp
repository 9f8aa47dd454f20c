// The transfers of orctm_amd/csrc/nh_xfer.cpp on the host, over a runtime of this file's own in which device memory
// is host memory, a copy is done when it is queued and a stream ends when the check says so. Each check is an argument; prints OK.
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <future>
#include <map>
#include <mutex>
#include <new>
#include <set>
#include <vector>

#include "../orctm_amd/csrc/nh_xfer.cpp"

static std::atomic<long> g_pins{0}, g_pin_limit{1 << 20}, g_copies{0}, g_waits{0};
static std::atomic<bool> g_no_new{false};
static thread_local hipError_t g_last = hipSuccess;
static std::mutex g_mu;
static std::condition_variable g_cv;
static std::set<hipStream_t> g_busy;  // streams whose work has not ended
static std::map<hipEvent_t, hipStream_t> g_at;
static const hipStream_t kStuck = reinterpret_cast<hipStream_t>(8);
static bool g_stuck = false;          // the copies on kStuck do not end
static std::set<const void*> g_held;  // arrays pinned by the caller
static const char* g_far = nullptr;   // an array on the device

void* operator new(size_t n) {
  if (g_no_new) throw std::bad_alloc();
  if (void* p = malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }

std::recursive_mutex& onh::device_lock() {
  static std::recursive_mutex m;
  return m;
}

extern "C" {
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  if (g_pins >= g_pin_limit) {
    *p = nullptr;
    return g_last = hipErrorOutOfMemory;
  }
  ++g_pins;
  *p = malloc(n);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  --g_pins;
  free(p);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = reinterpret_cast<hipEvent_t>(malloc(1));
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  free(e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t st) {
  std::lock_guard<std::mutex> lk(g_mu);
  g_at[e] = st;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t st) {
  ++g_waits;
  std::unique_lock<std::mutex> lk(g_mu);
  g_cv.wait(lk, [&] { return !g_busy.count(st); });
  return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t st) {
  std::lock_guard<std::mutex> lk(g_mu);
  return g_busy.count(st) ? g_last = hipErrorNotReady : hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  std::unique_lock<std::mutex> lk(g_mu);
  const hipStream_t st = g_at[e];
  g_cv.wait(lk, [&] { return !g_busy.count(st) && !(g_stuck && st == kStuck); });
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  if (g_far && p >= g_far && p < g_far + (size_t(1) << 28)) {
    a->type = hipMemoryTypeDevice;
    return hipSuccess;
  }
  for (const void* h : g_held)
    if (p >= h && p < (const char*)h + (size_t(1) << 30)) {
      a->type = hipMemoryTypeHost;
      return hipSuccess;
    }
  return g_last = hipErrorInvalidValue;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  ++g_copies;
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpy2D(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, hipMemcpyKind) {
  ++g_copies;
  for (size_t r = 0; r < h; ++r) memcpy((char*)d + r * dp, (const char*)s + r * sp, w);
  return hipSuccess;
}
}

hipError_t onh::launch_pack(hipStream_t, const double* src, size_t pitch, size_t plane, size_t nx, size_t ny, size_t first,
                            size_t n, double* out) {
  for (size_t t = 0; t < n; ++t) {
    const size_t e = first + t, row = e / nx;
    out[t] = src[row / ny * plane + row % ny * pitch + e % nx];
  }
  return hipSuccess;
}

using namespace onh;

static void need(bool ok, const char* what) {
  if (ok) return;
  printf("failed: %s\n", what);
  exit(1);
}

static std::vector<double> numbers(size_t n, double at) {
  std::vector<double> v(n);
  for (size_t i = 0; i < n; ++i) v[i] = at + (double)i;
  return v;
}

// An interior of IE x JE x KE to the host and two arrays each way, compared with loops.
static void round_trip(int IE, int JE, int KE, size_t flat, hipStream_t st = nullptr) {
  const size_t pitch = (size_t)(IE - 2 + 31) / 32 * 32, plane = pitch * (size_t)(JE - 2);
  const std::vector<double> dev = numbers(plane * KE, 0.5);
  std::vector<double> host = numbers((size_t)IE * JE * KE, -1e9), want = host;
  for (int k = 0; k < KE; ++k)
    for (int j = 0; j < JE - 2; ++j)
      for (int i = 0; i < IE - 2; ++i)
        want[(size_t)(i + 1) + (size_t)IE * (j + 1 + (size_t)JE * k)] = dev[(size_t)i + pitch * j + plane * k];
  const XferPiece p = xfer_interior((void*)dev.data(), host.data(), IE, JE, KE, pitch, plane);
  need(xfer_to_host(0, st, &p, 1) == hipSuccess && host == want, "interior to the host");
  for (const bool down : {false, true}) {
    const std::vector<double> a = numbers(flat, 1.0), b = numbers(flat / 3 + 1, 7.0);
    std::vector<double> x(a.size()), y(b.size());
    XferPiece two[2];
    if (down) {
      two[0] = xfer_flat((void*)a.data(), x.data(), a.size() * 8);
      two[1] = xfer_flat((void*)b.data(), y.data(), b.size() * 8);
    } else {
      two[0] = xfer_flat(x.data(), a.data(), a.size() * 8);
      two[1] = xfer_flat(y.data(), b.data(), b.size() * 8);
    }
    need((down ? xfer_to_host(0, st, two, 2) : xfer_to_device(0, st, two, 2)) == hipSuccess && x == a && y == b,
         down ? "arrays to the host" : "arrays to the device");
  }
}

static const struct {
  int IE, JE, KE;
  size_t flat;
} kSizes[] = {{3, 3, 1, 1}, {99, 43, 5, 1000}, {130, 130, 32, 600000}, {131, 129, 40, 2100000}, {333, 301, 41, 5000003}};

// As much memory as there is to pin, from none to all of it.
static void no_memory_to_pin() {
  for (long limit = 0; limit <= 2 * kXferWorkers + 1; ++limit) {
    xfer_retain();
    g_pin_limit = limit;
    for (const auto& s : kSizes) round_trip(s.IE, s.JE, s.KE, s.flat);
    need(g_last == hipSuccess, "no error is left behind");
    xfer_release();
    need(g_pins == 0, "the chunks are given back");
  }
}

// No thread to be had: nothing can be allocated while the transfer runs.
static void no_threads() {
  xfer_retain();
  round_trip(333, 301, 41, 5000003);
  const size_t n = 5000003;
  const std::vector<double> a = numbers(n, 3.0);
  std::vector<double> x(n);
  const XferPiece p = xfer_flat(x.data(), a.data(), n * 8);
  g_no_new = true;
  const hipError_t e = xfer_to_device(0, nullptr, &p, 1);
  g_no_new = false;
  need(e == hipSuccess && x == a, "one worker alone");
  xfer_release();
}

// Arrays that the caller pinned are copied by the runtime, in one piece each; an interior of fewer bytes than
// kXferHeldRows and one array of two that is pinned go through the chunks.
static void held_by_the_runtime() {
  xfer_retain();
  const size_t n = 5000003, IE = 402, JE = 302, KE = 100, pitch = 416, plane = pitch * 300;
  std::vector<double> dev = numbers(n, 3.0), box = numbers(plane * KE, 0.0);
  char* mem = (char*)calloc(size_t(1) << 30, 1);
  double* host = (double*)mem;
  g_held.insert(mem);
  XferPiece two[2] = {xfer_flat(dev.data(), host, n * 8), xfer_flat(dev.data(), host + n, n * 8)};
  g_copies = 0;
  need(xfer_to_host(0, nullptr, two, 2) == hipSuccess && g_copies == 2 && g_pins == 0, "pinned arrays to the host");
  need(!memcmp(host, dev.data(), n * 8) && !memcmp(host + n, dev.data(), n * 8), "their values");
  need(xfer_to_device(0, nullptr, two, 2) == hipSuccess && g_copies == 4 && g_pins == 0, "pinned arrays to the device");
  XferPiece in = xfer_interior(box.data(), host, IE, JE, KE, pitch, plane);
  need(in.bytes() >= kXferHeldRows && xfer_to_host(0, nullptr, &in, 1) == hipSuccess && g_pins == 0, "pinned rows");
  for (size_t k = 0; k < KE; ++k)
    for (size_t j = 0; j < JE - 2; ++j)
      need(!memcmp(host + 1 + IE * (j + 1 + JE * k), box.data() + plane * k + pitch * j, (IE - 2) * 8), "their values");
  in = xfer_interior(box.data(), host, IE, JE, 10, pitch, plane);
  need(xfer_to_host(0, nullptr, &in, 1) == hipSuccess && g_pins > 0, "few pinned rows");
  std::vector<double> other(n);
  two[0] = xfer_flat(dev.data(), other.data(), n * 8);
  g_copies = 0;
  need(xfer_to_host(0, nullptr, two, 2) == hipSuccess && g_copies > 2 && other == dev, "one of two pinned");
  need(g_last == hipSuccess, "no error is left behind");
  xfer_release();
  g_held.clear();
  free(mem);
}

// An array on the device in the place of the caller's is left to the runtime, whatever its size.
static void on_the_device() {
  xfer_retain();
  char* mem = (char*)calloc(size_t(1) << 28, 1);
  double* to = (double*)mem;
  g_far = mem;
  for (size_t KE : {1, 10, 100}) {
    const size_t IE = 402, JE = 302, pitch = 416, plane = pitch * 300;
    const std::vector<double> box = numbers(plane * KE, 0.5 + (double)KE);
    const XferPiece p = xfer_interior((void*)box.data(), to, IE, JE, (int)KE, pitch, plane);
    need(xfer_to_host(0, nullptr, &p, 1) == hipSuccess && g_pins == 0, "rows to the device's memory");
    for (size_t k = 0; k < KE; ++k)
      for (size_t j = 0; j < JE - 2; ++j)
        need(!memcmp(to + 1 + IE * (j + 1 + JE * k), box.data() + plane * k + pitch * j, (IE - 2) * 8), "their values");
  }
  const size_t n = 3000003;
  const std::vector<double> a = numbers(n, 3.0);
  std::vector<double> x(n);
  const XferPiece two[2] = {xfer_flat((void*)a.data(), to, n * 8), xfer_flat((void*)a.data(), x.data(), n * 8)};
  need(xfer_to_host(0, nullptr, two, 2) == hipSuccess && g_pins == 0 && !memcmp(to, a.data(), n * 8) && x == a,
       "one of two on the device");
  xfer_release();
  g_far = nullptr;
  free(mem);
}

// A small upload is queued and not waited for.
static void queued() {
  const std::vector<double> a = numbers(1000, 3.0);
  std::vector<double> x(1000), y(1000);
  const XferPiece two[2] = {xfer_flat(x.data(), a.data(), 8000), xfer_flat(y.data(), a.data(), 8000)};
  xfer_retain();
  need(xfer_to_device(0, nullptr, two, 2) == hipSuccess && g_copies == 2 && g_waits == 0 && x == a && y == a, "queued");
  xfer_release();
}

static bool ends(std::future<void>& f) { return f.wait_for(std::chrono::seconds(5)) == std::future_status::ready; }

// A transfer whose stream is busy, and one whose copies are on their way, leave the others alone.
static void side_by_side() {
  const hipStream_t busy = reinterpret_cast<hipStream_t>(16);
  const auto& s = kSizes[3];
  xfer_retain();
  g_busy.insert(busy);
  auto waits = std::async(std::launch::async, [&] { round_trip(s.IE, s.JE, s.KE, s.flat, busy); });
  std::this_thread::sleep_for(std::chrono::milliseconds(200));
  auto other = std::async(std::launch::async, [&] { round_trip(s.IE, s.JE, s.KE, s.flat); });
  const bool ended = ends(other);
  {
    std::lock_guard<std::mutex> lk(g_mu);
    g_busy.clear();
    g_cv.notify_all();
  }
  waits.wait();
  other.wait();
  need(ended, "a transfer beside one that waits for its stream");

  const size_t n = 5000003;
  const std::vector<double> a = numbers(n, 3.0), b = numbers(n, 5.0);
  std::vector<double> x(n), y(n);
  const XferPiece down = xfer_flat((void*)a.data(), x.data(), n * 8), up = xfer_flat(y.data(), b.data(), n * 8);
  g_stuck = true;
  auto first = std::async(std::launch::async, [&] { need(xfer_to_host(0, kStuck, &down, 1) == hipSuccess, "down"); });
  std::this_thread::sleep_for(std::chrono::milliseconds(200));
  auto second = std::async(std::launch::async, [&] { need(xfer_to_device(0, nullptr, &up, 1) == hipSuccess, "up"); });
  const bool passed = ends(second);
  {
    std::lock_guard<std::mutex> lk(g_mu);
    g_stuck = false;
    g_cv.notify_all();
  }
  first.wait();
  second.wait();
  need(passed && x == a && y == b, "up beside down");
  xfer_release();
}

// A program with one transfer under way at a time pins one stage, both ways.
static void one_stage() {
  xfer_retain();
  for (int q = 0; q < 2; ++q) round_trip(kSizes[4].IE, kSizes[4].JE, kSizes[4].KE, kSizes[4].flat);
  need(g_pins == 2 * kXferWorkers, "one stage");
  xfer_release();
  need(g_pins == 0, "given back");
}

int main(int argc, char** argv) {
  const char* what = argc > 1 ? argv[1] : "";
  if (!strcmp(what, "pin")) no_memory_to_pin();
  else if (!strcmp(what, "threads")) no_threads();
  else if (!strcmp(what, "held")) held_by_the_runtime();
  else if (!strcmp(what, "device")) on_the_device();
  else if (!strcmp(what, "beside")) side_by_side();
  else if (!strcmp(what, "stage")) one_stage();
  else if (!strcmp(what, "queued")) queued();
  else need(false, "an unknown check");
  printf("OK\n");
  return 0;
}
