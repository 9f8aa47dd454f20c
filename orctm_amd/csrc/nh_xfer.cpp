// nh_xfer.cpp -- bulk transfers through pinned chunks (nh_xfer.h).
#include "nh_xfer.h"

#include <string.h>

#include <algorithm>
#include <atomic>
#include <mutex>
#include <optional>
#include <thread>

#include "nh_lock.h"

namespace onh {
namespace {

struct Stage {
  bool taken = false;  // by a transfer, under Device::pick
  int device = -1;
  char* buf[kXferWorkers][2] = {};
  hipEvent_t ev[kXferWorkers][2] = {};
};

// One transfer to the device and one to the host at a time, each with a stage of its own: the first while it is free,
// so that a program that has one transfer under way at a time pins and gives back one stage.
struct Device {
  std::mutex way[2];  // to the device, to the host: held for a transfer; taken after device_lock() where both are
  std::mutex pick;
  Stage stage[2];
};

constexpr int kDevices = 16;  // device ordinals beyond share them
Device g_device[kDevices];
std::mutex g_count_mu;

// A stage for the holder of a way, given back at the end of the scope.
class Taken {
 public:
  explicit Taken(Device& d) : d_(d) {
    std::lock_guard<std::mutex> lk(d.pick);
    s_ = d.stage[0].taken ? &d.stage[1] : &d.stage[0];
    s_->taken = true;
  }
  ~Taken() {
    std::lock_guard<std::mutex> lk(d_.pick);
    s_->taken = false;
  }
  Taken(const Taken&) = delete;
  Taken& operator=(const Taken&) = delete;
  Stage& stage() { return *s_; }

 private:
  Device& d_;
  Stage* s_;
};
int g_handles = 0;

// Workers whose buffers and events are there.
int made(const Stage& s, int device) {
  int w = 0;
  while (s.device == device && w < kXferWorkers && s.buf[w][0] && s.buf[w][1] && s.ev[w][0] && s.ev[w][1]) ++w;
  return w;
}

void drop(Stage& s) {
  for (int w = 0; w < kXferWorkers; ++w)
    for (int q = 0; q < 2; ++q) {
      if (s.ev[w][q]) hipEventDestroy(s.ev[w][q]);
      if (s.buf[w][q]) hipHostFree(s.buf[w][q]);
      s.ev[w][q] = nullptr;
      s.buf[w][q] = nullptr;
    }
  s.device = -1;
}

// Buffers and events for `workers`, or for as many as there is memory to pin.
void make(Stage& s, int workers, int device) {
  if (s.device != device) drop(s);
  s.device = device;
  for (int w = 0; w < workers; ++w)
    for (int q = 0; q < 2; ++q) {
      hipError_t e = hipSuccess;
      if (!s.buf[w][q]) {
        void* p = nullptr;
        e = hipHostMalloc(&p, kXferChunk, hipHostMallocDefault);
        s.buf[w][q] = static_cast<char*>(p);
      }
      if (e == hipSuccess && !s.ev[w][q]) e = hipEventCreateWithFlags(&s.ev[w][q], hipEventDisableTiming);
      if (e != hipSuccess) {
        (void)hipGetLastError();  // or the next launch's check reports it
        return;
      }
    }
}

struct Chunk {
  const XferPiece* p = nullptr;
  size_t off = 0, len = 0;  // bytes of the piece
};

struct Plan {
  const XferPiece* p;
  int n;
  size_t step;                    // bytes of a chunk, a multiple of a double
  size_t first[kXferPieces + 1];  // chunk number at which a piece begins
  Plan(const XferPiece* pieces, int count, size_t chunk) : p(pieces), n(count), step(chunk) {
    first[0] = 0;
    for (int q = 0; q < n; ++q) first[q + 1] = first[q] + (p[q].bytes() + step - 1) / step;
  }
  size_t chunks() const { return first[n]; }
  Chunk chunk(size_t k) const {
    int q = 0;
    while (k >= first[q + 1]) ++q;
    const size_t off = (k - first[q]) * step;
    return Chunk{p + q, off, std::min(step, p[q].bytes() - off)};
  }
};

// The host half of a chunk.
void host_copy(const Chunk& c, char* buf, bool to_host) {
  const XferPiece& p = *c.p;
  for (size_t done = 0; done < c.len;) {
    const size_t at = c.off + done, row = at / p.row_bytes, in = at % p.row_bytes;
    const size_t m = std::min(p.row_bytes - in, c.len - done);
    char* h = p.host + row / p.rows * p.plane_stride + row % p.rows * p.row_stride + in;
    if (to_host) memcpy(h, buf + done, m);
    else memcpy(buf + done, h, m);
    done += m;
  }
}

hipError_t device_half(const Chunk& c, char* buf, bool to_host, hipStream_t st) {
  const XferPiece& p = *c.p;
  if (!p.dev_pitch)
    return to_host ? hipMemcpyAsync(buf, p.dev + c.off, c.len, hipMemcpyDeviceToHost, st)
                   : hipMemcpyAsync(p.dev + c.off, buf, c.len, hipMemcpyHostToDevice, st);
  const size_t w = sizeof(double);
  return launch_pack(st, reinterpret_cast<const double*>(p.dev), p.dev_pitch, p.dev_plane, p.row_bytes / w, p.rows,
                     c.off / w, c.len / w, reinterpret_cast<double*>(buf));
}

// One worker: chunks from the common counter through its two buffers. Every copy that it issued has
// finished when run() returns.
class Worker {
 public:
  Worker(Stage& s, int w, const Plan& plan, std::atomic<size_t>& next, bool to_host, hipStream_t st)
      : s_(s), w_(w), plan_(plan), next_(next), to_host_(to_host), st_(st) {}
  // The next chunk's copies, into a buffer that is not in use any more; false: no chunk left, or an error.
  bool issue() {
    if (err_ != hipSuccess) return false;
    const size_t k = next_++;
    if (k >= plan_.chunks()) return false;
    const int q = q_;
    settle(q);
    held_[q] = plan_.chunk(k);
    if (!to_host_) host_copy(held_[q], s_.buf[w_][q], false);
    hipError_t e = device_half(held_[q], s_.buf[w_][q], to_host_, st_);
    if (e == hipSuccess) e = hipEventRecord(s_.ev[w_][q], st_);
    if (e == hipSuccess) {
      pending_[q] = true;
    } else {
      hipStreamSynchronize(st_);  // a copy without an event may still use the buffer
      err_ = e;
    }
    q_ ^= 1;
    return true;
  }
  hipError_t run() {
    while (issue())
      if (to_host_) settle(q_);  // the chunk before, while this one is on its way
    settle(q_);
    settle(q_ ^ 1);
    return err_;
  }

 private:
  void settle(int q) {
    if (!pending_[q]) return;
    pending_[q] = false;
    const hipError_t e = hipEventSynchronize(s_.ev[w_][q]);
    if (err_ == hipSuccess) err_ = e;
    if (to_host_ && e == hipSuccess) host_copy(held_[q], s_.buf[w_][q], true);
  }
  Stage& s_;
  const int w_;
  const Plan& plan_;
  std::atomic<size_t>& next_;
  const bool to_host_;
  const hipStream_t st_;
  hipError_t err_ = hipSuccess;
  Chunk held_[2];
  bool pending_[2] = {false, false};
  int q_ = 0;
};

// What the runtime knows of the memory: pinned or managed by the caller, on a device, or nothing.
hipMemoryType type_of(const void* host) {
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, host) == hipSuccess) return a.type;
  (void)hipGetLastError();
  return hipMemoryTypeUnregistered;
}

// The pieces through the runtime's own copies: flat ones queued, rows a plane at a time.
hipError_t direct(hipStream_t st, const XferPiece* p, int n, bool to_host) {
  hipError_t e = hipSuccess;
  bool flat = true;
  for (int q = 0; q < n && e == hipSuccess; ++q) {
    flat = flat && p[q].flat();
    if (!p[q].flat()) continue;
    e = to_host ? hipMemcpyAsync(p[q].host, p[q].dev, p[q].bytes(), hipMemcpyDeviceToHost, st)
                : hipMemcpyAsync(p[q].dev, p[q].host, p[q].bytes(), hipMemcpyHostToDevice, st);
  }
  if (!to_host && e == hipSuccess && flat) return e;  // what is queued next follows; the caller waits for that anyway
  const hipError_t es = hipStreamSynchronize(st);
  if (e == hipSuccess) e = es;
  for (int q = 0; q < n; ++q) {
    if (p[q].flat() || !p[q].bytes()) continue;
    std::lock_guard<std::recursive_mutex> dev(device_lock());
    const size_t w = sizeof(double), pitch = p[q].dev_pitch ? p[q].dev_pitch * w : p[q].row_bytes,
                 plane = p[q].dev_pitch ? p[q].dev_plane * w : p[q].row_bytes * p[q].rows;
    for (size_t k = 0; k < p[q].planes && e == hipSuccess; ++k) {
      char *h = p[q].host + k * p[q].plane_stride, *d = p[q].dev + k * plane;
      e = to_host ? hipMemcpy2D(h, p[q].row_stride, d, pitch, p[q].row_bytes, p[q].rows, hipMemcpyDeviceToHost)
                  : hipMemcpy2D(d, pitch, h, p[q].row_stride, p[q].row_bytes, p[q].rows, hipMemcpyHostToDevice);
    }
  }
  return e;
}

hipError_t transfer(int device, hipStream_t st, const XferPiece* p, int n, bool to_host) {
  if (n < 0 || n > kXferPieces) return hipErrorInvalidValue;
  size_t bytes = 0;
  bool flat = true;
  for (int q = 0; q < n; ++q) {
    bytes += p[q].bytes();
    flat = flat && p[q].flat();
  }
  if (flat && bytes < (to_host ? kXferDirectHost : kXferDirectDevice)) return direct(st, p, n, to_host);
  bool held = flat || bytes >= kXferHeldRows, far = false;
  for (int q = 0; q < n; ++q) {
    const hipMemoryType t = type_of(p[q].host);
    held = held && t != hipMemoryTypeUnregistered;
    far = far || t == hipMemoryTypeDevice;  // not for the host's threads
  }
  if (held || far) return direct(st, p, n, to_host);
  const size_t part = (bytes / 12 + 7) / 8 * 8;
  const Plan plan(p, n, to_host ? std::min(std::max(part, kXferChunk / 8), kXferChunk) : kXferChunk);
  if (plan.chunks() == 0) return hipSuccess;
  int want = bytes >= kXferThreaded ? (int)std::min<size_t>(kXferWorkers, plan.chunks()) : 1;
  // kernels that the transfer follows end before it holds the stage: it holds others up for its copies' time alone
  // (asked first: a wait puts a marker of its own on the stream, 20 us of a 128x128x30 interior's 170)
  hipError_t es = hipStreamQuery(st);
  if (es == hipErrorNotReady) {
    (void)hipGetLastError();
    es = hipStreamSynchronize(st);
  }
  if (es != hipSuccess) return es;
  Device& d = g_device[(unsigned)device % kDevices];
  std::unique_lock<std::mutex> lk(d.way[to_host]);
  std::optional<Taken> at;  // given back before the way
  at.emplace(d);
  if (made(at->stage(), device) < want) {  // allocates: not while another thread captures a graph
    at.reset();
    lk.unlock();
    std::lock_guard<std::recursive_mutex> dev(device_lock());
    lk.lock();
    at.emplace(d);
    make(at->stage(), want, device);
  }
  Stage& s = at->stage();
  want = std::min(want, made(s, device));
  if (want == 0) {  // no memory to pin
    at.reset();
    lk.unlock();
    return direct(st, p, n, to_host);
  }
  std::atomic<size_t> next{0};
  hipError_t got[kXferWorkers] = {};
  std::thread team[kXferWorkers];
  Worker self(s, 0, plan, next, to_host, st);
  if (to_host && self.issue()) self.issue();  // on their way while the others are made
  for (int w = 1; w < want; ++w) {
    try {
      team[w] = std::thread([&, w] {
        const hipError_t e = hipSetDevice(device);
        got[w] = e == hipSuccess ? Worker(s, w, plan, next, to_host, st).run() : e;
      });
    } catch (...) {
      break;  // no thread or no memory for one to be had: the others take its share
    }
  }
  got[0] = self.run();
  for (std::thread& t : team)
    if (t.joinable()) t.join();
  for (hipError_t e : got)
    if (e != hipSuccess) return e;
  return hipSuccess;
}

}  // namespace

XferPiece xfer_flat(void* dev, const void* host, size_t bytes) {
  XferPiece p;
  p.dev = static_cast<char*>(dev);
  p.host = static_cast<char*>(const_cast<void*>(host));
  p.row_bytes = bytes;
  return p;
}

XferPiece xfer_interior(void* dev, const void* host, int IE, int JE, int KE, size_t dev_pitch, size_t dev_plane) {
  XferPiece p;
  p.dev = static_cast<char*>(dev);
  p.host = static_cast<char*>(const_cast<void*>(host)) + sizeof(double) * (1 + (size_t)IE);
  p.row_bytes = sizeof(double) * (size_t)(IE - 2);
  p.rows = (size_t)(JE - 2);
  p.planes = (size_t)KE;
  p.row_stride = sizeof(double) * (size_t)IE;
  p.plane_stride = p.row_stride * (size_t)JE;
  p.dev_pitch = dev_pitch;
  p.dev_plane = dev_plane;
  return p;
}

hipError_t xfer_to_device(int device, hipStream_t st, const XferPiece* p, int n) {
  for (int q = 0; q < n; ++q)
    if (p[q].dev_pitch) return hipErrorInvalidValue;
  return transfer(device, st, p, n, false);
}

hipError_t xfer_to_host(int device, hipStream_t st, const XferPiece* p, int n) {
  return transfer(device, st, p, n, true);
}

void xfer_retain() {
  std::lock_guard<std::mutex> lk(g_count_mu);
  ++g_handles;
}

void xfer_release() {
  std::lock_guard<std::recursive_mutex> dev(device_lock());
  std::lock_guard<std::mutex> lk(g_count_mu);
  if (--g_handles > 0) return;
  for (Device& d : g_device) {
    std::scoped_lock ways(d.way[0], d.way[1]);
    for (Stage& s : d.stage)
      if (s.device >= 0) drop(s);
  }
}

}  // namespace onh
