// nh_xfer.h -- bulk transfers between the caller's (pageable) arrays and the device.
//
// A transfer is a list of pieces, cut into chunks of at most kXferChunk bytes. Each chunk passes through a
// pinned buffer, so that the host half (the copy between the caller's rows and the buffer) of one chunk
// overlaps the device half of others, and a transfer of kXferThreaded bytes or more shares its chunks out
// between the caller and kXferWorkers - 1 threads that live as long as the call: one thread copies
// 31 GB/s here, two 57-62, four 75-78, and the link moves 57 GB/s. A 1024x768x60 interior (377 MB) takes
// 7.5 ms to the host (one strided runtime copy per level, as before: 338 ms), 8.4 ms to the device (one
// pageable runtime copy: 12.8 ms). Chunks to the host are a twelfth of the transfer, 512 KiB at least
// (203x194x35: 0.34 ms, 0.54 in chunks of 4 MiB by one thread); to the device they are 4 MiB, since smaller
// ones lose more to the copies' own overhead than the overlap gains (128x128x30: 0.20 ms in one chunk,
// 0.28 in 12).
// Contiguous transfers below kXferDirectDevice and kXferDirectHost go to the runtime as they are: its own
// staging is as fast there (128x128x30 to the device: 0.16 ms). So do arrays that the runtime holds already (pinned by
// the caller): the device reads and writes them itself (1024x768x60 to the device: 6.8 ms, 8.4 through the chunks;
// 256x256x33: 0.35, 0.53), rows of an interior from kXferHeldRows on (to the host 7.1 ms, 7.5 through the chunks;
// below, the copy commands of the levels cost more than the chunks: 400x300x40 0.98 ms, 0.88; 128x128x30 0.29, 0.17).
// A piece whose host side lies on a device goes to the runtime's copies at any size: no thread of the host touches it.
// The pinned buffers (kXferWorkers * 2 chunks, 32 MiB) and their events belong to the device. One transfer each way is
// under way at a time, and only while its copies run, not while it waits for kernels (two threads of 1024x768 surfaces:
// 2.4 ms a solve each, 3.2 while it was held over the sweeps); a second set of buffers is made where both ways meet (a
// set for each way cost a program that closes its last handle 6 ms of the next one's making, 323x293x42). They are
// freed with the process's last handle. Where no memory can be pinned, a transfer works with as many workers as have
// their buffers, or through the runtime.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

namespace onh {

constexpr size_t kXferChunk = size_t(4) << 20;
constexpr int kXferWorkers = 4;
constexpr size_t kXferThreaded = size_t(4) << 20;
constexpr size_t kXferDirectDevice = size_t(16) << 20;
constexpr size_t kXferDirectHost = size_t(1) << 20;
constexpr size_t kXferHeldRows = size_t(64) << 20;

// One piece: on the host `planes` planes of `rows` rows of `row_bytes` bytes; on the device the same bytes in
// that order, contiguous, or (dev_pitch != 0, reading from the device only) doubles at
// plane * dev_plane + row * dev_pitch + column.
struct XferPiece {
  char* host = nullptr;
  size_t row_bytes = 0, rows = 1, planes = 1;
  size_t row_stride = 0, plane_stride = 0;
  char* dev = nullptr;
  size_t dev_pitch = 0, dev_plane = 0;
  size_t bytes() const { return row_bytes * rows * planes; }
  bool flat() const { return rows * planes == 1 && !dev_pitch; }
};

XferPiece xfer_flat(void* dev, const void* host, size_t bytes);
// The interior (2..IE-1, 2..JE-1, 1..KE) of a Fortran array (IE,JE,KE) of doubles.
XferPiece xfer_interior(void* dev, const void* host, int IE, int JE, int KE, size_t dev_pitch, size_t dev_plane);

// At most this many pieces in a call.
constexpr int kXferPieces = 8;
// Ordered on `st`. To the host, it returns when every piece has arrived. To the device, work queued on `st` afterwards
// finds the pieces there, and the caller waits for `st` before it gives the host arrays back (a wait of its own here
// took 2 us of a small set_rhs's 36).
hipError_t xfer_to_device(int device, hipStream_t st, const XferPiece* p, int n);
hipError_t xfer_to_host(int device, hipStream_t st, const XferPiece* p, int n);

// Every handle that transfers holds one.
void xfer_retain();
void xfer_release();

// nh_kernels.hip: elements first .. first + n - 1, in the order i, j, k of an nx x ny x (any) box, of a
// padded array, to out.
hipError_t launch_pack(hipStream_t st, const double* src, size_t pitch, size_t plane, size_t nx, size_t ny,
                       size_t first, size_t n, double* out);

}  // namespace onh
