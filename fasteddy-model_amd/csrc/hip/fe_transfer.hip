/*
 * fe_transfer.hip -- host arrays to and from the device, in pieces through pinned memory.
 *
 * The host modules' arrays are ordinary (pageable) memory, as the reference allocates them
 * (cuda_timeIntDevice.cu:53-87,198-257 copies them with cudaMemcpy).  The runtime copies pageable
 * memory at 30 GB/s to the device and 18 GB/s back, and a synchronisation per field left the bus
 * idle in between; the bus itself carries 57 GB/s to and from pinned memory.  So a transfer is
 * cut into pieces of at most 4 MB that go through a ring of pinned slots: while one piece is on
 * the bus, a few threads copy the next ones between the slots and the caller's arrays (one
 * thread copies at 24 GB/s, four at 82; a process bound to one core has no helpers, and still
 * gains: a moist 256 x 256 x 96 state 7.8 against 8.4 ms up, 7.9 against 13.6 down).  Everything is
 * enqueued on the caller's stream; an upload has read the caller's array when it returns, a download
 * has written it after xfer_finish.  A batch of the 512 x 512 x 128 model moves 0.86 GB up and 1.01 GB
 * down.
 */
#include "fe_host_copy.h"

namespace {

/* The ring: slot k is free, or on the bus (its event pending), towards `host` if that is set. */
constexpr int XF_SLOTS = 12;
constexpr size_t XF_PIECE = 4 << 20;
struct Xfer {
  char *buf = nullptr;
  size_t piece = 0;
  hipEvent_t ev[XF_SLOTS] = {};
  bool busy[XF_SLOTS] = {};
  char *host[XF_SLOTS] = {};
  size_t len[XF_SLOTS] = {};
  int next = 0;
} X;

int xfer_release() {
  if (!X.buf) return FE_OK;
  for (int k = 0; k < XF_SLOTS; ++k)
    if (X.busy[k]) (void)hipEventSynchronize(X.ev[k]);
  for (auto &e : X.ev) if (e) (void)hipEventDestroy(e);
  (void)hipHostFree(X.buf);
  X = Xfer();
  return FE_OK;
}

/* Slots for pieces of `bytes` (a whole field where it is smaller than XF_PIECE).  Without pinned
 * memory or events to be had, transfers are the runtime's copies of pageable memory. */
int xfer_reserve(size_t bytes) {
  const size_t want = (std::min(bytes, XF_PIECE) + 4095) / 4096 * 4096;
  if (X.buf && X.piece >= want) return FE_OK;
  xfer_release();
  void *p = nullptr;
  if (hipHostMalloc(&p, want * XF_SLOTS, hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();
    return FE_OK;
  }
  X.buf = (char *)p;
  X.piece = want;
  for (auto &e : X.ev)
    if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
      (void)hipGetLastError();
      e = nullptr;
      return xfer_release();
    }
  return FE_OK;
}

/* Waits for slot k; a piece on its way to the host goes on to the caller's array. */
int xfer_settle(int k) {
  if (!X.busy[k]) return FE_OK;
  X.busy[k] = false;
  HIPCHK(hipEventSynchronize(X.ev[k]));
  if (X.host[k]) g_copy.copy(X.host[k], X.buf + (size_t)k * X.piece, X.len[k]);
  X.host[k] = nullptr;
  return FE_OK;
}

/* n bytes of host memory to device memory on stream s. */
int xfer_up(hipStream_t s, void *dev, const void *host, size_t n) {
  int rc;
  if (!X.buf) {
    HIPCHK(hipMemcpyAsync(dev, host, n, hipMemcpyHostToDevice, s));
    HIPCHK(hipStreamSynchronize(s));
    return FE_OK;
  }
  for (size_t o = 0; o < n; o += X.piece) {
    const size_t len = std::min(X.piece, n - o);
    const int k = X.next;
    if ((rc = xfer_settle(k))) return rc;
    X.next = (k + 1) % XF_SLOTS;
    char *b = X.buf + (size_t)k * X.piece;
    g_copy.copy(b, (const char *)host + o, len);
    HIPCHK(hipMemcpyAsync((char *)dev + o, b, len, hipMemcpyHostToDevice, s));
    HIPCHK(hipEventRecord(X.ev[k], s));
    X.busy[k] = true;
    X.host[k] = nullptr;
  }
  return FE_OK;
}

/* n bytes of device memory to host memory on stream s; complete after xfer_finish. */
int xfer_down(hipStream_t s, void *host, const void *dev, size_t n) {
  int rc;
  if (!X.buf) {
    HIPCHK(hipMemcpyAsync(host, dev, n, hipMemcpyDeviceToHost, s));
    HIPCHK(hipStreamSynchronize(s));
    return FE_OK;
  }
  for (size_t o = 0; o < n; o += X.piece) {
    const size_t len = std::min(X.piece, n - o);
    const int k = X.next;
    if ((rc = xfer_settle(k))) return rc;
    X.next = (k + 1) % XF_SLOTS;
    HIPCHK(hipMemcpyAsync(X.buf + (size_t)k * X.piece, (const char *)dev + o, len, hipMemcpyDeviceToHost, s));
    HIPCHK(hipEventRecord(X.ev[k], s));
    X.busy[k] = true;
    X.host[k] = (char *)host + o;
    X.len[k] = len;
  }
  return FE_OK;
}

/* Every piece under way settled, oldest first, and the stream done. */
int xfer_finish(hipStream_t s) {
  int rc;
  for (int i = 0; i < XF_SLOTS; ++i)
    if ((rc = xfer_settle((X.next + i) % XF_SLOTS))) return rc;
  HIPCHK(hipStreamSynchronize(s));
  return FE_OK;
}

/* Below this, one array by itself is better left to the runtime's own copy: 8.4 MB 0.30 ms against
 * 0.34 through the ring, whose helpers are still waking; 67 MB 2.5 against 1.6 ms. */
constexpr size_t XF_LONE = 16 << 20;

/* A set of transfers: helpers poll while it is open; on an error, pieces that have not arrived are
 * dropped rather than copied to the caller's arrays later. */
struct XferScope {
  XferScope() { g_copy.begin(); }
  ~XferScope() {
    g_copy.end();
    for (int k = 0; k < XF_SLOTS; ++k)
      if (X.busy[k]) {
        (void)hipEventSynchronize(X.ev[k]);
        X.busy[k] = false;
        X.host[k] = nullptr;
      }
  }
};

}  // namespace
