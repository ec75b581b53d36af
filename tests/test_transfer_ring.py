"""The pinned ring of the transfers (csrc/hip/fe_transfer.hip) in a C++ program of its own, on a stand-in
for the runtime whose device memory is host memory: arrays of less than a piece to many pieces arrive
whole both ways, with the ring, without pinned memory and where an event of the ring cannot be had (then
the copies are the runtime's own), and the ring comes and goes without a trace."""
import os
import subprocess

import pytest

SOURCE = r"""
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <algorithm>
#include <vector>
/* the stand-in: copies happen when they are enqueued; resources are counted and can run out */
typedef void *hipStream_t;
struct Event { bool recorded; };
typedef Event *hipEvent_t;
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };
enum { hipHostMallocDefault = 0, hipEventDisableTiming = 2 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
static int events_left = 1 << 30, pinned_left = 1 << 30, events = 0, pinned = 0;
static hipError_t hipGetLastError() { return hipSuccess; }
static hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  if (pinned_left-- <= 0) return hipErrorOutOfMemory;
  ++pinned;
  *p = malloc(n);
  return hipSuccess;
}
static hipError_t hipHostFree(void *p) { --pinned; free(p); return hipSuccess; }
static hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  if (events_left-- <= 0) return hipErrorOutOfMemory;
  ++events;
  *e = new Event{false};
  return hipSuccess;
}
static hipError_t hipEventDestroy(hipEvent_t e) { --events; delete e; return hipSuccess; }
static hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { if (!e) abort(); e->recorded = true; return hipSuccess; }
static hipError_t hipEventSynchronize(hipEvent_t e) { if (!e || !e->recorded) abort(); return hipSuccess; }
static hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
static hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
enum { FE_OK = 0, FE_ERR_HIP = 9 };
#define HIPCHK(x) do { if ((x) != hipSuccess) return FE_ERR_HIP; } while (0)
#include "fe_transfer.hip"

static int round_trip(size_t n, unsigned seed) {
  std::vector<unsigned char> a(n), d(n), b(n, 0);
  for (size_t i = 0; i < n; ++i) a[i] = (unsigned char)((i + seed) * 2654435761u >> 11);
  int rc;
  if ((rc = xfer_reserve(n))) return rc;
  XferScope scope;
  if ((rc = xfer_up(nullptr, d.data(), a.data(), n))) return rc;
  if ((rc = xfer_finish(nullptr))) return rc;
  if ((rc = xfer_down(nullptr, b.data(), d.data(), n))) return rc;
  if ((rc = xfer_finish(nullptr))) return rc;
  return a == b && a == d ? 0 : 100;
}

int main(int argc, char **argv) {
  if (!strcmp(argv[1], "events")) events_left = atoi(argv[2]);
  if (!strcmp(argv[1], "pinned")) pinned_left = atoi(argv[2]);
  const size_t sizes[] = {1, 4096, 4097, 1 << 20, XF_PIECE, XF_PIECE + 1, 13 * XF_PIECE + 5, 3};
  int rc;
  for (int k = 0; k < 2; ++k)
    for (size_t n : sizes)
      if ((rc = round_trip(n, (unsigned)n + k))) {
        printf("%zu bytes: %d\n", n, rc);
        return 1;
      }
  xfer_release();
  if (events != 0 || pinned != 0) return 2;
  return (rc = round_trip(9000, 1)) ? 1 : 0;
}
"""


@pytest.fixture(scope="module")
def program(repo, tmp_path_factory):
    d = tmp_path_factory.mktemp("ring")
    (d / "main.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O2", "-pthread", "-I" + os.path.join(repo, "fasteddy-model_amd", "csrc", "hip"),
                    str(d / "main.cpp"), "-o", str(d / "main")], check=True)
    return str(d / "main")


@pytest.mark.parametrize("what,left", [("all", 0), ("pinned", 0), ("pinned", 1), ("events", 0), ("events", 5), ("events", 12),
                                       ("events", 17)])
def test_ring(program, what, left):
    r = subprocess.run([program, what, str(left)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout)
