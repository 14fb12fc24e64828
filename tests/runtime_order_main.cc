// poly_hip_order_after's own part of the runtime (csrc/runtime_hip.cc) against a HIP runtime
// that is acted out here: streams and events as plain records, no device.
//
//   threads    events left after calls from many short-lived threads
//   device     a caller whose current device is another one than the backend's
//   capture    a stream that is being captured, and others while it is
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <set>
#include <thread>
#include <vector>

#include "runtime_hip.h"

struct FakeStream { int device; bool busy, capturing; };
struct FakeEvent { int device; bool in_capture; };

static std::mutex lock;
static std::set<FakeEvent *> events;
static int created = 0, most = 0, waits = 0, bad = 0;
static thread_local int current = 0;
static FakeStream default_streams[4] = {{0, false, false}, {1, false, false}, {2, false, false}, {3, false, false}};
static hipStream_t waited_on_behalf;        // that of the last wait
static thread_local hipStream_t recorded;   // the stream of the thread's last record
static FakeStream *as(hipStream_t s) { return s ? (FakeStream *)s : &default_streams[current]; }

extern "C" {
hipError_t hipGetDeviceCount(int *n) { *n = 4; return hipSuccess; }
hipError_t hipSetDevice(int d) { current = d; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = current; return hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t *d) { *d = as(s)->device; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t) new FakeStream{current, false, false}; return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *c) {
  *c = as(s)->capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t s) { return as(s)->busy ? hipErrorNotReady : hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "refused"; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  std::lock_guard<std::mutex> g(lock);
  FakeEvent *f = new FakeEvent{current, false};
  events.insert(f);
  created++;
  if ((int)events.size() > most) most = (int)events.size();
  *e = (hipEvent_t)f;
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  std::lock_guard<std::mutex> g(lock);
  if (!events.erase((FakeEvent *)e)) return hipErrorInvalidHandle;
  delete (FakeEvent *)e;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  FakeEvent *f = (FakeEvent *)e;
  if (f->device != as(s)->device) return hipErrorInvalidHandle;    // an event and its stream are one device's
  if (f->in_capture) bad++;                                        // an event that a capture still knows, used again
  f->in_capture = as(s)->capturing;
  recorded = (hipStream_t)as(s);
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) {
  std::lock_guard<std::mutex> g(lock);
  waits++;
  waited_on_behalf = recorded;
  return hipSuccess;
}
}

#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)

int main(int argc, char **argv) {
  if (argc < 2) return 2;
  setenv("POLY_HIP_DEVICE", "2", 1);
  if (polyhip::runtime_init() != 0) return 3;
  FakeStream side{2, true, false}, idle{2, false, false};
  if (!strcmp(argv[1], "threads")) {
    for (int round = 0; round < 16; round++) {
      std::vector<std::thread> t;
      std::atomic<int> failed{0};
      for (int i = 0; i < 8; i++) t.emplace_back([&] { current = 2; for (int k = 0; k < 4; k++) failed += polyhip::runtime_order_after(&side) != 0; });
      for (auto &x : t) x.join();
      CHECK(failed == 0);
    }
    CHECK(waits == 16 * 8 * 4);
    CHECK(most <= 8);              // no more than callers at a time
  } else if (!strcmp(argv[1], "device")) {
    int after = -1;
    int rc[3] = {-1, -1, -1};
    std::thread([&] {              // (a thread starts on device 0)
      rc[0] = polyhip::runtime_order_after(&side);
      default_streams[2].busy = true;
      rc[1] = polyhip::runtime_order_after(nullptr);
      rc[2] = waited_on_behalf == (hipStream_t)&default_streams[2] ? 0 : 1;
      after = current;
    }).join();
    CHECK(rc[0] == 0);
    CHECK(rc[1] == 0 && rc[2] == 0);
    CHECK(after == 0);             // the caller's device is as it was
    FakeStream far{1, true, false};      // a stream of another device than the backend's
    CHECK(polyhip::runtime_order_after(&far) == 0 && polyhip::runtime_order_after(&side) == 0);
  } else if (!strcmp(argv[1], "capture")) {
    FakeStream captured{2, false, true};
    CHECK(polyhip::runtime_order_after(&captured) == 0 && waits == 1);
    CHECK(polyhip::runtime_order_after(&side) == 0 && waits == 2);
    CHECK(polyhip::runtime_order_after(&captured) == 0 && waits == 3);
    CHECK(bad == 0);
    CHECK(polyhip::runtime_order_after(&idle) == 0 && waits == 3);
  } else {
    return 2;
  }
  printf("ok\n");
  return 0;
}
