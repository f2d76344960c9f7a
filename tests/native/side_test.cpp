// The side-stream pool against stubbed HIP calls: prints one line per check that fails.
#include <atomic>
#include <cstdio>
#include <memory>
#include <thread>
#include <vector>

#include "../../fermix_amd/csrc/side.hip"

static int g_device = 0, g_streams = 0, g_events = 0;
static bool g_capturing = false;
hipError_t hipGetDevice(int* d) { *d = g_device; return 0; }
hipError_t hipDeviceGetAttribute(int* v, int, int) { *v = 256; return 0; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* c) { *c = g_capturing; return 0; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)(size_t)(0x1000 + 16 * ++g_streams); return 0; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t)(size_t)(0x9000 + 16 * ++g_events); return 0; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return 0; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return 0; }

static int fails = 0;
#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); ++fails; } } while (0)

static hipStream_t caller(int k) { return (hipStream_t)(size_t)(16 * k); }

static hipStream_t side_of(hipStream_t s) {
  fx::SideStream x(s, true);
  CHECK(x.ok());
  CHECK(x.fork() == FX_OK && x.fork() != FX_OK && x.join() == FX_OK && x.join() == FX_OK);
  return x.side();
}

int main() {
  // two callers on streams of their own do not share a side stream; each keeps its own
  const hipStream_t a = side_of(caller(1)), b = side_of(caller(2));
  CHECK(a != b && a != caller(1) && b != caller(2));
  CHECK(side_of(caller(1)) == a && side_of(caller(2)) == b && side_of(caller(1)) == a);
  CHECK(g_streams == 2 && g_events == 4);
  // the null stream is a caller like any other
  const hipStream_t z = side_of(nullptr);
  CHECK(z != a && z != b && side_of(nullptr) == z && side_of(caller(1)) == a);
  // bounded: many callers share four, the one unused for longest first
  std::vector<hipStream_t> seen;
  for (int k = 10; k < 60; ++k) seen.push_back(side_of(caller(k)));
  CHECK(g_streams == 4 && g_events == 8);
  for (size_t k = 4; k < seen.size(); ++k) CHECK(seen[k] == seen[k - 4]);
  {  // held by running calls: never handed out twice, and nobody waits
    std::vector<std::unique_ptr<fx::SideStream>> run;
    for (int k = 0; k < 4; ++k) run.emplace_back(new fx::SideStream(caller(70 + k), true));
    for (int i = 0; i < 4; ++i)
      for (int j = 0; j < i; ++j) CHECK(run[i]->ok() && run[i]->side() != run[j]->side());
    fx::SideStream full(caller(80), true);
    CHECK(!full.ok() && full.side() == caller(80) && full.fork() != FX_OK && full.join() == FX_OK);
  }
  CHECK(side_of(caller(70)) != caller(70));
  g_capturing = true;
  { fx::SideStream x(caller(1), true); CHECK(!x.ok() && x.side() == caller(1)); }
  g_capturing = false;
  { fx::SideStream x(caller(1), false); CHECK(!x.ok()); }
  g_device = 1;  // another device, another pool
  const hipStream_t d1 = side_of(caller(1));
  g_device = 0;
  CHECK(side_of(caller(1)) != d1);
  std::atomic<int> busy[64] = {};
  std::atomic<int> clash{0};
  std::vector<std::thread> th;
  for (int t = 0; t < 8; ++t)
    th.emplace_back([&, t] {
      for (int r = 0; r < 20000; ++r) {
        fx::SideStream x(caller(90 + t), true);
        if (!x.ok()) continue;
        const size_t k = ((size_t)x.side() - 0x1000) / 16;
        if (busy[k].fetch_add(1)) clash++;
        busy[k].fetch_sub(1);
      }
    });
  for (auto& t : th) t.join();
  CHECK(clash == 0);
  if (!fails) printf("ok\n");
  return fails != 0;
}
