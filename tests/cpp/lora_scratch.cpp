// ltx25_lora_add's host side on a CPU: this program stands in for the HIP runtime calls and the
// kernel launchers that the library makes (its definitions come first in the symbol search), so
// that what a call allocates, launches and hands to a launch can be seen without a GPU. The
// planners are the library's own.
//
//   lora_scratch SCENARIO [ARGS]    exits 0 and prints nothing, or says what is wrong
#include "common.h"
#include "ltx25_qlinear.h"

#include <dlfcn.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>
#include <vector>

namespace {

int g_failures = 0;

#define EXPECT(cond, ...)              \
  do {                                 \
    if (!(cond)) {                     \
      ++g_failures;                    \
      std::printf("line %d: ", __LINE__); \
      std::printf(__VA_ARGS__);        \
      std::printf("\n");               \
    }                                  \
  } while (0)

// ---- device memory: addresses only, never touched ----
std::map<uintptr_t, size_t> g_mem;
uintptr_t g_next = (uintptr_t)1 << 44;
std::set<hipStream_t> g_capturing;   // streams

// The bytes left in the allocation that holds p, 0 outside of all
size_t room(const void* p)
{
  auto it = g_mem.upper_bound((uintptr_t)p);
  if (it == g_mem.begin()) { return 0; }
  --it;
  const uintptr_t end = it->first + it->second;
  return (uintptr_t)p < end ? end - (uintptr_t)p : 0;
}

// ---- launches ----
struct Launch {
  std::string what;
  hipStream_t stream;
  std::vector<std::pair<uintptr_t, size_t>> scratch;   // library scratch it reads or writes
};
std::vector<Launch> g_launches;   // and the event calls between them

void note(const char* what, hipStream_t st, std::initializer_list<std::pair<const void*, size_t>> use)
{
  Launch l{what, st, {}};
  for (const auto& u : use) {
    if (u.first == nullptr || u.second == 0 || room(u.first) == 0) { continue; }   // the caller's
    EXPECT(room(u.first) >= u.second, "%s: %zu bytes at %p, %zu allocated", what, u.second,
           u.first, room(u.first));
    l.scratch.push_back({(uintptr_t)u.first, u.second});
  }
  g_launches.push_back(l);
}

bool g_busy = false;                   // no stream's work ends
hipError_t g_error = hipSuccess;       // what hipGetLastError finds
int g_plans = 0;                       // made by the present call
int g_set_after = 0, g_set_tile = 0;   // another thread sets the tile after that many of them

}  // namespace

// ---- the HIP runtime ----
extern "C" {

hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int)
{
  std::memset(p, 0, sizeof *p);
  std::strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n)
{
  if (!g_capturing.empty()) { return hipErrorStreamCaptureUnsupported; }
  *p = (void*)g_next;
  g_mem[g_next] = n;
  g_next += (n + 0xffff) & ~(size_t)0xffff;
  return hipSuccess;
}
hipError_t hipFree(void* p) { return g_mem.erase((uintptr_t)p) ? hipSuccess : hipErrorInvalidValue; }
hipError_t hipDeviceSynchronize()
{
  return g_capturing.empty() ? hipSuccess : hipErrorStreamCaptureUnsupported;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned)
{
  static uintptr_t next = 0x100;
  *e = (hipEvent_t)next++;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t st)
{
  g_launches.push_back({"record " + std::to_string((uintptr_t)e), st, {}});
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t st, hipEvent_t e, unsigned)
{
  g_launches.push_back({"wait " + std::to_string((uintptr_t)e), st, {}});
  return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t) { return g_busy ? g_error = hipErrorNotReady : hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t)
{
  EXPECT(!g_busy, "the host waits for a stream");
  return hipSuccess;
}
hipError_t hipGetLastError()
{
  const hipError_t e = g_error;
  g_error = hipSuccess;
  return e;
}
hipError_t hipStreamIsCapturing(hipStream_t st, hipStreamCaptureStatus* s)
{
  *s = g_capturing.count(st) != 0 ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode*) { return hipSuccess; }

}  // extern "C"

// ---- the kernels' launchers ----
namespace ltx25 {

GemmPlan plan_gemm(int M, int N, int K, int bits, int cu_count, int force, bool panels)
{
  using Fn = GemmPlan (*)(int, int, int, int, int, int, bool);
  static const Fn real = (Fn)dlsym(RTLD_NEXT, "_ZN5ltx259plan_gemmEiiiiiib");
  if (real == nullptr) { std::printf("no planner in the library\n"); std::exit(2); }
  const GemmPlan p = real(M, N, K, bits, cu_count, force, panels);
  if (++g_plans == g_set_after) { ltx25_set_tile(g_set_tile); }
  return p;
}

hipError_t launch_gemm(const GemmDesc& d, const GemmPlan& plan, float* ws, hipStream_t st)
{
  EXPECT(plan.workspace_bytes == 0 || room(ws) >= plan.workspace_bytes,
         "GEMM %d x %d -> %d: %zu bytes of partials, %zu at %p", d.M, d.K, d.N,
         plan.workspace_bytes, room(ws), (void*)ws);
  EXPECT(g_error == hipSuccess, "an error is left for the launch's check");
  note("gemm", st, {{ws, plan.workspace_bytes}, {d.x, (size_t)d.M * d.K * 2},
                    {d.w, (size_t)(d.wn > 0 ? d.wn : d.N) * d.K * 2}, {d.y, (size_t)d.M * d.N * 2}});
  return d.done != nullptr ? hipEventRecord(d.done, st) : hipSuccess;
}

hipError_t launch_lora(const uint16_t*, const uint16_t*, const uint16_t* b, uint16_t*, int M, int,
                       int N, int rank, int ldb, bool, int, hipStream_t st, const uint16_t* r_in,
                       bool, hipEvent_t done)
{
  note(r_in != nullptr ? "lora y" : "lora", st,
       {{b, ((size_t)(N - 1) * ldb + rank) * 2}, {r_in, (size_t)M * rank * 2}});
  return done != nullptr ? hipEventRecord(done, st) : hipSuccess;
}

hipError_t launch_lora_pad(const uint16_t*, int rows, int, int, uint16_t* dst, int ld_dst,
                           hipStream_t st, int)
{
  note("pad", st, {{dst, (size_t)rows * ld_dst * 2}});
  return hipSuccess;
}

}  // namespace ltx25

namespace {

// A call's operands: four addresses that no allocation holds
int add(hipStream_t st, int M, int K, int N, int rank, int b_off = 0)
{
  char* const x = (char*)((uintptr_t)1 << 40);
  return ltx25_lora_add(st, x, x + (1 << 30), x + (2ul << 30) + b_off, x + (3ul << 30), nullptr,
                        nullptr, M, K, N, rank);
}

// The last kernel
std::string last_launch()
{
  for (size_t i = g_launches.size(); i-- > 0;) {
    if (g_launches[i].what.find(' ') == std::string::npos || g_launches[i].what == "lora y") {
      return g_launches[i].what;
    }
  }
  return "";
}

// The tile switch changes after the call's n-th plan: what runs fits what was reserved for it, also
// where the y GEMM splits K under one setting and not under the other.
void tile_switch(int rank, int from, int to, int n)
{
  ltx25_set_tile(from);
  g_set_after = n;
  g_set_tile = to;
  EXPECT(add((hipStream_t)0x1000, 128, 2048, 16384, rank) == LTX25_OK, "%s", ltx25_last_error());
  EXPECT(last_launch() == "gemm", "not the GEMM pair");
}

// Calls on several streams at once: no two of them use the same bytes of scratch.
void overlap(int M, int K, int N, int rank, int b_off)
{
  for (int i = 0; i < 3; ++i) {
    for (int s = 1; s <= 4; ++s) {
      EXPECT(add((hipStream_t)(uintptr_t)(0x1000 * s), M, K, N, rank, b_off) == LTX25_OK, "%s",
             ltx25_last_error());
    }
  }
  EXPECT(g_launches.size() > 12, "the one-pass kernel alone");
  for (const Launch& l : g_launches) {
    for (const Launch& o : g_launches) {
      if (l.stream == o.stream) { continue; }
      for (const auto& p : l.scratch) {
        for (const auto& q : o.scratch) {
          EXPECT(p.first + p.second <= q.first || q.first + q.second <= p.first,
                 "%s of one stream and %s of another share scratch", l.what.c_str(),
                 o.what.c_str());
        }
      }
    }
  }
}

// A call, then the same under capture, on its own stream and on another one: it allocates nothing.
void capture(int M, int K, int N, int rank, int b_off)
{
  const hipStream_t st = (hipStream_t)0x1000, other = (hipStream_t)0x2000;
  EXPECT(add(st, M, K, N, rank, b_off) == LTX25_OK, "%s", ltx25_last_error());
  for (hipStream_t c : {st, other}) {
    g_capturing = {c};
    g_launches.clear();
    EXPECT(add(c, M, K, N, rank, b_off) == LTX25_OK, "captured: %s", ltx25_last_error());
    EXPECT(last_launch() == "lora", "not the one-pass kernel");
    g_capturing.clear();
  }
}

// One stream after another, each idle before the next: every one gets scratch, eight allocations
// serve them all. With eight of them busy a ninth runs the one-pass kernel, until one is idle.
void streams_come_and_go()
{
  for (int s = 1; s <= 30; ++s) {
    EXPECT(add((hipStream_t)(uintptr_t)(0x1000 * s), 128, 4096, 1032, 32) == LTX25_OK, "%s",
           ltx25_last_error());
    EXPECT(last_launch() == "lora y", "stream %d runs the one-pass kernel", s);
  }
  EXPECT(g_mem.size() == 8, "%zu allocations", g_mem.size());
  g_busy = true;
  EXPECT(add((hipStream_t)0x100, 128, 4096, 1032, 32) == LTX25_OK, "%s", ltx25_last_error());
  EXPECT(last_launch() == "lora", "a ninth stream beside eight busy ones: %s",
         last_launch().c_str());
  EXPECT(g_error == hipSuccess, "an error is left behind");
  EXPECT(add((hipStream_t)0x1e000, 128, 4096, 1032, 32) == LTX25_OK, "%s", ltx25_last_error());
  EXPECT(last_launch() == "lora y", "a busy stream with scratch of its own");
  g_busy = false;
  EXPECT(add((hipStream_t)0x100, 128, 8192, 1032, 64) == LTX25_OK, "%s", ltx25_last_error());
  EXPECT(last_launch() == "lora y", "an idle slot is not taken");
  EXPECT(g_mem.size() == 8, "%zu allocations", g_mem.size());
}

// A handle that comes back may be another stream's, while the one that had it still runs: the
// second call waits for the event that the first recorded behind its launches.
void recycled_handle(int M, int K, int N, int rank)
{
  const hipStream_t st = (hipStream_t)0x1000;
  g_busy = true;
  EXPECT(add(st, M, K, N, rank) == LTX25_OK, "%s", ltx25_last_error());
  const std::string last = g_launches.empty() ? "" : g_launches.back().what;
  EXPECT(last.rfind("record ", 0) == 0, "no event behind the launches");
  const std::string e = last.size() > 7 ? last.substr(7) : "";
  g_launches.clear();
  EXPECT(add(st, M, K, N, rank) == LTX25_OK, "%s", ltx25_last_error());
  EXPECT(!g_launches.empty() && g_launches.front().what == "wait " + e, "no wait before launches");
}

}  // namespace

int main(int argc, char** argv)
{
  const std::string s = argc > 1 ? argv[1] : "";
  auto arg = [&](int i) { return argc > i ? std::atoi(argv[i]) : 0; };
  if (s == "tile_switch") { tile_switch(arg(2), arg(3), arg(4), arg(5)); }
  else if (s == "overlap") { overlap(arg(2), arg(3), arg(4), arg(5), arg(6)); }
  else if (s == "capture") { capture(arg(2), arg(3), arg(4), arg(5), arg(6)); }
  else if (s == "streams_come_and_go") { streams_come_and_go(); }
  else if (s == "recycled_handle") { recycled_handle(arg(2), arg(3), arg(4), arg(5)); }
  else { std::printf("unknown scenario %s\n", s.c_str()); return 2; }
  return g_failures == 0 ? 0 : 1;
}
