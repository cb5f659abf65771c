// launch.hpp against a runtime that refuses launches: the error is reported once, by the call that met it, and is not left behind in the
// runtime for the next one.
#include <cstdio>

#include "launch.hpp"

namespace {
hipError_t g_last = hipSuccess, g_lookup = hipSuccess, g_launch = hipSuccess;
hipError_t done(hipError_t e) {
  if (e != hipSuccess) g_last = e;
  return e;
}
int g_failed = 0;
void expect(bool ok, const char* what) {
  if (!ok) { std::printf("failed: %s\n", what); ++g_failed; }
}
void kernel(uint32_t, uint64_t) {}
}  // namespace

extern "C" {
hipError_t hipGetLastError() {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
hipError_t hipGetFuncBySymbol(hipFunction_t* f, const void*) {
  if (g_lookup == hipSuccess) *f = reinterpret_cast<hipFunction_t>(16);
  return done(g_lookup);
}
hipError_t hipModuleLaunchKernel(hipFunction_t, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned, hipStream_t, void**, void**) {
  return done(g_launch);
}
}

namespace rmlx {
DeviceCtx& ctx() {
  static DeviceCtx c;
  return c;
}
}  // namespace rmlx

int main() {
  using namespace rmlx;
  auto launch = [] { Launch<kernel>::go(dim3(1), dim3(64), 0, nullptr, 1u, 2ull); };
  for (hipError_t* at : {&g_lookup, &g_launch}) {
    *at = hipErrorInvalidValue;
    launch();
    *at = hipSuccess;
    launch();  // (a launch behind the one that failed does not hide it)
    expect(take_launch_error() == hipErrorInvalidValue, "the error of a launch");
    expect(hipGetLastError() == hipSuccess, "nothing left for the next call");
    launch();
    expect(take_launch_error() == hipSuccess, "a launch behind it");
  }
  if (g_failed == 0) std::printf("launch errors ok\n");
  return g_failed;
}
