// CPU test of the launches of the driver kernels (fishfry_amd/csrc/ff_field.hip),
// host side only: the HIP launch calls are link stand-ins that refuse what the
// runtime may refuse -- more than 64 KB of dynamic LDS for a kernel that
// has not been given it (hipFuncAttributeMaxDynamicSharedMemorySize), grids of
// no or of too many workgroups -- and record the tiles, which must cover the
// grid.  No kernel runs.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

#include "ff_internal.hpp"

#define REQUIRE(c)                                                     \
  do {                                                                 \
    if (!(c)) {                                                        \
      std::fprintf(stderr, "FAILED %s (line %d)\n", #c, __LINE__);     \
      std::exit(1);                                                    \
    }                                                                  \
  } while (0)

namespace {

std::map<const void*, int> g_max_lds;  // kernel -> dynamic LDS it was given
struct {
  dim3 grid, block;
  size_t lds = 0;
  hipStream_t stream = nullptr;
} g_cfg, g_first;       // pushed configuration; first launch since reset()
int g_launches = 0;
hipError_t g_last = hipSuccess;
std::string g_error;

void reset() { g_launches = 0; }

}  // namespace

extern "C" {

hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s) {
  g_cfg = {grid, block, lds, s};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* s) {
  *grid = g_cfg.grid;
  *block = g_cfg.block;
  *lds = g_cfg.lds;
  *s = g_cfg.stream;
  return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void* fn, hipFuncAttribute attr, int value) {
  if (attr != hipFuncAttributeMaxDynamicSharedMemorySize || value > 160 * 1024) return hipErrorInvalidValue;
  g_max_lds[fn] = value;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* fn, dim3 grid, dim3 block, void**, size_t lds, hipStream_t s) {
  const size_t limit = g_max_lds.count(fn) ? (size_t)g_max_lds[fn] : 65536;
  hipError_t e = hipSuccess;
  if (lds > limit || !grid.x || (uint64_t)grid.x * block.x > UINT32_MAX) e = hipErrorInvalidValue;
  if (e == hipSuccess && !g_launches++) g_first = {grid, block, lds, s};
  if (e != hipSuccess) g_last = e;
  return e;
}
hipError_t hipGetLastError() {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
void __hipUnregisterFatBinary(void**) {}

}  // extern "C"

namespace ff {

ff_status set_error(ff_status st, const std::string& msg) {
  g_error = msg;
  return st;
}
ff_status hip_check(hipError_t e, const char* what) { return e == hipSuccess ? FF_OK : set_error(FF_ERR_HIP, what); }
ff_status device_scratch(size_t, double** out) {
  static double buf[kDiffDoubles];
  *out = buf;
  return FF_OK;
}

}  // namespace ff

static ff_field field(int ni, int nj, int nk, int nmodes) {
  ff_field f;
  std::memset(&f, 0, sizeof f);
  f.n[0] = ni, f.n[1] = nj, f.n[2] = nk;
  for (int a = 0; a < 3; ++a) f.d[a] = f.dd[a] = 1.0;
  f.scale = 1.0;
  f.nmodes = nmodes;
  return f;
}

// Both kernels launch, with the workgroups the grid needs (16 rows, 64 columns
// and at most 64 planes to a tile; field_init runs up to 2^20 of them at once, the error
// sums up to 1024).
static void check(int ni, int nj, int nk, int nmodes) {
  const ff_field f = field(ni, nj, nk, nmodes);
  double out[3];
  double* phi = reinterpret_cast<double*>(0x1000);  // never read: no kernel runs
  const long long across = (1 + (nj - 1LL) / 16) * (1 + (nk - 1LL) / 64);
  const long long fewest = across * (1 + (ni - 1LL) / 64), most = across * (1 + (ni - 1LL) / 4);
  std::printf("%d x %d x %d, %d modes\n", ni, nj, nk, nmodes);
  std::fflush(stdout);
  for (int diff = 0; diff < 2; ++diff) {
    reset();
    const ff_status st = diff ? ff::field_diff(&f, phi, out, nullptr) : ff::field_init(&f, phi, nullptr);
    if (st != FF_OK) std::fprintf(stderr, "%s\n", g_error.c_str());
    REQUIRE(st == FF_OK);
    REQUIRE(g_launches == 1 + diff);
    const long long cap = diff ? 1024 : 1 << 20;
    REQUIRE(g_first.block.x == 256);
    REQUIRE(g_first.grid.x >= std::min(fewest, cap) && g_first.grid.x <= std::min(most, cap));
    const size_t modes = nmodes == 0 ? 0 : nmodes <= 16 ? 16 : 32;
    REQUIRE(g_first.lds <= 160 * 1024 - 3 * 256 * 8);
    REQUIRE(g_first.lds >= 16 * (4 + 16 + 64) * (modes + 1));  // a (cos, sin) pair per coordinate and mode
  }
}

int main() {
  // around the planes per tile (4 to 64, by the grid), for each number of mode registers
  for (int nmodes : {0, 1, 16, 17, 32})
    for (int n : {1, 5, 64, 130, 484, 512, 1024}) {
      check(n, n, n, nmodes);
      check(n, 1, 3 * n, nmodes);
    }
  // extents up to the type's largest
  const int top = 2147483647;
  for (int n : {top, top - 1, top - 15, top - 16, top - 62, top - 63, top - 255, top - 256}) {
    check(n, 1, 1, 17);
    check(1, n, 1, 17);
    check(1, 1, n, 17);
  }
  std::printf("field launches ok\n");
  return 0;
}
