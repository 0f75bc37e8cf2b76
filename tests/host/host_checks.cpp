// Checks of the library's host side that need no GPU: the program stands in
// for the HIP runtime (memory is host memory, a launch is noted and not run),
// so that what the host code allocates, keeps, launches and does after a
// failing call can be looked at.  Built and run by tests/test_host_side.py.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <string>
#include <vector>

#include "internal.hpp"

using namespace omega_hip;

#define CHECK(cond)                                                     \
  do {                                                                  \
    if (!(cond)) {                                                      \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #cond);            \
      std::exit(1);                                                     \
    }                                                                   \
  } while (0)

// ---------------------------------------------------------------------------
// The HIP runtime this program runs on
// ---------------------------------------------------------------------------
namespace fake {
std::map<void *, size_t> live; // device allocations
size_t bytes = 0;
int fail_after = -1; // allocations until one fails, -1: none does

struct Launched {
  dim3 grid, block;
  hipStream_t stream;
};
std::vector<Launched> launches;
} // namespace fake

extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
  if (fake::fail_after == 0) return hipErrorOutOfMemory;
  if (fake::fail_after > 0) --fake::fail_after;
  *p = std::calloc(1, n); // pages are taken when they are first written
  if (!*p) return hipErrorOutOfMemory;
  fake::live[*p] = n;
  fake::bytes += n;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  if (!p) return hipSuccess;
  CHECK(fake::live.count(p));
  fake::bytes -= fake::live[p];
  fake::live.erase(p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemset(void *p, int v, size_t n) {
  if (v || !fake::live.count(p)) std::memset(p, v, n);
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *, dim3 grid, dim3 block, void **, size_t, hipStream_t s) {
  fake::launches.push_back({grid, block, s});
  return hipSuccess;
}
static fake::Launched pushed;
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t, hipStream_t s) {
  pushed = {grid, block, s};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, hipStream_t *s) {
  *grid = pushed.grid;
  *block = pushed.block;
  *shared = 0;
  *s = pushed.stream;
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "no GPU here"; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s) {
  return *s = hipStreamCaptureStatusNone, hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return *e = nullptr, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 1, hipSuccess; }
}

// Tables of a lattice whose rows have as many levels as 24-bit byte strides
// hold, and one more: 8 bytes a level in a row, 24 in a cell's three edges.
static void tall() {
  for (int L : {64, 699050, 699051, 2097151, 2097152}) {
    DeviceMesh dm;
    build_planar_hex(dm.host, 6, 4, 1.0, L);
    dm.build_device(OMEGA_ORDER_HILBERT);
    std::printf("L %d off32 %d stage %d\n", L, (int)dm.off32, (int)dm.stage_ok);
    CHECK(dm.hex_ok && dm.coef_uni);
    CHECK(dm.off32 == (8.0 * L < 1 << 24));
    CHECK(dm.stage_ok == (24.0 * L < 1 << 24));
  }
}

int main(int argc, char **argv) {
  const std::map<std::string, std::function<void()>> checks = {{"tall", tall}};
  CHECK(argc == 2 && checks.count(argv[1]));
  checks.at(argv[1])();
  std::printf("%s ok\n", argv[1]);
}
