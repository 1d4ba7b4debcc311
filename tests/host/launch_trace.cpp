// Stand-in for the HIP runtime symbols that libsbq.so links: no GPU, no
// launch.  Each kernel launch is recorded (kernel name, grid, block, LDS
// bytes) and reported as successful, so that a host program sees which
// kernels a call of the C ABI dispatches to.  Loaded before the library, with
// its symbols global (dispatch.py).
#include <stddef.h>
#include <stdint.h>
#include <string.h>

#include <map>
#include <string>
#include <vector>

namespace {

struct Dim3 {
  uint32_t x, y, z;
};
struct Launch {
  std::string kernel;
  Dim3 grid, block;
  size_t lds;
};
std::map<const void*, std::string>& names() {
  static std::map<const void*, std::string> m;
  return m;
}
std::vector<Launch> launches;
Dim3 pushed_grid, pushed_block;
size_t pushed_lds;
void* pushed_stream;
alignas(256) char symbol[256];

}  // namespace

extern "C" {

void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*,
                           int*) {
  names()[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t lds, void* stream) {
  pushed_grid = grid;
  pushed_block = block;
  pushed_lds = lds;
  pushed_stream = stream;
  return 0;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* lds, void** stream) {
  *grid = pushed_grid;
  *block = pushed_block;
  *lds = pushed_lds;
  *stream = pushed_stream;
  return 0;
}
int hipLaunchKernel(const void* host, Dim3 grid, Dim3 block, void**, size_t lds, void*) {
  launches.push_back({names()[host], grid, block, lds});
  return 0;
}
int hipGetLastError() { return 0; }
int hipGetDevice(int* dev) {
  *dev = 0;
  return 0;
}
int hipGetDevicePropertiesR0600(void*, int) { return 1; }
int hipGetSymbolAddress(void** p, const void*) {
  *p = symbol;
  return 0;
}

// The recorded launches: their number, launch i (0 if there is no such
// launch), and forgetting them.
int trace_count() { return (int)launches.size(); }
int trace_get(int i, char* kernel, size_t len, int64_t* dims /* grid xyz, block xyz, LDS */) {
  if (i < 0 || i >= (int)launches.size() || len == 0) return 0;
  const Launch& l = launches[i];
  strncpy(kernel, l.kernel.c_str(), len - 1);
  kernel[len - 1] = 0;
  const int64_t d[7] = {l.grid.x, l.grid.y, l.grid.z, l.block.x, l.block.y, l.block.z, (int64_t)l.lds};
  memcpy(dims, d, sizeof(d));
  return 1;
}
void trace_reset() { launches.clear(); }

}  // extern "C"
