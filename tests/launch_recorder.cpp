// Stand-in for the HIP runtime's host entry points that libcmpext3_attn.so
// calls (no GPU, nothing runs): every launch is recorded as (calling thread's
// tag, kernel name, workgroups, threads), so that tests can see which launches
// a call makes, and in which order those of several threads reach a stream.
// Loaded with RTLD_GLOBAL before the library, whose references then bind here.
#include <unistd.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {

struct Dim3 {
  uint32_t x, y, z;
};
struct Launch {
  int tag;
  const char* name;
  uint64_t workgroups, threads;
};

std::mutex mu;
std::vector<Launch> launches;
std::string slow_kernel;
int slow_us = 0;
std::map<const void*, std::string>& names() {
  static std::map<const void*, std::string> n;  // filled by the library's constructors
  return n;
}
thread_local int my_tag = 0;
thread_local Dim3 cfg_grid, cfg_block;
thread_local size_t cfg_shared;
thread_local void* cfg_stream;
alignas(256) char symbol_space[256];  // stands for a device variable: addressed, never read

}  // namespace

extern "C" {

// ---- used by the tests
void recorder_tag(int tag) { my_tag = tag; }
void recorder_clear() {
  std::lock_guard<std::mutex> l(mu);
  launches.clear();
}
int recorder_count() {
  std::lock_guard<std::mutex> l(mu);
  return (int)launches.size();
}
int recorder_get(int i, const char** name, uint64_t* workgroups, uint64_t* threads) {
  std::lock_guard<std::mutex> l(mu);
  *name = launches[i].name;
  *workgroups = launches[i].workgroups;
  *threads = launches[i].threads;
  return launches[i].tag;
}
// every launch of a kernel whose name contains `part` takes this long to return
void recorder_slow(const char* part, int us) {
  std::lock_guard<std::mutex> l(mu);
  slow_kernel = part;
  slow_us = us;
}

// ---- the runtime's side
void** __hipRegisterFatBinary(const void*) {
  static void* handle = nullptr;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* device, unsigned, void*, void*, void*, void*, int*) {
  names()[host] = device;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t shared, void* stream) {
  cfg_grid = grid;
  cfg_block = block;
  cfg_shared = shared;
  cfg_stream = stream;
  return 0;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* shared, void** stream) {
  *grid = cfg_grid;
  *block = cfg_block;
  *shared = cfg_shared;
  *stream = cfg_stream;
  return 0;
}
int hipLaunchKernel(const void* host, Dim3 grid, Dim3 block, void**, size_t, void*) {
  int us = 0;
  {
    std::lock_guard<std::mutex> l(mu);
    const auto it = names().find(host);
    const char* name = it == names().end() ? "?" : it->second.c_str();
    const uint64_t n = (uint64_t)grid.x * grid.y * grid.z;
    launches.push_back({my_tag, name, n, n * block.x * block.y * block.z});
    if (slow_us > 0 && strstr(name, slow_kernel.c_str())) us = slow_us;
  }
  if (us > 0) usleep(us);
  return 0;
}
int hipGetLastError() { return 0; }
int hipGetDevice(int* dev) {
  *dev = 0;
  return 0;
}
int hipDeviceGetAttribute(int* value, int, int) {
  *value = 256;
  return 0;
}
int hipGetSymbolAddress(void** ptr, const void*) {
  *ptr = symbol_space;
  return 0;
}

}  // extern "C"
