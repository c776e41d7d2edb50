// A stand-in for the HIP runtime calls that the C entry points of librnnt_hip.so make, for tests
// without a device.  Loaded with RTLD_GLOBAL ahead of the library, so that the library binds to it.
// A launch of the length check is kept until its (device, stream) has been asked about `delay`
// times; only then does "the kernel" write its verdict.  Other kernels must be launched with
// `lose` set: nothing runs, and device pointers are never looked at.  The test sets the knobs below.
#include <stdint.h>
#include <stdlib.h>

#include <map>
#include <utility>
#include <vector>

struct dim3 {
  uint32_t x, y, z;
};

namespace {
struct Launch {
  const int *in, *lab;
  int B, T, U;
  int* word;
};
std::map<std::pair<int, void*>, std::vector<Launch>> waiting;

void run(std::vector<Launch>& launches) {
  for (const Launch& l : launches) {
    int bad = 0;
    for (int b = 0; b < l.B; ++b) bad |= (l.in[b] > l.T ? 1 : 0) | (l.lab[b] > l.U - 1 ? 2 : 0);
    __atomic_store_n(l.word, bad, __ATOMIC_RELEASE);
  }
  launches.clear();
}

struct Call {
  dim3 grid, block;
  size_t lds;
  void* stream;
} pushed;
}  // namespace

extern "C" {

int current_device = 0;
int delay = 0;          // questions a launch stays unfinished for
int asked = 0;          // hipStreamQuery calls
int launches = 0;       // kernels enqueued
int last_error = 0;     // what hipGetLastError reports next
int launch_error = 0;   // what hipLaunchKernel returns (and enqueues nothing)
int sync_error = 0;     // what hipStreamSynchronize returns
int query_error = 0;    // what hipStreamQuery returns instead of an answer
int capturing = 0;      // hipStreamCaptureStatus of every stream
int capture_error = 0;  // what hipStreamIsCapturing returns instead
int lose = 0;           // launches are accepted and never run
uint64_t pool_limit = UINT64_MAX;  // the largest allocation a memory pool grants
uint64_t pool_last = 0;            // the last one it granted

int hipGetDevice(int* d) { *d = current_device; return 0; }
int hipSetDevice(int d) { current_device = d; return 0; }
int hipHostMalloc(void** p, size_t n, unsigned) { *p = calloc(n, 1); return *p ? 0 : 2; }
int hipGetLastError() { const int e = last_error; last_error = 0; return e; }
int hipStreamIsCapturing(void*, int* status) {
  *status = capturing;
  return capture_error ? last_error = capture_error : 0;
}

int hipMemPoolCreate(void** pool, const void*) { *pool = &pool_limit; return 0; }
int hipMemPoolSetAttribute(void*, int, void*) { return 0; }
int hipMallocFromPoolAsync(void** p, size_t n, void*, void*) {
  if (n > pool_limit) return last_error = 2;  // hipErrorOutOfMemory
  pool_last = n;
  *p = reinterpret_cast<void*>(uintptr_t{1} << 40);
  return 0;
}
int hipFreeAsync(void*, void*) { return 0; }
int hipGetSymbolAddress(void** p, const void*) { *p = reinterpret_cast<void*>(uintptr_t{1} << 32); return 0; }
int hipFuncSetAttribute(const void*, int, int) { return 0; }

int __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, void* stream) {
  pushed = Call{grid, block, lds, stream};
  return 0;
}
int __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, void** stream) {
  *grid = pushed.grid; *block = pushed.block; *lds = pushed.lds; *stream = pushed.stream;
  return 0;
}
int hipLaunchKernel(const void*, dim3, dim3, void** args, size_t, void* stream) {
  if (launch_error) return last_error = launch_error;
  ++launches;
  if (lose) return 0;
  waiting[{current_device, stream}].push_back(
      Launch{*(const int**)args[0], *(const int**)args[1], *(int*)args[2], *(int*)args[3],
             *(int*)args[4], *(int**)args[5]});
  return 0;
}
int hipStreamQuery(void* stream) {
  ++asked;
  if (query_error) return last_error = query_error;
  auto& launches_here = waiting[{current_device, stream}];
  if (launches_here.empty()) return 0;
  if (delay-- > 0) return last_error = 600;  // hipErrorNotReady
  run(launches_here);
  return 0;
}
int hipStreamSynchronize(void* stream) {
  if (sync_error) return last_error = sync_error;
  run(waiting[{current_device, stream}]);
  return 0;
}
}
