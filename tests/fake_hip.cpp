// A HIP runtime without a device, for tests of what the library does on the host: which kernels it launches, and what
// becomes of a launch that is refused.  Memory is the host's, streams finish at once, and of the kernels only those
// that move bytes and clear error records do anything.  An event's time is the number of launches and asynchronous copies before it, in ms.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
std::map<const void *, std::string> kernels;   // by their host side
std::map<const void *, size_t> variables;
std::map<const void *, void *> addresses;
std::string launched, refused;
hipError_t standing = hipSuccess;
size_t work = 0;

struct Call {
  dim3 grid, block;
  size_t shared;
  hipStream_t stream;
} pushed;

hipError_t fails(hipError_t code) { return standing = code; }

template <typename Piece>
void move(void **args) {
  memcpy(*(void **)args[1], *(void **)args[0], *(uint32_t *)args[2] * sizeof(Piece));
}
}  // namespace

extern "C" {

// ---- what a test sees and sets
const char *fake_launched() { return launched.c_str(); }   // names of the launched kernels, one to a line
void fake_forget() { launched.clear(); }
void fake_refuse(const char *part) { refused = part; }      // kernels whose name holds it (empty: none)
void fake_fail() { standing = hipErrorOutOfMemory; }        // what a failed call elsewhere in the program leaves
int fake_standing() { return standing; }

// ---- the runtime
void **__hipRegisterFatBinary(const void *) {
  static void *module;
  return &module;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned int, void *, void *, dim3 *,
                           dim3 *, int *) {
  kernels[host] = name;
}
void __hipRegisterVar(void **, void *host, char *, char *, int, size_t size, int, int) { variables[host] = size; }
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) {
  pushed = Call{grid, block, shared, stream};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, hipStream_t *stream) {
  *grid = pushed.grid, *block = pushed.block, *shared = pushed.shared, *stream = pushed.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *host, dim3 grid, dim3, void **args, size_t, hipStream_t) {
  const std::string &name = kernels[host];
  if (grid.x == 0 || grid.y == 0 || grid.z == 0) return fails(hipErrorInvalidConfiguration);
  if (!refused.empty() && name.find(refused) != std::string::npos) return fails(hipErrorLaunchFailure);
  launched += name + "\n";
  ++work;
  if (name.find("move_bytes_kernelIh") != std::string::npos) move<uint8_t>(args);
  else if (name.find("move_bytes_kernelIj") != std::string::npos) move<uint32_t>(args);
  else if (name.find("move_bytes_kernel") != std::string::npos) move<uint32_t[4]>(args);
  else if (name.find("init_errors_kernel") != std::string::npos) memset(*(void **)args[0], 0, *(uint32_t *)args[1] * 8);   // {flag, value}
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t code = standing;
  standing = hipSuccess;
  return code;
}
hipError_t hipMalloc(void **ptr, size_t bytes) {
  bytes = (bytes + 255) / 256 * 256;
  *ptr = aligned_alloc(256, bytes);
  return *ptr ? memset(*ptr, 0, bytes), hipSuccess : fails(hipErrorOutOfMemory);
}
hipError_t hipFree(void *ptr) { return free(ptr), hipSuccess; }
hipError_t hipHostMalloc(void **ptr, size_t bytes, unsigned int) { return hipMalloc(ptr, bytes); }
hipError_t hipHostFree(void *ptr) { return free(ptr), hipSuccess; }
hipError_t hipMemcpy(void *to, const void *from, size_t bytes, hipMemcpyKind) { return memcpy(to, from, bytes), hipSuccess; }
hipError_t hipMemcpyAsync(void *to, const void *from, size_t bytes, hipMemcpyKind, hipStream_t) {
  ++work;
  return memcpy(to, from, bytes), hipSuccess;
}
hipError_t hipMemsetAsync(void *to, int value, size_t bytes, hipStream_t) { return memset(to, value, bytes), hipSuccess; }
hipError_t hipGetSymbolAddress(void **ptr, const void *symbol) {
  void *&at = addresses[symbol];
  if (!at) at = calloc(1, variables[symbol]);
  *ptr = at;
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *event) { return *event = (hipEvent_t)calloc(1, sizeof(size_t)), hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t event) { return free(event), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t event, hipStream_t) { return *(size_t *)event = work, hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t from, hipEvent_t to) {
  *ms = (float)(*(size_t *)to - *(size_t *)from);
  return hipSuccess;
}
hipError_t hipStreamCreate(hipStream_t *stream) { return *stream = (hipStream_t)&pushed, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int *count) { return *count = 1, hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *props, int) {   // (a macro names the version of the call)
  memset(props, 0, sizeof(*props));
  strcpy(props->gcnArchName, "gfx950");
  props->totalGlobalMem = 288ull << 30;
  props->sharedMemPerBlock = 160 << 10;
  props->multiProcessorCount = 256;
  props->warpSize = 64;
  return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *blocks, const void *, int, size_t) { return *blocks = 2, hipSuccess; }
}
