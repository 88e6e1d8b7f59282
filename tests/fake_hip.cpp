// A HIP runtime without a device: memory is the host's, kernels do nothing and
// are written down by name, the device has FAKE_HIP_CUS compute units.  Loaded
// with its symbols global before libekpnp.so, it shows on the CPU which kernels
// a context of given channels launches.
#include <cxxabi.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
struct Dim3 { unsigned x, y, z; };
struct Call { Dim3 grid, block; size_t lds; void* stream; } call;
std::map<const void*, std::string>& names() {
  static std::map<const void*, std::string> m;
  return m;
}
std::string log_text;
int handle;
}  // namespace

extern "C" {

// kernels launched since the last call, one "name grid_x" a line
const char* fake_hip_launches() {
  static std::string out;
  out.swap(log_text);
  log_text.clear();
  return out.c_str();
}

void** __hipRegisterFatBinary(const void*) { return reinterpret_cast<void**>(&handle); }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* device, unsigned, void*, void*, void*, void*,
                           int*) {
  int status = 0;
  char* d = abi::__cxa_demangle(device, nullptr, nullptr, &status);
  std::string s = status == 0 ? d : device;
  std::free(d);
  // "void ekpnp::k_lbm<float, ...>(args)" without the type, namespace and arguments
  if (s.compare(0, 5, "void ") == 0) s.erase(0, 5);
  if (s.compare(0, 7, "ekpnp::") == 0) s.erase(0, 7);
  s.erase(std::min(s.find('('), s.size()));
  names()[host] = s;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t lds, void* stream) {
  call = {grid, block, lds, stream};
  return 0;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* lds, void** stream) {
  *grid = call.grid;
  *block = call.block;
  *lds = call.lds;
  *stream = call.stream;
  return 0;
}
int hipLaunchKernel(const void* f, Dim3 grid, Dim3, void**, size_t, void*) {
  log_text += names()[f] + " " + std::to_string(grid.x) + "\n";
  return 0;
}

int hipDeviceGetAttribute(int* v, int attribute, int) {
  const char* cus = std::getenv("FAKE_HIP_CUS");
  *v = attribute == 63 ? (cus ? std::atoi(cus) : 256) : 163840;  // 63: compute units; else LDS bytes
  return 0;
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  *n = 4;
  return 0;
}
int hipGetSymbolAddress(void** p, const void*) {
  static double scratch[1 << 16];
  *p = scratch;
  return 0;
}
int hipMalloc(void** p, size_t n) { return (*p = std::calloc(n ? n : 1, 1)) ? 0 : 2; }
int hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
int hipFree(void* p) {
  std::free(p);
  return 0;
}
int hipHostFree(void* p) { return hipFree(p); }
int hipMemcpy(void* d, const void* s, size_t n, int) {
  std::memcpy(d, s, n);
  return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int k, void*) { return hipMemcpy(d, s, n, k); }
int hipMemset(void*, int, size_t) { return 0; }  // fresh memory is zero
int hipMemsetAsync(void*, int, size_t, void*) { return 0; }
int hipStreamCreateWithFlags(void** s, unsigned) {
  *s = &handle;
  return 0;
}
int hipEventCreateWithFlags(void** e, unsigned) {
  *e = &handle;
  return 0;
}
int hipPointerGetAttributes(void*, const void*) { return 1; }
int hipSetDevice(int) { return 0; }
int hipGetDevice(int* d) { return *d = 0; }
int hipGetLastError() { return 0; }
const char* hipGetErrorString(int) { return "fake HIP"; }
int hipDeviceSynchronize() { return 0; }
int hipStreamSynchronize(void*) { return 0; }
int hipStreamQuery(void*) { return 0; }
int hipStreamDestroy(void*) { return 0; }
int hipEventDestroy(void*) { return 0; }
int hipEventRecord(void*, void*) { return 0; }
int hipEventSynchronize(void*) { return 0; }

}  // extern "C"
