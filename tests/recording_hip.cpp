// A stand-in for the HIP runtime calls the library makes, for tests on a host without a GPU: nothing is launched; what is kept is
// which kernels had their dynamic LDS limit raised and which were launched with more than the limit they had.
#include <hip/hip_runtime_api.h>

#include <cstring>
#include <map>

namespace {
std::map<const void*, size_t> limits;
int attributes = 0, launches = 0, over = 0;
dim3 grid_, block_;
size_t smem_;
hipStream_t stream_;
char image[64 << 10];
int record(const void* f, size_t smem) {
  const auto it = limits.find(f);
  ++launches;
  if (smem > (it == limits.end() ? size_t(48) << 10 : it->second)) ++over;
  return 0;
}
}  // namespace

extern "C" {
int recorded_attributes() { return attributes; }
int recorded_launches() { return launches; }
int recorded_over_limit() { return over; }

void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t st) { grid_ = g; block_ = b; smem_ = s; stream_ = st; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* s, hipStream_t* st) { *g = grid_; *b = block_; *s = smem_; *st = stream_; return hipSuccess; }
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void**, size_t smem, hipStream_t) { return hipError_t(record(f, smem)); }
hipError_t hipExtLaunchKernel(const void* f, dim3, dim3, void**, size_t smem, hipStream_t, hipEvent_t, hipEvent_t, int) { return hipError_t(record(f, smem)); }
hipError_t hipFuncSetAttribute(const void* f, hipFuncAttribute a, int v) {
  if (a == hipFuncAttributeMaxDynamicSharedMemorySize) limits[f] = size_t(v);
  ++attributes;
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) { *p = image; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stand-in"; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {  // the header's macro gives it the versioned name
  std::memset(p, 0, sizeof *p);
  std::strcpy(p->gcnArchName, "gfx950");
  return hipSuccess;
}
}
