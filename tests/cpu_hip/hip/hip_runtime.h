// Stand-in for the HIP runtime on the CPU: kernels run one workgroup at a time
// with a fiber per thread (runtime.cpp), and every allocation lies against
// pages that fault.  Streams are in order by construction; a graph launch does
// nothing more (its capture has run the calls).
#pragma once
#include <algorithm>
#include <climits>
#include <cmath>
#include <cstddef>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <vector>
using std::fabs;
using std::isfinite;
using std::isnan;
using std::pow;
using std::sqrt;
inline int min(int a, int b) { return b < a ? b : a; }
inline int max(int a, int b) { return a < b ? b : a; }
inline int64_t min(int64_t a, int64_t b) { return b < a ? b : a; }
#define amdgpu_waves_per_eu(...) unused
#define __host__
#define __device__
#define __global__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __shared__ static
#define __align__(x) __attribute__((aligned(x)))
#define HIP_SYMBOL(x) (&(x))

struct dim3 {
  unsigned x, y, z;
  dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {}
};
namespace cpu_hip {
struct Index {
  unsigned x, y, z;
};
extern Index tid, bid;
extern dim3 grid, block;
void barrier();
// the value that lane src(lane, arg) of the wave passes in the same operation
uint64_t exchange(uint64_t v, int (*src)(int lane, int arg), int arg, bool* valid);
void launch(const char* name, dim3 g, dim3 b, const std::function<void()>& f);
}  // namespace cpu_hip
#define threadIdx cpu_hip::tid
#define blockIdx cpu_hip::bid
#define gridDim cpu_hip::grid
#define blockDim cpu_hip::block
#define __syncthreads() cpu_hip::barrier()
#define hipLaunchKernelGGL(K, G, B, S, ST, ...) cpu_hip::launch(#K, dim3(G), dim3(B), [&] { (K)(__VA_ARGS__); })

#define __builtin_amdgcn_readfirstlane(x) (x)
#define __builtin_amdgcn_sched_barrier(x) ((void)0)
#define __builtin_amdgcn_rcp(x) (1.0 / (x))
inline uint64_t double_bits(double d) {
  uint64_t b;
  memcpy(&b, &d, 8);
  return b;
}
inline double bits_double(uint64_t b) {
  double d;
  memcpy(&d, &b, 8);
  return d;
}
inline int __double2loint(double d) { return int(uint32_t(double_bits(d))); }
inline int __double2hiint(double d) { return int(uint32_t(double_bits(d) >> 32)); }
inline double __hiloint2double(int h, int l) { return bits_double((uint64_t(uint32_t(h)) << 32) | uint32_t(l)); }
// quad permutations, row shifts and row rotations
inline int dpp_source(int lane, int ctrl) {
  const int row = lane & ~15, i = lane & 15;
  int j;
  if (ctrl < 0x100) {
    j = (i & ~3) | ((ctrl >> (2 * (i & 3))) & 3);
  } else if (ctrl >= 0x101 && ctrl <= 0x10f) {
    j = i + (ctrl - 0x100);
    if (j > 15) return -1;
  } else if (ctrl >= 0x111 && ctrl <= 0x11f) {
    j = i - (ctrl - 0x110);
    if (j < 0) return -1;
  } else if (ctrl >= 0x121 && ctrl <= 0x12f) {
    j = (i - (ctrl - 0x120) + 16) & 15;
  } else {
    abort();
  }
  return row | j;
}
inline int update_dpp(int old, int src, int ctrl) {
  bool ok;
  const uint64_t r = cpu_hip::exchange(uint32_t(src), dpp_source, ctrl, &ok);
  return ok ? int(uint32_t(r)) : old;
}
#define __builtin_amdgcn_update_dpp(o, s, c, rm, bm, b) update_dpp(o, s, c)
inline int xor_source(int lane, int d) { return lane ^ d; }
inline double __shfl_xor(double v, int d) {
  bool ok;
  const uint64_t r = cpu_hip::exchange(double_bits(v), xor_source, d, &ok);
  return ok ? bits_double(r) : v;
}
inline int atomicMin(int* p, int v) {
  const int o = *p;
  if (v < o) *p = v;
  return o;
}

typedef int hipError_t;
enum {
  hipSuccess = 0,
  hipErrorInvalidValue = 1,
  hipErrorOutOfMemory = 2,
  hipErrorNotInitialized = 3,
  hipErrorNotSupported = 801
};
typedef struct hipStreamImpl* hipStream_t;
typedef struct hipEventImpl* hipEvent_t;
typedef struct hipGraphImpl* hipGraph_t;
typedef struct hipGraphExecImpl* hipGraphExec_t;
typedef struct hipModImpl* hipModule_t;
typedef struct hipFuncImpl* hipFunction_t;
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost, hipMemcpyDeviceToDevice, hipMemcpyDefault };
enum hipStreamCaptureMode { hipStreamCaptureModeGlobal, hipStreamCaptureModeThreadLocal, hipStreamCaptureModeRelaxed };
enum { hipStreamNonBlocking = 1, hipEventDisableTiming = 2 };
struct hipDeviceProp_t {
  char name[64];
  char gcnArchName[64];
  int multiProcessorCount;
  size_t totalGlobalMem;
};
extern "C" {
hipError_t cpu_hip_malloc(void**, size_t);
hipError_t cpu_hip_free(void*);
}
template <class T>
hipError_t hipMalloc(T** p, size_t n) {
  return cpu_hip_malloc((void**)p, n);
}
template <class T>
hipError_t hipHostMalloc(T** p, size_t n, unsigned = 0) {
  return cpu_hip_malloc((void**)p, n);
}
inline hipError_t hipFree(void* p) { return cpu_hip_free(p); }
inline hipError_t hipHostFree(void* p) { return cpu_hip_free(p); }
inline hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) {
  *d = h;
  return 0;
}
inline hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  memcpy(d, s, n);
  return 0;
}
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t = nullptr) {
  memcpy(d, s, n);
  return 0;
}
inline hipError_t hipMemset(void* d, int v, size_t n) {
  memset(d, v, n);
  return 0;
}
inline hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
  memset(d, v, n);
  return 0;
}
inline hipError_t hipGetLastError() { return 0; }
inline const char* hipGetErrorString(hipError_t) { return "cpu_hip"; }
inline hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return 0;
}
inline hipError_t hipSetDevice(int) { return 0; }
inline hipError_t hipGetDevice(int* d) {
  *d = 0;
  return 0;
}
inline hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
  memset(p, 0, sizeof *p);
  strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  return 0;
}
template <class H>
hipError_t some_handle(H* h) {
  *h = (H)1;
  return 0;
}
inline hipError_t hipStreamCreate(hipStream_t* s) { return some_handle(s); }
inline hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return some_handle(s); }
inline hipError_t hipStreamDestroy(hipStream_t) { return 0; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return 0; }
inline hipError_t hipDeviceSynchronize() { return 0; }
inline hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return 0; }
inline hipError_t hipEventCreate(hipEvent_t* e) { return some_handle(e); }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return some_handle(e); }
inline hipError_t hipEventDestroy(hipEvent_t) { return 0; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t = nullptr) { return 0; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return 0; }
inline hipError_t hipEventElapsedTime(float* f, hipEvent_t, hipEvent_t) {
  *f = 1.0f;
  return 0;
}
inline hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return 0; }
inline hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { return some_handle(g); }
inline hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, void*, void*, size_t) { return some_handle(e); }
inline hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return 0; }
inline hipError_t hipGraphDestroy(hipGraph_t) { return 0; }
inline hipError_t hipGraphExecDestroy(hipGraphExec_t) { return 0; }
inline hipError_t hipModuleUnload(hipModule_t) { return 0; }
inline hipError_t hipModuleLaunchKernel(hipFunction_t, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned,
                                        unsigned, hipStream_t, void**, void**) {
  return hipErrorNotSupported;
}
inline hipError_t hipGetSymbolAddress(void** p, const void* s) {
  *p = (void*)s;
  return 0;
}
