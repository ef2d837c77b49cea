// hip_runtime.h -- the HIP names that csrc/ uses, for a CPU build in which
// host_exec.cpp runs every block of a launch in turn (bounds checks without a
// GPU). Test code only.
#pragma once

#include <math.h>
#include <stddef.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#include <functional>
#include <utility>

#define __global__
#define __device__
#define __host__
#define __shared__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __align__(n) __attribute__((aligned(n)))
#define amdgpu_waves_per_eu(...) noinline

struct dim3 {
  unsigned x, y, z;
  dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {}
};
struct SimIdx {
  unsigned x;
};
extern SimIdx threadIdx, blockIdx, blockDim, gridDim;

__attribute__((convergent, noduplicate)) void sim_block_barrier();
__attribute__((convergent, noduplicate)) void sim_wave_barrier();
// v of lane `src` of this wave, all of whose lanes make the call
__attribute__((convergent, noduplicate)) int sim_lane(int v, int src);
[[noreturn]] void sim_unsupported(const char *what);
void sim_launch(const char *name, dim3 grid, dim3 block, size_t lds,
                const std::function<void()> &body);
#define hipLaunchKernelGGL(K, grid, block, lds, stream, ...) \
  sim_launch(__PRETTY_FUNCTION__, grid, block, lds, [=] { K(__VA_ARGS__); })

#define __syncthreads() sim_block_barrier()
#define __builtin_amdgcn_fence(...) ((void)0)
#define __builtin_amdgcn_wave_barrier() sim_wave_barrier()
inline int __lane_id() { return (int)(threadIdx.x & 63); }
inline uint32_t __umulhi(uint32_t a, uint32_t b) { return (uint32_t)(((uint64_t)a * b) >> 32); }
inline float __uint_as_float(uint32_t u) { return __builtin_bit_cast(float, u); }

// cross-lane operations, in the forms that kernels_xlane.hpp uses
inline int sim_dpp(int x, int ctrl) {
  const int l = __lane_id();
  if (ctrl < 0x100) return sim_lane(x, (l & ~3) | ((ctrl >> (2 * (l & 3))) & 3));      // quad_perm
  if (ctrl > 0x120 && ctrl < 0x130) return sim_lane(x, (l & ~15) | ((l - ctrl) & 15));  // row_ror
  sim_unsupported("dpp control");
}
#define __builtin_amdgcn_update_dpp(old, x, ctrl, rm, bm, bc) sim_dpp(x, ctrl)
inline int sim_swizzle(int x, int off) {  // bit-mask mode
  const int l = __lane_id();
  return sim_lane(x, (l & 32) | ((((l & 31) & (off & 31)) | ((off >> 5) & 31)) ^ ((off >> 10) & 31)));
}
#define __builtin_amdgcn_ds_swizzle(x, off) sim_swizzle(x, off)
struct SimPair {
  unsigned v[2];
  unsigned operator[](int i) const { return v[i]; }
};
inline SimPair sim_permlane32_swap(unsigned a, unsigned b) {
  const int l = __lane_id();
  const unsigned pa = (unsigned)sim_lane((int)a, l ^ 32), pb = (unsigned)sim_lane((int)b, l ^ 32);
  return l < 32 ? SimPair{{a, pa}} : SimPair{{pb, b}};
}
#define __builtin_amdgcn_permlane32_swap(a, b, fi, bc) sim_permlane32_swap(a, b)
template <class A, class B, class D>
D sim_mfma(A, B, D) {
  sim_unsupported("matrix instruction");
}
#define __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, d, x, y, z) sim_mfma(a, b, d)
template <class V>
int sim_sdot2(V a, V b, int c) {
  return (int)((unsigned)c + (unsigned)(a[0] * b[0]) + (unsigned)(a[1] * b[1]));
}
#define __builtin_amdgcn_sdot2(a, b, c, clamp) sim_sdot2(a, b, c)

typedef int hipError_t;
typedef struct SimStream *hipStream_t;
typedef struct SimEvent *hipEvent_t;
enum : int {
  hipSuccess = 0,
  hipErrorInvalidValue = 1,
  hipErrorInvalidDevice = 101,
  hipErrorInvalidSymbol = 13,
};
enum { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
enum { hipDeviceAttributeMultiprocessorCount };
enum { hipFuncAttributeMaxDynamicSharedMemorySize };
enum { hipStreamNonBlocking };
enum { hipMemoryTypeDevice, hipMemoryTypeManaged };
struct hipPointerAttribute_t {
  int type;
};
struct hipDeviceProp_t {
  char gcnArchName[256];
  int multiProcessorCount;
};
#define HIP_SYMBOL(s) ((const void *)(s))

extern int sim_cus;  // compute units that the planner sees
hipError_t sim_malloc(void **p, size_t bytes);
template <class T>
hipError_t hipMalloc(T **p, size_t bytes) {
  return sim_malloc(reinterpret_cast<void **>(p), bytes);
}
hipError_t hipFree(void *p);
inline hipError_t hipMemcpy(void *d, const void *s, size_t n, int) {
  memcpy(d, s, n);
  return hipSuccess;
}
inline hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
  memset(d, v, n);
  return hipSuccess;
}
inline const char *hipGetErrorString(hipError_t) { return "error"; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
inline hipError_t hipDeviceGetAttribute(int *v, int, int) { return *v = sim_cus, hipSuccess; }
inline hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) {
  memset(p, 0, sizeof(*p));
  p->multiProcessorCount = sim_cus;
  return hipSuccess;
}
inline hipError_t hipFuncSetAttribute(const void *, int, int) { return hipSuccess; }
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *) {
  return a->type = hipMemoryTypeDevice, hipSuccess;
}
inline hipError_t hipGetSymbolAddress(void **p, const void *s) {
  return *p = const_cast<void *>(s), hipSuccess;
}
template <class K>
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, K, int, size_t) {
  return *n = 2, hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return *s = nullptr, hipSuccess; }
inline hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
inline hipError_t hipEventCreate(hipEvent_t *) { return hipErrorInvalidValue; }  // no timing
inline hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipErrorInvalidValue; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipErrorInvalidValue; }
inline hipError_t hipEventElapsedTime(float *, hipEvent_t, hipEvent_t) { return hipErrorInvalidValue; }
