// Test infrastructure: a stand-in for the HIP runtime calls that meep_amd's host code makes,
// so that the host code (planning, halo lists, source boxes, batch tables, kernel-argument
// validation) can be compiled with g++ and exercised on a machine without a GPU.  "Device"
// memory is host memory, streams, events and graphs do nothing, and the kernel launchers are
// empty stubs (tests/host_mock/build.py), so no field values are computed: the library built
// from it checks host logic only and is never loaded by the product.
#pragma once
#include <cstdlib>
#include <cstring>
#include <cstddef>
#include <cstdint>
typedef int hipError_t;
enum { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorNotReady = 600 };
typedef void *hipStream_t;
typedef void *hipEvent_t;
typedef void *hipGraph_t;
typedef void *hipGraphExec_t;
typedef void *hipGraphNode_t;
enum hipMemcpyKind { hipMemcpyHostToHost, hipMemcpyHostToDevice, hipMemcpyDeviceToHost, hipMemcpyDeviceToDevice, hipMemcpyDefault };
enum hipStreamCaptureMode { hipStreamCaptureModeGlobal, hipStreamCaptureModeThreadLocal, hipStreamCaptureModeRelaxed };
struct double2 { double x, y; };
struct float2 { float x, y; };
struct int2 { int x, y; };
inline double2 make_double2(double a, double b) { return {a, b}; }
inline float2 make_float2(float a, float b) { return {a, b}; }
// allocations that succeed before the next one fails (-1: none fails), and the calls made so far
inline long mock_mallocs_left = -1, mock_mallocs = 0;
inline hipError_t hipMalloc(void **p, size_t n) {
  ++mock_mallocs;
  if (mock_mallocs_left == 0) {
    mock_mallocs_left = -1;
    return hipErrorOutOfMemory;
  }
  if (mock_mallocs_left > 0) --mock_mallocs_left;
  *p = calloc(1, n ? n : 1);
  return hipSuccess;
}
// free and total device memory as hipMemGetInfo gives them
inline size_t mock_free = size_t(256) << 30, mock_total = size_t(288) << 30;
inline hipError_t hipMemGetInfo(size_t *f, size_t *t) { *f = mock_free, *t = mock_total; return hipSuccess; }
template <class T> inline hipError_t hipMalloc(T **p, size_t n) { return hipMalloc((void **)p, n); }
inline hipError_t hipFree(void *p) { free(p); return hipSuccess; }
inline hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { if (n) memmove(d, s, n); return hipSuccess; }
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t = 0) { return hipMemcpy(d, s, n, k); }
inline hipError_t hipMemset(void *d, int v, size_t n) { memset(d, v, n); return hipSuccess; }
inline hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t = 0) { memset(d, v, n); return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipStreamCreate(hipStream_t *s) { *s = (void *)1; return hipSuccess; }
inline hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
inline hipError_t hipEventCreate(hipEvent_t *e) { *e = (void *)1; return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t = 0) { return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 0; return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline const char *hipGetErrorString(hipError_t) { return "mock"; }
inline hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
inline hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
// a __device__ variable is an ordinary host variable here, and its "device address" its address
#define __device__
#define HIP_SYMBOL(x) (&(x))
#define __align__(n) __attribute__((aligned(n)))
template <class T> inline hipError_t hipGetSymbolAddress(void **p, const T *sym) { *p = (void *)sym; return hipSuccess; }
inline hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
inline hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { *g = (void *)1; return hipSuccess; }
inline hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) { *e = (void *)1; return hipSuccess; }
inline hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
inline hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
