/* Stand-in for the HIP runtime in host-only tests: the declarations that the
 * headers under test use.  Streams, copies and kernels are the test's own. */
#pragma once

#include <math.h>
#include <stddef.h>
#include <stdint.h>
#include <string.h>

#define __device__
#define __host__
#define __forceinline__ inline

struct float2 { float x, y; };
struct float4 { float x, y, z, w; };
struct int4 { int32_t x, y, z, w; };
inline uint32_t __float_as_uint(float v) { uint32_t u; memcpy(&u, &v, 4); return u; }
inline float __uint_as_float(uint32_t u) { float v; memcpy(&v, &u, 4); return v; }
inline uint32_t min(uint32_t a, uint32_t b) { return b < a ? b : a; }
inline uint32_t max(uint32_t a, uint32_t b) { return b > a ? b : a; }

typedef enum { hipSuccess = 0, hipErrorNotReady = 600, hipErrorUnknown = 999 } hipError_t;
typedef struct test_stream* hipStream_t;
typedef struct test_event* hipEvent_t;
enum { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
enum { hipHostMallocCoherent = 0x40000000 };
enum { hipEventDisableTiming = 2 };

hipError_t hipMalloc(void** p, size_t bytes);
hipError_t hipFree(void* p);
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned flags);
hipError_t hipHostFree(void* p);
hipError_t hipMemcpy(void* dst, const void* src, size_t bytes, int kind);
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, int kind, hipStream_t s);
hipError_t hipStreamSynchronize(hipStream_t s);
hipError_t hipStreamQuery(hipStream_t s);
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned flags);
hipError_t hipEventDestroy(hipEvent_t e);
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s);
hipError_t hipEventSynchronize(hipEvent_t e);
hipError_t hipEventQuery(hipEvent_t e);
hipError_t hipGetLastError();
