/* The HIP calls that the library makes, answered on the CPU for tests of its host side (preloaded): allocations are host
 * memory, copies are memcpy, launches and waits do nothing. Calls are counted. */
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>
#include <stdlib.h>
#include <string.h>

long counts[5];      /* launches, allocations, copies, waits, frees */
void *copy_dst;      /* the last copy */
size_t copy_bytes;
long shapes[64][4];  /* launch i: grid x and y, block x, dynamic LDS bytes (modulo 64 launches) */

static hipError_t get(void **p, size_t n) { counts[1]++; *p = malloc(n ? n : 1); return *p ? hipSuccess : hipErrorOutOfMemory; }
static hipError_t copy(void *d, const void *s, size_t n) { counts[2]++; copy_dst = d; copy_bytes = n; memcpy(d, s, n); return hipSuccess; }

hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int d) {
    (void)d;
    memset(p, 0, sizeof *p);
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int d) {
    (void)d;
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 1;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *s) {
    static void *mem;
    (void)s;
    if (!mem) mem = malloc(32u << 20);
    *p = mem;
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) { return get(p, n); }
hipError_t hipMallocAsync(void **p, size_t n, hipStream_t s) { (void)s; return get(p, n); }
hipError_t hipFree(void *p) { counts[4]++; free(p); return hipSuccess; }
hipError_t hipFreeAsync(void *p, hipStream_t s) { (void)s; counts[4]++; free(p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned f) { (void)f; *p = malloc(n); return hipSuccess; }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) { (void)k; return copy(d, s, n); }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st) { (void)k; (void)st; return copy(d, s, n); }
hipError_t hipMemset(void *d, int v, size_t n) { memset(d, v, n); return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { counts[3]++; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { (void)s; counts[3]++; return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *c) { (void)s; *c = hipStreamCaptureStatusNone; return hipSuccess; }
hipError_t hipFuncSetAttribute(const void *f, hipFuncAttribute a, int v) { (void)f; (void)a; (void)v; return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t l, hipStream_t s) {
    long *r = shapes[counts[0] % 64];
    (void)s;
    r[0] = g.x;
    r[1] = g.y;
    r[2] = b.x;
    r[3] = (long)l;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *l, hipStream_t *s) {
    g->x = g->y = g->z = b->x = b->y = b->z = 1;
    *l = 0;
    *s = 0;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **a, size_t l, hipStream_t s) {
    (void)f; (void)g; (void)b; (void)a; (void)l; (void)s;
    counts[0]++;
    return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
