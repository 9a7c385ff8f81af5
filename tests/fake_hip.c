/* The HIP runtime calls that libuaii_amd.so makes, on host memory: allocations against a
 * capacity, copies that copy, kernels that do nothing. For tests of what the host code
 * allocates, frees and launches; built and loaded by test_host_memory.py. */
#include <stddef.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

typedef struct { uint32_t x, y, z; } dim3;
typedef struct { void* p; size_t n; } block;

static block blocks[65536];
static size_t used, capacity = (size_t)-1, launches;
static char dummy[1 << 22];

void fake_capacity(size_t n) { capacity = n; }
size_t fake_used(void) { return used; }

int hipMalloc(void** p, size_t n) {
  if (used + n > capacity) return 2; /* hipErrorOutOfMemory */
  for (int i = 0; i < 65536; ++i) {
    if (blocks[i].p) continue;
    if (posix_memalign(&blocks[i].p, 256, n ? n : 1)) return 2;
    blocks[i].n = n;
    used += n;
    *p = blocks[i].p;
    return 0;
  }
  return 2;
}
int hipFree(void* p) {
  if (!p) return 0;
  for (int i = 0; i < 65536; ++i) {
    if (blocks[i].p != p) continue;
    used -= blocks[i].n;
    free(p);
    blocks[i].p = NULL;
    return 0;
  }
  abort(); /* not a live allocation */
}
int hipMemcpy(void* d, const void* s, size_t n, int k) { memcpy(d, s, n); return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int k, void* st) { memcpy(d, s, n); return 0; }
int hipMemset(void* d, int v, size_t n) { memset(d, v, n); return 0; }
int hipMemsetAsync(void* d, int v, size_t n, void* st) { memset(d, v, n); return 0; }
int hipLaunchKernel(const void* f, dim3 g, dim3 b, void** a, size_t sh, void* st) { ++launches; return 0; }
int hipExtLaunchKernel(const void* f, dim3 g, dim3 b, void** a, size_t sh, void* st, void* e0, void* e1, int fl) {
  ++launches;
  return 0;
}
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, void* st) { return 0; }
int __hipPopCallConfiguration(dim3* g, dim3* b, size_t* sh, void** st) {
  memset(g, 0, sizeof *g);
  memset(b, 0, sizeof *b);
  *sh = 0;
  *st = NULL;
  return 0;
}
void** __hipRegisterFatBinary(const void* d) { static void* h; return &h; }
void __hipRegisterFunction(void) {}
void __hipRegisterVar(void) {}
void __hipUnregisterFatBinary(void** h) {}
int hipGetDeviceCount(int* n) { *n = 1; return 0; }
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipSetDevice(int d) { return 0; }
/* CUs, or bytes of LDS */
int hipDeviceGetAttribute(int* v, int a, int d) { *v = a == FAKE_CU_ATTRIBUTE ? 256 : 160 * 1024; return 0; }
int hipDeviceSynchronize(void) { return 0; }
int hipFuncSetAttribute(const void* f, int a, int v) { return 0; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void* f, int b, size_t s) { *n = 2; return 0; }
int hipGetLastError(void) { return 0; }
const char* hipGetErrorString(int e) { return e == 2 ? "out of memory" : "error"; }
int hipGetSymbolAddress(void** p, const void* s) { *p = dummy; return 0; }
int hipPointerGetAttributes(void* a, const void* p) { return 1; }
int hipEventCreate(void** e) { *e = dummy; return 0; }
int hipEventCreateWithFlags(void** e, unsigned f) { *e = dummy; return 0; }
int hipEventDestroy(void* e) { return 0; }
int hipEventRecord(void* e, void* s) { return 0; }
int hipEventSynchronize(void* e) { return 0; }
int hipEventQuery(void* e) { return 0; }
int hipEventElapsedTime(float* ms, void* a, void* b) { *ms = 0; return 0; }
int hipStreamCreateWithFlags(void** s, unsigned f) { *s = dummy; return 0; }
int hipStreamDestroy(void* s) { return 0; }
int hipStreamSynchronize(void* s) { return 0; }
int hipStreamWaitEvent(void* s, void* e, unsigned f) { return 0; }
int hipStreamIsCapturing(void* s, int* c) { *c = 0; return 0; }
int hipStreamBeginCapture(void* s, int m) { return 0; }
int hipStreamEndCapture(void* s, void** g) { *g = dummy; return 0; }
int hipThreadExchangeStreamCaptureMode(int* m) { return 0; }
int hipGraphInstantiate(void** x, void* g, void* n, char* b, size_t s) { *x = dummy; return 0; }
int hipGraphLaunch(void* x, void* s) { return 0; }
int hipGraphDestroy(void* g) { return 0; }
int hipGraphExecDestroy(void* x) { return 0; }
