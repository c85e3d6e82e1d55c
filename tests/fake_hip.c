/* The HIP runtime functions the library calls, on host memory: allocations are
 * calloc, copies are memcpy, kernel launches do nothing. For tests of what the
 * host code does when an allocation fails. */
#include <stdlib.h>
#include <string.h>

static long live, fail_after = -1, streams;
static size_t bytes_live, bytes_limit;

long fake_live(void) { return live; }
/* streams created so far */
long fake_streams(void) { return streams; }
size_t fake_bytes(void) { return bytes_live; }
/* the allocation after the next n fails, once (n < 0: none) */
void fake_fail_after(long n) { fail_after = n; }
/* allocations that would exceed `bytes` in all fail (0: no limit) */
void fake_limit(size_t bytes) { bytes_limit = bytes; }

int hipMalloc(void** p, size_t n) {
  *p = 0;
  if (bytes_limit && bytes_live + n > bytes_limit) return 2; /* hipErrorOutOfMemory */
  if (fail_after >= 0 && fail_after-- == 0) return 2;
  size_t* q = calloc(n + 64, 1);
  q[0] = n;
  live++;
  bytes_live += n;
  *p = (char*)q + 64;
  return 0;
}
int hipFree(void* p) {
  if (p) {
    size_t* q = (size_t*)((char*)p - 64);
    live--;
    bytes_live -= q[0];
    free(q);
  }
  return 0;
}
int hipHostMalloc(void** p, size_t n, unsigned f) { return (*p = calloc(n, 1)) == 0; }
int hipHostFree(void* p) { free(p); return 0; }
int hipMemcpy(void* d, const void* s, size_t n, int k) { memcpy(d, s, n); return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int k, void* st) { memcpy(d, s, n); return 0; }
int hipMemset(void* d, int v, size_t n) { memset(d, v, n); return 0; }
int hipMemsetAsync(void* d, int v, size_t n, void* st) { memset(d, v, n); return 0; }
static int handle(void** p) { *p = (void*)1; return 0; }
int hipEventCreate(void** e) { return handle(e); }
int hipEventCreateWithFlags(void** e, unsigned f) { return handle(e); }
int hipStreamCreateWithFlags(void** s, unsigned f) { streams++; return handle(s); }
int hipEventDestroy(void* e) { return 0; }
int hipEventElapsedTime(float* ms, void* a, void* b) { *ms = 0; return 0; }
int hipEventRecord(void* e, void* s) { return 0; }
int hipEventSynchronize(void* e) { return 0; }
int hipStreamDestroy(void* s) { return 0; }
int hipStreamSynchronize(void* s) { return 0; }
int hipStreamWaitEvent(void* s, void* e, unsigned f) { return 0; }
int hipDeviceSynchronize(void) { return 0; }
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipGetDeviceCount(int* n) { *n = 1; return 0; }
int hipDeviceGetAttribute(int* v, int a, int d) { *v = 0; return 0; }
int hipGetDevicePropertiesR0600(void* p, int d) { memset(p, 0, 1024); return 0; }
int hipGetStreamDeviceId(void* s) { return 0; }
int hipGetLastError(void) { return 0; }
const char* hipGetErrorString(int e) { return e == 2 ? "out of memory" : "error"; }
int hipFuncSetAttribute(const void* f, int a, int v) { return 0; }
int hipGetSymbolAddress(void** p, const void* s) { *p = 0; return 1; }
int hipLaunchKernel(const void* f, long gx, int gz, long bx, int bz, void** a, size_t sh, void* s) { return 0; }
int hipExtLaunchKernel(const void* f, long gx, int gz, long bx, int bz, void** a, size_t sh, void* s, void* e0, void* e1,
                       int fl) { return 0; }
int __hipPushCallConfiguration(long gx, int gz, long bx, int bz, size_t sh, void* s) { return 0; }
int __hipPopCallConfiguration(void* g, void* b, size_t* sh, void** s) { *sh = 0; *s = 0; return 0; }
void** __hipRegisterFatBinary(const void* d) { static void* h; return &h; }
void __hipRegisterFunction(void) {}
void __hipRegisterVar(void) {}
void __hipUnregisterFatBinary(void** h) {}
