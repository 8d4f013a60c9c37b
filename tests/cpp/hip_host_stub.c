/* A HIP runtime of two devices without any: "device" memory is host memory, kernels do nothing.  It counts
 * what is allocated while each device is current, and the launches. */
#include <stdlib.h>
#include <string.h>

static int current, allocs[2], launches;
int stub_allocs(int dev) { return allocs[dev]; }
int stub_launches(void) { return launches; }

#define NOTE allocs[current]++
int hipGetDeviceCount(int* n) { *n = 2; return 0; }
int hipGetDevice(int* d) { *d = current; return 0; }
int hipSetDevice(int d) { current = d; return 0; }
int hipDeviceGetAttribute(int* v, int attr, int dev) { (void)attr; (void)dev; *v = 256; return 0; }
int hipMalloc(void** p, size_t n) { NOTE; *p = calloc(1, n ? n : 1); return 0; }
int hipHostMalloc(void** p, size_t n, unsigned f) { (void)f; NOTE; *p = calloc(1, n ? n : 1); return 0; }
int hipFree(void* p) { free(p); return 0; }
int hipHostFree(void* p) { free(p); return 0; }
int hipMemcpy(void* d, const void* s, size_t n, int k) { (void)k; memcpy(d, s, n); return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int k, void* st) { (void)k; (void)st; memcpy(d, s, n); return 0; }
int hipMemset(void* d, int v, size_t n) { memset(d, v, n); return 0; }
int hipMemsetAsync(void* d, int v, size_t n, void* st) { (void)st; memset(d, v, n); return 0; }
int hipEventCreate(void** e) { NOTE; *e = malloc(1); return 0; }
int hipEventCreateWithFlags(void** e, unsigned f) { (void)f; NOTE; *e = malloc(1); return 0; }
int hipEventDestroy(void* e) { free(e); return 0; }
int hipEventElapsedTime(float* ms, void* a, void* b) { (void)a; (void)b; *ms = 1.0f; return 0; }
int hipEventRecord(void* e, void* st) { (void)e; (void)st; return 0; }
int hipEventSynchronize(void* e) { (void)e; return 0; }
const char* hipGetErrorString(int e) { (void)e; return "stub"; }
int hipGetLastError(void) { return 0; }
int hipGetSymbolAddress(void** p, const void* s) { *p = (void*)s; return 0; }
int hipStreamCreate(void** s) { *s = malloc(1); return 0; }
int hipStreamCreateWithFlags(void** s, unsigned f) { (void)f; *s = malloc(1); return 0; }
int hipStreamDestroy(void* s) { free(s); return 0; }
int hipStreamSynchronize(void* s) { (void)s; return 0; }
int hipStreamBeginCapture(void* s, int m) { (void)s; (void)m; return 0; }
int hipStreamEndCapture(void* s, void** g) { (void)s; *g = 0; return 0; }
int hipGraphAddChildGraphNode(void** n, void* g, void* const* d, size_t k, void* c) {
  (void)g; (void)d; (void)k; (void)c; *n = 0; return 0;
}
int hipGraphCreate(void** g, unsigned f) { (void)f; *g = 0; return 0; }
int hipGraphDestroy(void* g) { (void)g; return 0; }
int hipGraphExecDestroy(void* g) { (void)g; return 0; }
int hipGraphInstantiate(void** e, void* g, void* n, char* b, size_t k) {
  (void)g; (void)n; (void)b; (void)k; *e = 0; return 0;
}
int hipGraphLaunch(void* e, void* s) { (void)e; (void)s; return 0; }
int hipLaunchKernel(const void* f, ...) { (void)f; launches++; return 0; }
int __hipPushCallConfiguration(void) { return 0; }
int __hipPopCallConfiguration(void* g, void* b, size_t* shm, void** st) {
  memset(g, 0, 12); memset(b, 0, 12); *shm = 0; *st = 0; return 0;
}
void** __hipRegisterFatBinary(const void* d) { (void)d; return (void**)calloc(1, 8); }
void __hipRegisterFunction(void) {}
void __hipRegisterVar(void) {}
void __hipUnregisterFatBinary(void** m) { free(m); }
