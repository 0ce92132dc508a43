/* The part of the HIP runtime that the library's host code calls, on host
 * memory: device memory comes from calloc, up to a limit that a test sets,
 * copies are memcpy, kernels do nothing.  Loaded before the library
 * (RTLD_GLOBAL), it lets tests follow the library's bookkeeping where device
 * memory runs out, without a device. */
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

enum { OK = 0, OUT_OF_MEMORY = 2 };

static size_t live, limit = ~(size_t)0;
static int last;
static long launches;

size_t stub_live(void) { return live; }
void stub_limit(size_t bytes) { limit = bytes; }
long stub_launches(void) { return launches; }

int hipMalloc(void** p, size_t bytes) {
  *p = NULL;
  if (bytes > limit || live > limit - bytes) return last = OUT_OF_MEMORY;
  char* m = calloc(1, bytes + 64); /* its size in front */
  if (!m) return last = OUT_OF_MEMORY;
  memcpy(m, &bytes, sizeof bytes);
  live += bytes;
  *p = m + 64;
  return OK;
}
int hipFree(void* p) {
  if (!p) return OK;
  char* m = (char*)p - 64;
  size_t bytes;
  memcpy(&bytes, m, sizeof bytes);
  live -= bytes;
  free(m);
  return OK;
}
int hipHostMalloc(void** p, size_t bytes, unsigned flags) {
  (void)flags;
  *p = malloc(bytes);
  return *p ? OK : OUT_OF_MEMORY;
}
int hipHostFree(void* p) { free(p); return OK; }
int hipMemcpy(void* d, const void* s, size_t n, int k) { (void)k; memcpy(d, s, n); return OK; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int k, void* st) { (void)k; (void)st; memcpy(d, s, n); return OK; }
int hipMemsetAsync(void* d, int v, size_t n, void* st) { (void)st; memset(d, v, n); return OK; }
int hipMemcpyToSymbolAsync(const void* y, const void* s, size_t n, size_t o, int k, void* st) {
  (void)y; (void)s; (void)n; (void)o; (void)k; (void)st;
  return OK;
}
int hipGetSymbolAddress(void** p, const void* y) { (void)y; static char room[64]; *p = room; return OK; }
int hipPointerGetAttributes(void* at, const void* p) { (void)p; *(int*)at = 0; return OK; } /* pageable */
int hipGetLastError(void) { int e = last; last = OK; return e; }
const char* hipGetErrorString(int e) { return e ? "out of memory" : "no error"; }
int hipGetDevice(int* d) { *d = 0; return OK; }
int hipSetDevice(int d) { (void)d; return OK; }
int hipStreamCreateWithFlags(void** s, unsigned f) { (void)f; *s = (void*)1; return OK; }
int hipStreamDestroy(void* s) { (void)s; return OK; }
int hipStreamSynchronize(void* s) { (void)s; return OK; }
int hipEventCreate(void** e) { *e = (void*)1; return OK; }
int hipEventCreateWithFlags(void** e, unsigned f) { (void)f; *e = (void*)1; return OK; }
int hipEventDestroy(void* e) { (void)e; return OK; }
int hipEventRecord(void* e, void* s) { (void)e; (void)s; return OK; }
int hipEventSynchronize(void* e) { (void)e; return OK; }

typedef struct { unsigned x, y, z; } dim3_t;
int __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t lds, void* st) { (void)g; (void)b; (void)lds; (void)st; return OK; }
int __hipPopCallConfiguration(dim3_t* g, dim3_t* b, size_t* lds, void** st) {
  g->x = g->y = g->z = b->x = b->y = b->z = 1;
  *lds = 0;
  *st = NULL;
  return OK;
}
int hipLaunchKernel(const void* f, dim3_t g, dim3_t b, void** args, size_t lds, void* st) {
  (void)f; (void)g; (void)b; (void)args; (void)lds; (void)st;
  ++launches;
  return OK;
}
void* __hipRegisterFatBinary(const void* d) { (void)d; static void* h; return &h; }
void __hipUnregisterFatBinary(void* h) { (void)h; }
void __hipRegisterFunction(void* h, const void* f, char* n, const char* d, unsigned t, void* a, void* b, void* c, void* e, int* w) {
  (void)h; (void)f; (void)n; (void)d; (void)t; (void)a; (void)b; (void)c; (void)e; (void)w;
}
void __hipRegisterVar(void* h, void* v, char* a, char* n, int e, size_t s, int c, int g) {
  (void)h; (void)v; (void)a; (void)n; (void)e; (void)s; (void)c; (void)g;
}
