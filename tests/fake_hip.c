/* A HIP runtime without a device, for tests of the engine's host side: device
 * memory is counted, not given; kernels and copies do nothing.  Loaded with
 * RTLD_GLOBAL before the engine, whose references then bind to it. */
#include <pthread.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>
#include <unistd.h>

enum { OK = 0, INVALID = 1, OUT_OF_MEMORY = 2, MAXBUF = 4096 };

static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;
static struct { uintptr_t at; size_t bytes; } buf[MAXBUF];
static size_t capacity = (size_t)1 << 40, used;
static uintptr_t next = (uintptr_t)1 << 44;
static int bad_frees;
static volatile int hold, held;

void fake_capacity(size_t bytes) { capacity = bytes; }
size_t fake_used(void) { return used; }
int fake_bad_frees(void) { return bad_frees; }
void fake_hold(int on) { hold = on; }  /* the next wait for an event lasts until fake_hold(0) */
int fake_held(void) { return held; }

int hipMalloc(void** p, size_t bytes) {
  int e = OUT_OF_MEMORY;
  pthread_mutex_lock(&mu);
  *p = NULL;
  if (used + bytes <= capacity)
    for (int q = 0; q < MAXBUF && e; ++q)
      if (!buf[q].at) {
        buf[q].at = next;
        buf[q].bytes = bytes;
        *p = (void*)next;
        next += (bytes + 4095) / 4096 * 4096 + 4096;
        used += bytes;
        e = OK;
      }
  pthread_mutex_unlock(&mu);
  return e;
}
int hipFree(void* p) {
  int e = p ? INVALID : OK;
  pthread_mutex_lock(&mu);
  for (int q = 0; q < MAXBUF && e; ++q)
    if (buf[q].at == (uintptr_t)p) {
      used -= buf[q].bytes;
      buf[q].at = 0;
      e = OK;
    }
  if (e) ++bad_frees;
  pthread_mutex_unlock(&mu);
  return e;
}
int hipMemGetInfo(size_t* f, size_t* t) {
  *t = capacity;
  *f = capacity - used;
  return OK;
}
int hipHostMalloc(void** p, size_t bytes, unsigned flags) {
  *p = calloc(1, bytes);
  return *p ? OK : OUT_OF_MEMORY;
}
int hipHostFree(void* p) { free(p); return OK; }
int hipHostGetDevicePointer(void** d, void* h, unsigned flags) { *d = h; return OK; }
int hipGetDeviceCount(int* n) { *n = 1; return OK; }
int hipSetDevice(int d) { return OK; }
int hipDeviceGetAttribute(int* v, int what, int d) { *v = 256; return OK; }
int hipStreamCreateWithFlags(void** s, unsigned flags) { *s = (void*)8; return OK; }
int hipStreamSynchronize(void* s) { return OK; }
int hipStreamDestroy(void* s) { return OK; }
int hipEventCreate(void** e) { *e = (void*)16; return OK; }
int hipEventCreateWithFlags(void** e, unsigned flags) { *e = (void*)16; return OK; }
int hipEventRecord(void* e, void* s) { return OK; }
int hipEventDestroy(void* e) { return OK; }
int hipEventElapsedTime(float* ms, void* a, void* b) { *ms = 0.f; return OK; }
int hipEventSynchronize(void* e) {
  for (held = hold; hold;) usleep(1000);
  held = 0;
  return OK;
}
int hipMemcpy(void* d, const void* s, size_t bytes, int kind) { return OK; }
int hipMemcpyAsync(void* d, const void* s, size_t bytes, int kind, void* stream) { return OK; }
int hipMemsetAsync(void* d, int v, size_t bytes, void* stream) { return OK; }
int hipGetSymbolAddress(void** p, const void* symbol) { *p = (void*)32; return OK; }
const char* hipGetErrorString(int e) { return e == OUT_OF_MEMORY ? "out of memory" : "error"; }
int hipGetLastError(void) { return OK; }
typedef struct { unsigned x, y, z; } dim3_;
int hipLaunchKernel(const void* f, dim3_ g, dim3_ b, void** a, size_t lds, void* s) { return OK; }
int __hipPushCallConfiguration(dim3_ g, dim3_ b, size_t lds, void* s) { return OK; }
int __hipPopCallConfiguration(dim3_* g, dim3_* b, size_t* lds, void** s) {
  memset(g, 0, sizeof(*g));
  memset(b, 0, sizeof(*b));
  *lds = 0;
  *s = NULL;
  return OK;
}
void** __hipRegisterFatBinary(const void* data) { static void* h; return &h; }
void __hipRegisterFunction(void** m, const void* f, char* d, const char* n, unsigned t, void* ti,
                           void* bi, void* bd, void* gd, int* w) {}
void __hipRegisterVar(void** m, void* v, char* h, char* n, int e, size_t s, int c, int g) {}
void __hipUnregisterFatBinary(void** m) {}
