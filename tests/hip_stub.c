/* Stands in for the HIP runtime on a machine without a GPU: nothing runs, every call that matters to the library's
 * workspace is written down, and a test chooses what the runtime answers.  Loaded with global symbols before
 * libgemmzoo.so, so that the library's references find these definitions first. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <pthread.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

enum { OK = 0, OUT_OF_MEMORY = 2, LAUNCH_FAILURE = 719, CAPTURE_UNSUPPORTED = 900, MODE_GLOBAL = 0, MODE_RELAXED = 2 };
typedef struct { uint32_t x, y, z; } dim;

static pthread_mutex_t mutex = PTHREAD_MUTEX_INITIALIZER;
static char text[1 << 20];
static size_t used;
static uintptr_t capturing;              /* the stream that is being captured, 0: none */
static int sync_status, room, memory = 1 << 30;
static uintptr_t next_address = 0x7f0000000000;
static __thread int mode = MODE_GLOBAL;

static void note(const char* what, uintptr_t a, uintptr_t b, const char* name) {
  pthread_mutex_lock(&mutex);
  if (used + 512 < sizeof(text))
    used += (size_t)snprintf(text + used, 512, "%s %llu %llu %.400s\n", what, (unsigned long long)a, (unsigned long long)b, name);
  pthread_mutex_unlock(&mutex);
}

/* for the test */
void stub_capture(uintptr_t stream) { capturing = stream; }
void stub_sync_status(int status) { sync_status = status; }
void stub_memory(int allocations) { memory = allocations; }   /* how many more allocations succeed */
void stub_room(int on) { room = on, memory = on ? 0 : memory; }   /* every free makes room for one allocation */
const char* stub_take(void) {
  static char out[sizeof(text)];
  memcpy(out, text, used);
  out[used] = 0;
  used = 0;
  return out;
}

int hipMalloc(void** p, size_t bytes) {
  *p = 0;
  if (capturing && mode != MODE_RELAXED) return note("refused", bytes, 0, "-"), CAPTURE_UNSUPPORTED;
  if (memory <= 0) return note("nomemory", bytes, 0, "-"), OUT_OF_MEMORY;
  memory--;
  pthread_mutex_lock(&mutex);
  *p = (void*)next_address;
  next_address += (bytes + 0xfffff) & ~(uintptr_t)0xfffff;
  pthread_mutex_unlock(&mutex);
  note("malloc", bytes, (uintptr_t)*p, "-");
  return OK;
}
int hipFree(void* p) { return memory += room, note("free", (uintptr_t)p, 0, "-"), OK; }
int hipStreamSynchronize(void* s) { return note("sync", (uintptr_t)s, 0, "-"), sync_status; }
int hipStreamIsCapturing(void* s, int* status) { return *status = (uintptr_t)s == capturing && capturing != 0, OK; }
int hipThreadExchangeStreamCaptureMode(int* m) {
  const int old = mode;
  mode = *m;
  *m = old;
  return OK;
}
int hipGetDevice(int* d) { return *d = 0, OK; }
int hipDeviceGetAttribute(int* v, int attribute, int device) { return (void)attribute, (void)device, *v = 256, OK; }
int hipFuncSetAttribute(const void* f, int attribute, int v) { return (void)f, (void)attribute, (void)v, OK; }
int hipGetSymbolAddress(void** p, const void* symbol) { return (void)symbol, *p = (void*)0x600000000000, OK; }
int hipGetLastError(void) { return OK; }
const char* hipGetErrorString(int e) { return e == OUT_OF_MEMORY ? "out of memory" : "an error"; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void* st) { return (void)d, (void)s, (void)n, (void)kind, (void)st, OK; }

static __thread dim grid_, block_;
static __thread size_t lds_;
static __thread void* stream_;
int __hipPushCallConfiguration(dim grid, dim block, size_t lds, void* s) { return grid_ = grid, block_ = block, lds_ = lds, stream_ = s, OK; }
int __hipPopCallConfiguration(dim* grid, dim* block, size_t* lds, void** s) { return *grid = grid_, *block = block_, *lds = lds_, *s = stream_, OK; }
int hipLaunchKernel(const void* f, dim grid, dim block, void** args, size_t lds, void* s) {
  Dl_info info;
  (void)args;
  note("launch", (uintptr_t)s, grid.x, dladdr(f, &info) && info.dli_sname ? info.dli_sname : "?");
  note("group", (uintptr_t)block.x * block.y * block.z, lds, "-");   /* threads and LDS bytes of its work-groups */
  return OK;
}

void** __hipRegisterFatBinary(const void* data) { static void* handle; return (void)data, &handle; }
void __hipRegisterFunction(void** h, const void* f, char* df, const char* name, unsigned n, void* a, void* b, void* c, void* d, int* e) {
  (void)h; (void)f; (void)df; (void)name; (void)n; (void)a; (void)b; (void)c; (void)d; (void)e;
}
void __hipRegisterVar(void** h, void* v, char* hv, char* dv, int ext, size_t size, int constant, int global) {
  (void)h; (void)v; (void)hv; (void)dv; (void)ext; (void)size; (void)constant; (void)global;
}
void __hipUnregisterFatBinary(void** h) { (void)h; }
