/* launch_recorder.c -- a stand-in for the HIP runtime entry points the library imports, for CPU
 * tests of its host side: nothing runs on a device, every launch is recorded.  Loaded RTLD_GLOBAL
 * ahead of the library (tests/launch_recorder.py), so the library's calls bind to these. */
#include <pthread.h>
#include <stdint.h>
#include <string.h>
#include <unistd.h>

typedef struct { uint32_t x, y, z; } dim3_;
typedef struct {
  const char* name;
  uint64_t first;  /* the first kernel argument's 8 bytes (a reduction's workspace) */
  uint32_t grid, block;
  void* stream;
  int thread;
} Launch;

enum { MAX_KERNELS = 4096, MAX_LAUNCHES = 65536 };
static struct { const void* fn; const char* name; } kernels[MAX_KERNELS];
static int n_kernels;
static Launch launches[MAX_LAUNCHES];
static int n_launches;
static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;
static void* capturing;    /* the stream under capture (NULL: none) */
static int delay_us;       /* after each launch */
static uintptr_t next_mem = 0x10000000;
static _Thread_local struct { dim3_ g, b; size_t sh; void* s; } conf;
static _Thread_local int thread_id;

/* ---- the test's side ---- */
void rec_reset(void) { n_launches = 0; }
int rec_count(void) { return n_launches; }
const Launch* rec_get(int i) { return &launches[i]; }
void rec_capture(void* s) { capturing = s; }
void rec_delay(int us) { delay_us = us; }
void rec_thread(int id) { thread_id = id; }

/* ---- the runtime's side ---- */
void** __hipRegisterFatBinary(const void* data) { static void* h; (void)data; return &h; }
void __hipUnregisterFatBinary(void** m) { (void)m; }
void __hipRegisterFunction(void** m, const void* fn, char* dev, const char* name, unsigned tl,
                           void* tid, void* bid, void* bd, void* gd, int* ws) {
  (void)m; (void)dev; (void)tl; (void)tid; (void)bid; (void)bd; (void)gd; (void)ws;
  if (n_kernels < MAX_KERNELS) { kernels[n_kernels].fn = fn; kernels[n_kernels++].name = name; }
}
void __hipRegisterVar(void** m, void* v, char* a, char* b, int e, size_t s, int c, int g) {
  (void)m; (void)v; (void)a; (void)b; (void)e; (void)s; (void)c; (void)g;
}
int __hipPushCallConfiguration(dim3_ g, dim3_ b, size_t sh, void* s) {
  conf.g = g; conf.b = b; conf.sh = sh; conf.s = s;
  return 0;
}
int __hipPopCallConfiguration(dim3_* g, dim3_* b, size_t* sh, void** s) {
  *g = conf.g; *b = conf.b; *sh = conf.sh; *s = conf.s;
  return 0;
}
int hipLaunchKernel(const void* fn, dim3_ g, dim3_ b, void** args, size_t sh, void* s) {
  (void)sh;
  pthread_mutex_lock(&mu);
  if (n_launches < MAX_LAUNCHES) {
    Launch* l = &launches[n_launches++];
    l->name = "?";
    for (int i = 0; i < n_kernels; ++i)
      if (kernels[i].fn == fn) l->name = kernels[i].name;
    memcpy(&l->first, args[0], 8);
    l->grid = g.x; l->block = b.x; l->stream = s; l->thread = thread_id;
  }
  pthread_mutex_unlock(&mu);
  if (delay_us) usleep(delay_us);
  return 0;
}
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipGetLastError(void) { return 0; }
int hipGetSymbolAddress(void** p, const void* sym) { (void)sym; *p = (void*)0x7000000000; return 0; }
int hipMalloc(void** p, size_t n) {
  pthread_mutex_lock(&mu);
  *p = (void*)next_mem;
  next_mem += (n + 0xffff) & ~(uintptr_t)0xffff;
  pthread_mutex_unlock(&mu);
  return 0;
}
int hipStreamIsCapturing(void* s, int* st) { *st = capturing && s == capturing ? 1 : 0; return 0; }
int hipThreadExchangeStreamCaptureMode(int* m) { (void)m; return 0; }
