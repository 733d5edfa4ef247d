/* A stand-in for the HIP runtime, for tests of the library's host side without a GPU
 * (host_hip.py): device memory is host memory, kernels are recorded instead of run, and an
 * allocation can be made to fail.  Copies and fills outside the live allocations are refused and
 * counted. */
#define _GNU_SOURCE
#include <stdint.h>
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>

enum { kOk = 0, kInvalid = 1, kNoMemory = 2 };
typedef struct { uint32_t x, y, z; } dim3;

/* --- device memory ------------------------------------------------------------------------- */
#define MAX_ALLOCS 4096
static struct { char* p; size_t n; int live; } g_alloc[MAX_ALLOCS];
static int g_allocs, g_fail, g_bad, g_copies, g_strided;

int hipMalloc(void** p, size_t n) {
  *p = NULL;
  if (g_fail > 0 && --g_fail == 0) return kNoMemory;
  if (g_allocs == MAX_ALLOCS) return kNoMemory;
  /* (pages that nothing touches take no memory) */
  char* q = mmap(NULL, n ? n : 1, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  if (q == MAP_FAILED) return kNoMemory;
  g_alloc[g_allocs].p = q;
  g_alloc[g_allocs].n = n;
  g_alloc[g_allocs++].live = 1;
  *p = q;
  return kOk;
}
int hipFree(void* p) {
  if (!p) return kOk;
  for (int i = 0; i < g_allocs; ++i)
    if (g_alloc[i].live && g_alloc[i].p == p) {
      g_alloc[i].live = 0;
      return munmap(p, g_alloc[i].n ? g_alloc[i].n : 1) ? kInvalid : kOk;
    }
  ++g_bad;
  return kInvalid;
}
static int inside(const void* p, size_t n) {
  for (int i = 0; i < g_allocs; ++i)
    if (g_alloc[i].live && (const char*)p >= g_alloc[i].p && (const char*)p + n <= g_alloc[i].p + g_alloc[i].n) return 1;
  ++g_bad;
  return 0;
}
/* kind: 1 host to device, 2 device to host, 3 device to device */
static int copy(void* d, const void* s, size_t n, int kind) {
  if (((kind & 1) && !inside(d, n)) || ((kind & 2) && !inside(s, n))) return kInvalid;
  memcpy(d, s, n);
  return kOk;
}
int hipMemcpy(void* d, const void* s, size_t n, int kind) {
  ++g_copies;
  return copy(d, s, n, kind);
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void* st) {
  (void)st;
  return hipMemcpy(d, s, n, kind);
}
int hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, int kind, void* st) {
  (void)st;
  ++g_strided;
  for (size_t r = 0; r < h; ++r) {
    const int e = copy((char*)d + r * dp, (const char*)s + r * sp, w, kind);
    if (e) return e;
  }
  return kOk;
}
int hipMemset(void* p, int v, size_t n) {
  if (!inside(p, n)) return kInvalid;
  if (v) memset(p, v, n);  /* fresh pages are zero */
  return kOk;
}
int hipHostMalloc(void** p, size_t n, unsigned flags) {
  (void)flags;
  *p = calloc(1, n);
  return *p ? kOk : kNoMemory;
}
int hipHostFree(void* p) {
  free(p);
  return kOk;
}
int hipMemGetInfo(size_t* f, size_t* t) {
  *f = (size_t)280 << 30;
  *t = (size_t)288 << 30;
  return kOk;
}

/* --- kernels ------------------------------------------------------------------------------- */
#define MAX_KERNELS 8192
#define MAX_LAUNCHES 65536
static struct { const void* f; const char* name; } g_kernel[MAX_KERNELS];
static struct { int k; dim3 grid, block; size_t lds; } g_launch[MAX_LAUNCHES];
static int g_kernels, g_launches;
static struct { dim3 grid, block; size_t lds; void* st; } g_cfg;

void** __hipRegisterFatBinary(const void* d) {
  static void* module;
  (void)d;
  return &module;
}
void __hipUnregisterFatBinary(void** m) { (void)m; }
void __hipRegisterFunction(void** m, const void* f, char* dev, const char* name, unsigned limit, void* tid, void* bid,
                           void* bdim, void* gdim, int* ws) {
  (void)m, (void)dev, (void)limit, (void)tid, (void)bid, (void)bdim, (void)gdim, (void)ws;
  if (g_kernels == MAX_KERNELS) abort();
  g_kernel[g_kernels].f = f;
  g_kernel[g_kernels++].name = strdup(name);
}
void __hipRegisterVar(void** m, void* var, char* hv, char* dv, int ext, size_t n, int c, int g) {
  (void)m, (void)var, (void)hv, (void)dv, (void)ext, (void)n, (void)c, (void)g;
}
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, void* st) {
  g_cfg.grid = g, g_cfg.block = b, g_cfg.lds = lds, g_cfg.st = st;
  return kOk;
}
int __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, void** st) {
  *g = g_cfg.grid, *b = g_cfg.block, *lds = g_cfg.lds, *st = g_cfg.st;
  return kOk;
}
int hipLaunchKernel(const void* f, dim3 g, dim3 b, void** args, size_t lds, void* st) {
  (void)args, (void)st;
  for (int i = 0; i < g_kernels; ++i)
    if (g_kernel[i].f == f) {
      if (g_launches == MAX_LAUNCHES) abort();
      g_launch[g_launches].k = i;
      g_launch[g_launches].grid = g;
      g_launch[g_launches].block = b;
      g_launch[g_launches++].lds = lds;
      return kOk;
    }
  return kInvalid;
}
int hipFuncSetAttribute(const void* f, int a, int v) { return (void)f, (void)a, (void)v, kOk; }
int hipGetSymbolAddress(void** p, const void* s) {
  static char* zero;  /* the arrays are never read: kernels are not run */
  (void)s;
  if (!zero) hipMalloc((void**)&zero, (size_t)128 << 20);
  *p = zero;
  return *p ? kOk : kNoMemory;
}

/* --- device, streams, events, graphs: nothing to do ----------------------------------------- */
int hipGetDevice(int* d) { return *d = 0, kOk; }
int hipSetDevice(int d) { return (void)d, kOk; }
int hipDeviceSynchronize(void) { return kOk; }
int hipGetLastError(void) { return kOk; }
const char* hipGetErrorString(int e) { return e == kNoMemory ? "out of memory" : e ? "invalid argument" : "no error"; }
static void* handle(void) { return malloc(8); }
static int g_streams;
int hipStreamCreateWithFlags(void** s, unsigned f) { return (void)f, ++g_streams, *s = handle(), kOk; }
int hipStreamDestroy(void* s) { return free(s), kOk; }
int hipStreamSynchronize(void* s) { return (void)s, kOk; }
int hipStreamWaitEvent(void* s, void* e, unsigned f) { return (void)s, (void)e, (void)f, kOk; }
int hipStreamBeginCapture(void* s, int m) { return (void)s, (void)m, kOk; }
int hipStreamEndCapture(void* s, void** g) { return (void)s, *g = handle(), kOk; }
int hipEventCreate(void** e) { return *e = handle(), kOk; }
int hipEventCreateWithFlags(void** e, unsigned f) { return (void)f, *e = handle(), kOk; }
int hipEventDestroy(void* e) { return free(e), kOk; }
int hipEventRecord(void* e, void* s) { return (void)e, (void)s, kOk; }
int hipEventSynchronize(void* e) { return (void)e, kOk; }
int hipEventElapsedTime(float* ms, void* a, void* b) { return (void)a, (void)b, *ms = 1.0f, kOk; }
int hipGraphInstantiate(void** x, void* g, void** n, char* log, size_t len) {
  return (void)g, (void)n, (void)log, (void)len, *x = handle(), kOk;
}
int hipGraphLaunch(void* x, void* s) { return (void)x, (void)s, kOk; }
int hipGraphDestroy(void* g) { return free(g), kOk; }
int hipGraphExecDestroy(void* x) { return free(x), kOk; }

/* --- what the tests ask -------------------------------------------------------------------- */
void host_hip_fail(int nth) { g_fail = nth; }  /* the nth hipMalloc from now fails (0: none) */
int host_hip_bad(void) { return g_bad; }       /* copies, fills and frees outside live memory */
int host_hip_streams(void) { return g_streams; }  /* created so far */
int host_hip_allocs(void) { return g_allocs; }
long long host_hip_alloc_bytes(int i) { return (long long)g_alloc[i].n; }
int host_hip_alloc_live(int i) { return g_alloc[i].live; }
int host_hip_launches(void) { return g_launches; }
void host_hip_forget(void) { g_launches = g_copies = g_strided = 0; }
int host_hip_copies(int strided) { return strided ? g_strided : g_copies; }
const char* host_hip_kernel(int i) { return g_kernel[g_launch[i].k].name; }
int host_hip_launch(int i, int what) {
  return what == 0 ? (int)g_launch[i].grid.x : what == 1 ? (int)g_launch[i].block.x : (int)g_launch[i].lds;
}
