/* A stand-in for the HIP runtime: records kernel launches by name and does
 * nothing else. Loaded before the library (RTLD_GLOBAL), it takes the
 * library's runtime calls, so a test sees without a GPU which kernel a call
 * launches, on which grid. hipMemPoolCreate can be told to fail. */
#include <stddef.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

typedef struct {
  unsigned x, y, z;
} Dim3;

enum { kMax = 4096, kArgBytes = 128, kOk = 0, kErr = 2 /* hipErrorOutOfMemory */ };

static struct {
  const void* host;
  const char* name;
} kernels[kMax];
static int kernel_count;

static struct {
  const char* name;
  Dim3 grid, block;
  char arg[kArgBytes]; /* of the tile GEMM: the start of its argument */
} launches[kMax];
static int launch_count, pool_fails, capturing, pool_allocs, pool_frees;

static struct {
  Dim3 grid, block;
  size_t shared;
  void* stream;
} pushed;

void stub_reset(void) { launch_count = pool_allocs = pool_frees = 0; }
void stub_fail_pool_create(int n) { pool_fails = n; }
void stub_capturing(int on) { capturing = on; }
int stub_pool_allocs(void) { return pool_allocs; }
int stub_pool_frees(void) { return pool_frees; }
int stub_launches(void) { return launch_count; }
const char* stub_name(int i) { return launches[i].name; }
void stub_grid(int i, unsigned* out) {
  out[0] = launches[i].grid.x;
  out[1] = launches[i].grid.y;
  out[2] = launches[i].grid.z;
  out[3] = launches[i].block.x;
}

const char* stub_arg(int i) { return launches[i].arg; }

void** __hipRegisterFatBinary(const void* data) {
  static void* handle;
  (void)data;
  return &handle;
}
void __hipUnregisterFatBinary(void** m) { (void)m; }
void __hipRegisterVar(void** m, void* v, char* h, char* d, int e, size_t s, int c, int g) {
  (void)m, (void)v, (void)h, (void)d, (void)e, (void)s, (void)c, (void)g;
}
void __hipRegisterFunction(void** m, const void* host, char* dev, const char* name, unsigned limit, void* tid,
                           void* bid, void* bd, void* gd, int* ws) {
  (void)m, (void)dev, (void)limit, (void)tid, (void)bid, (void)bd, (void)gd, (void)ws;
  if (kernel_count < kMax) {
    kernels[kernel_count].host = host;
    kernels[kernel_count++].name = name;
  }
}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t shared, void* stream) {
  pushed.grid = grid;
  pushed.block = block;
  pushed.shared = shared;
  pushed.stream = stream;
  return kOk;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* shared, void** stream) {
  *grid = pushed.grid;
  *block = pushed.block;
  *shared = pushed.shared;
  *stream = pushed.stream;
  return kOk;
}
int hipLaunchKernel(const void* f, Dim3 grid, Dim3 block, void** args, size_t shared, void* stream) {
  (void)shared, (void)stream;
  const char* name = "?";
  for (int i = 0; i < kernel_count; ++i)
    if (kernels[i].host == f) name = kernels[i].name;
  if (launch_count < kMax) {
    launches[launch_count].name = name;
    if (strstr(name, "gemm_tile_kernel") != NULL) memcpy(launches[launch_count].arg, args[0], kArgBytes);
    launches[launch_count].grid = grid;
    launches[launch_count++].block = block;
  }
  return kOk;
}
int hipLaunchCooperativeKernel(const void* f, Dim3 grid, Dim3 block, void** args, unsigned shared, void* stream) {
  return hipLaunchKernel(f, grid, block, args, shared, stream);
}

int hipGetDevice(int* dev) { return *dev = 0, kOk; }
int hipDeviceGetAttribute(int* v, int attr, int dev) {
  (void)attr, (void)dev;
  return *v = 256, kOk; /* the CU count */
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void* f, int threads, size_t shared) {
  (void)f, (void)threads, (void)shared;
  return *n = 2, kOk;
}
int hipStreamIsCapturing(void* s, int* status) {
  (void)s;
  return *status = capturing ? 1 : 0, kOk;
}
int hipMemPoolCreate(void** pool, const void* props) {
  (void)props;
  static char p;
  if (pool_fails > 0) return --pool_fails, kErr;
  return *pool = &p, kOk;
}
int hipMemPoolDestroy(void* pool) { return (void)pool, kOk; }
int hipMemPoolSetAttribute(void* pool, int attr, void* value) { return (void)pool, (void)attr, (void)value, kOk; }
int hipMallocFromPoolAsync(void** p, size_t bytes, void* pool, void* stream) {
  (void)bytes, (void)pool, (void)stream;
  ++pool_allocs;
  return *p = (void*)(uintptr_t)0x7f0000000000, kOk;
}
int hipFreeAsync(void* p, void* stream) { return (void)p, (void)stream, ++pool_frees, kOk; }
int hipMalloc(void** p, size_t n) { return *p = malloc(n), *p != NULL ? kOk : kErr; }
int hipFree(void* p) { return free(p), kOk; }
int hipMemcpy(void* d, const void* s, size_t n, int k) { return (void)d, (void)s, (void)n, (void)k, kOk; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int k, void* st) {
  return (void)d, (void)s, (void)n, (void)k, (void)st, kOk;
}
int hipGetSymbolAddress(void** p, const void* sym) { return *p = (void*)sym, kOk; }
int hipGetDevicePropertiesR0600(void* props, int dev) { return (void)props, (void)dev, kErr; }
int hipStreamSynchronize(void* s) { return (void)s, kOk; }
int hipGetLastError(void) { return kOk; }
const char* hipGetErrorString(int e) { return (void)e, "stub"; }
