// Stands in for the HIP runtime on the CPU (preloaded ahead of it), so that
// the library's host code can be run without a GPU: device memory is host
// memory, launches are recorded instead of run, and a copy to a device symbol
// can be made to fail.  Only the entry points that the tests reach are here.
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

typedef struct {
  uint32_t x, y, z;
} dim3_t;
typedef struct {
  dim3_t grid, block;
  size_t lds;
  void *stream;
} config_t;

typedef struct {
  const void *host;
  const char *name;
  size_t bytes;
  void *memory;
} symbol_t;

typedef struct {
  const char *name;
  dim3_t grid, block;
  uint64_t words[4];  // the first 32 bytes of the first argument, where asked for
} launch_t;

enum { MAX_SYMBOLS = 4096, MAX_LAUNCHES = 1 << 16 };
static symbol_t kernels[MAX_SYMBOLS], vars[MAX_SYMBOLS];
static int num_kernels, num_vars;
static launch_t launches[MAX_LAUNCHES];
static int num_launches;
static int symbol_copies, failing_copy = -1;
static _Thread_local config_t config;
static void *fat_binary;

// ---- what the tests ask
int fake_launches(void) { return num_launches; }
const char *fake_kernel(int i) { return launches[i].name; }
void fake_shape(int i, uint32_t *out) {
  memcpy(out, &launches[i].grid, sizeof(dim3_t));
  memcpy(out + 3, &launches[i].block, sizeof(dim3_t));
}
uint64_t fake_arg_word(int i, int w) { return launches[i].words[w]; }
void fake_reset(void) { num_launches = symbol_copies = 0; }
// Copy number n (from 0, counted from the last reset) to a symbol fails.
void fake_fail_symbol_copy(int n) { failing_copy = n; }

// ---- registration
void **__hipRegisterFatBinary(const void *data) {
  (void)data;
  return &fat_binary;
}
void __hipUnregisterFatBinary(void **modules) { (void)modules; }
void __hipRegisterFunction(void **modules, const void *host, char *device, const char *name, unsigned limit, void *tid,
                           void *bid, dim3_t *block, dim3_t *grid, int *wave) {
  (void)modules, (void)device, (void)limit, (void)tid, (void)bid, (void)block, (void)grid, (void)wave;
  if (num_kernels < MAX_SYMBOLS) kernels[num_kernels++] = (symbol_t){host, name, 0, 0};
}
void __hipRegisterVar(void **modules, void *host, char *host_name, char *name, int ext, size_t bytes, int constant,
                      int global) {
  (void)modules, (void)host_name, (void)ext, (void)constant, (void)global;
  if (num_vars < MAX_SYMBOLS) vars[num_vars++] = (symbol_t){host, name, bytes, 0};
}

// ---- launches
int __hipPushCallConfiguration(dim3_t grid, dim3_t block, size_t lds, void *stream) {
  config = (config_t){grid, block, lds, stream};
  return 0;
}
int __hipPopCallConfiguration(dim3_t *grid, dim3_t *block, size_t *lds, void **stream) {
  *grid = config.grid;
  *block = config.block;
  *lds = config.lds;
  *stream = config.stream;
  return 0;
}
static int record(const void *host, dim3_t grid, dim3_t block, void **args) {
  const char *name = "?";
  for (int i = 0; i < num_kernels; ++i)
    if (kernels[i].host == host) name = kernels[i].name;
  if (num_launches < MAX_LAUNCHES) {
    launch_t *l = &launches[num_launches++];
    *l = (launch_t){name, grid, block, {0}};
    if (strstr(name, "ntt_") && args) memcpy(l->words, args[0], sizeof l->words);  // pass arguments by value
  }
  // the runtime's limits
  if (!grid.x || !grid.y || !grid.z || grid.y > 65535 || grid.z > 65535 || (uint64_t)grid.x * block.x > 0xFFFFFFFFull)
    return 9;  // hipErrorInvalidConfiguration
  return 0;
}
int hipLaunchKernel(const void *host, dim3_t grid, dim3_t block, void **args, size_t lds, void *stream) {
  (void)lds, (void)stream;
  return record(host, grid, block, args);
}
int hipLaunchCooperativeKernel(const void *host, dim3_t grid, dim3_t block, void **args, unsigned lds, void *stream) {
  (void)lds, (void)stream;
  return record(host, grid, block, args);
}
int hipGetLastError(void) { return 0; }

// ---- memory
int hipMalloc(void **p, size_t n) { return (*p = calloc(1, n ? n : 1)) ? 0 : 2; }
int hipFree(void *p) {
  free(p);
  return 0;
}
int hipMemcpy(void *dst, const void *src, size_t n, int kind) {
  (void)kind;
  memcpy(dst, src, n);
  return 0;
}
int hipMemcpyAsync(void *dst, const void *src, size_t n, int kind, void *stream) {
  (void)stream;
  return hipMemcpy(dst, src, n, kind);
}
int hipGetSymbolAddress(void **p, const void *host) {
  for (int i = 0; i < num_vars; ++i)
    if (vars[i].host == host) {
      if (!vars[i].memory) vars[i].memory = calloc(1, vars[i].bytes);
      *p = vars[i].memory;
      return *p ? 0 : 2;
    }
  return 13;  // hipErrorInvalidSymbol
}
int hipMemcpyToSymbol(const void *host, const void *src, size_t n, size_t offset, int kind) {
  void *p;
  const int err = hipGetSymbolAddress(&p, host);
  if (err) return err;
  if (symbol_copies++ == failing_copy) return 1;
  return hipMemcpy((char *)p + offset, src, n, kind);
}

// ---- device
int hipGetDevice(int *dev) {
  *dev = 0;
  return 0;
}
int hipSetDevice(int dev) { return dev ? 101 : 0; }
int hipDeviceSynchronize(void) { return 0; }
int hipDeviceGetAttribute(int *v, int attr, int dev) {
  (void)attr, (void)dev;
  *v = 256;
  return 0;
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *blocks, const void *host, int threads, size_t lds) {
  (void)host, (void)threads, (void)lds;
  *blocks = 3;
  return 0;
}
int hipStreamIsCapturing(void *stream, int *status) {
  (void)stream;
  *status = 0;
  return 0;
}
