/* Host side of the HIP runtime entry points that libjqmc_hip.so uses, without a device: memory is host memory,
 * launches are recorded (kernel, grid, block, dynamic LDS, device) instead of run, and refused as the runtime
 * refuses them (2^32 work-items or more along x, more dynamic LDS than 64 KiB or than allowed for the kernel on
 * the current device).  Loaded before the library into a process that uses no GPU, it shows what the C entry
 * points would launch. */
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

typedef struct {
  uint32_t x, y, z;
} dim3_t;
enum { MAX_FN = 1 << 20, MAX_REC = 65536 };
static struct { const void* host; const char* name; } fns[MAX_FN];
static int n_fns;
static struct rec { const char* name; dim3_t g, b; uint64_t lds; int dev, error; } recs[MAX_REC];
static struct { const void* f; int dev, bytes; } allowed[MAX_REC];
static int n_recs, n_allowed, device, last_error;
static struct { dim3_t g, b; uint64_t lds; void* st; } cfg[16];
static int n_cfg;

static const char* name_of(const void* f) {
  for (int i = n_fns - 1; i >= 0; --i)
    if (fns[i].host == f) return fns[i].name;
  return "?";
}

void** __hipRegisterFatBinary(const void* d) { static void* h; (void)d; return &h; }
void __hipUnregisterFatBinary(void** m) { (void)m; }
void __hipRegisterFunction(void** m, const void* host, char* dev, const char* name, unsigned lim, void* a, void* b,
                           void* c, void* d, int* w) {
  (void)m, (void)dev, (void)lim, (void)a, (void)b, (void)c, (void)d, (void)w;
  if (n_fns < MAX_FN) fns[n_fns].host = host, fns[n_fns++].name = name;
}
void __hipRegisterVar(void** m, void* var, char* h, char* n, int e, size_t s, int c, int g) {
  (void)m, (void)var, (void)h, (void)n, (void)e, (void)s, (void)c, (void)g;
}
int __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t lds, void* st) {
  cfg[n_cfg].g = g, cfg[n_cfg].b = b, cfg[n_cfg].lds = lds, cfg[n_cfg++].st = st;
  return 0;
}
int __hipPopCallConfiguration(dim3_t* g, dim3_t* b, size_t* lds, void** st) {
  --n_cfg;
  *g = cfg[n_cfg].g, *b = cfg[n_cfg].b, *lds = cfg[n_cfg].lds, *st = cfg[n_cfg].st;
  return 0;
}
int hipLaunchKernel(const void* f, dim3_t g, dim3_t b, void** args, size_t lds, void* st) {
  (void)args, (void)st;
  uint64_t limit = 65536;
  for (int i = 0; i < n_allowed; ++i)
    if (allowed[i].f == f && allowed[i].dev == device) limit = (uint64_t)allowed[i].bytes;
  const int bad = (uint64_t)g.x * b.x > 0xffffffffull || g.x == 0 || g.y > 65535 || g.z > 65535 || lds > limit;
  if (bad) last_error = 9;
  if (n_recs < MAX_REC) {
    struct rec r = {name_of(f), g, b, lds, device, bad};
    recs[n_recs++] = r;
  }
  return bad ? 9 : 0;
}
int hipFuncSetAttribute(const void* f, int attr, int value) {
  if (attr == 8 && n_allowed < MAX_REC) /* the largest dynamic LDS */
    allowed[n_allowed].f = f, allowed[n_allowed].dev = device, allowed[n_allowed++].bytes = value;
  return 0;
}
int hipGetDevice(int* d) { *d = device; return 0; }
int hipMalloc(void** p, size_t n) { *p = calloc(1, n ? n : 1); return *p ? 0 : 2; }
int hipFree(void* p) { free(p); return 0; }
int hipHostMalloc(void** p, size_t n, unsigned f) { (void)f; return hipMalloc(p, n); }
int hipHostFree(void* p) { free(p); return 0; }
int hipMemcpy(void* d, const void* s, size_t n, int k) { (void)k; memcpy(d, s, n); return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int k, void* st) { (void)d, (void)s, (void)n, (void)k, (void)st; return 0; }
int hipMemsetAsync(void* d, int v, size_t n, void* st) { (void)d, (void)v, (void)n, (void)st; return 0; }
int hipStreamSynchronize(void* st) { (void)st; return 0; }
int hipGetLastError(void) {
  const int e = last_error;
  last_error = 0;
  return e;
}
const char* hipGetErrorString(int e) { (void)e; return "refused"; }
int hipGetSymbolAddress(void** p, const void* s) { (void)s; *p = 0; return 1; }

void shim_set_device(int d) { device = d; }
void shim_clear(void) { n_recs = 0; }
int shim_count(void) { return n_recs; }
/* kernel (mangled), grid x y z, block x, dynamic LDS, device, refused */
const char* shim_record(int i) {
  static char line[4096];
  const struct rec* r = &recs[i];
  snprintf(line, sizeof line, "%s %u %u %u %u %llu %d %d", r->name, r->g.x, r->g.y, r->g.z, r->b.x,
           (unsigned long long)r->lds, r->dev, r->error);
  return line;
}
