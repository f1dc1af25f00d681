/* The HIP calls of the host library, without a GPU: a module with one kernel whose block size and
 * lanes per state the test sets, launches recorded, and the runtime's limit of fewer than 2^32
 * threads per launch. */
#include <stdint.h>
#include <string.h>

int stub_block = 256, stub_lanes = 0;           /* 0: the kernel exports no lanes per state */
struct launch { uint32_t grid, block; int n; const void *state, *rates; };
struct launch stub_log[64];
int stub_launches = 0;

int hipSetDevice(int d) { (void)d; return 0; }
int hipGetLastError(void) { return 0; }
const char* hipGetErrorString(int e) { (void)e; return "stub error"; }
int hipModuleLoad(void** m, const char* f) { (void)f; *m = &stub_block; return 0; }
int hipModuleLoadData(void** m, const void* d) { (void)d; *m = &stub_block; return 0; }
int hipModuleUnload(void* m) { (void)m; return 0; }
int hipGetSymbolAddress(void** p, const void* s) { (void)s; *p = &stub_block; return 0; }
int hipModuleGetFunction(void** f, void* m, const char* name)
{
  (void)m;
  *f = &stub_launches;
  return strcmp(name, "kx_bk1_fp64") ? 500 : 0;
}
int hipFuncGetAttribute(int* v, int a, const void* f) { (void)a; (void)f; *v = stub_block; return 0; }
int hipModuleGetGlobal(void** p, size_t* n, void* m, const char* name)
{
  (void)m;
  if (strcmp(name, "kx_bk1_fp64_lanes_per_state") || !stub_lanes) return 500;
  *p = &stub_lanes;
  *n = sizeof(int);
  return 0;
}
int hipMemcpyDtoH(void* d, void* s, size_t n) { memcpy(d, s, n); return 0; }
int hipModuleLaunchKernel(void* f, uint32_t gx, uint32_t gy, uint32_t gz, uint32_t bx, uint32_t by,
                          uint32_t bz, uint32_t lds, void* stream, void** args, void** extra)
{
  struct launch* l = &stub_log[stub_launches & 63];
  (void)f; (void)gy; (void)gz; (void)by; (void)bz; (void)lds; (void)stream; (void)extra;
  if ((uint64_t)gx * bx > 0xffffffffu) return 9;                 /* hipErrorInvalidConfiguration */
  l->grid = gx;
  l->block = bx;
  l->n = *(int*)args[0];
  l->state = *(void**)args[5];
  l->rates = *(void**)args[6];
  ++stub_launches;
  return 0;
}
