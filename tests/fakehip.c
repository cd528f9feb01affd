/* A HIP runtime without a GPU, for tests of the library's host paths: memory is
 * the host's, up to a limit that the test sets, launches do nothing, and a
 * chosen clear can be made to fail. Loaded before the library with global
 * symbols, so that the library's calls come here. */
#include <hip/hip_runtime_api.h>
#include <stdlib.h>
#include <string.h>

typedef struct Block {
  void* p;
  size_t n;
  struct Block* next;
} Block;
static Block* blocks;
static size_t used, limit = (size_t)8 << 30;
static int fail_clear;        /* the clear to fail, counted from 1 */
static size_t clears[4096];   /* sizes of the clears that succeeded */
static int nclears;

void fake_limit(size_t n) { limit = n; }
size_t fake_used(void) { return used; }
void fake_fail_clear(int k) { fail_clear = k; }
int fake_clears(size_t n) {
  int c = 0;
  for (int i = 0; i < nclears; ++i) c += clears[i] == n;
  return c;
}

hipError_t hipMalloc(void** p, size_t n) {
  *p = NULL;
  if (used + n > limit) return hipErrorOutOfMemory;
  Block* b = malloc(sizeof *b);
  b->p = malloc(n ? n : 1);
  b->n = n;
  b->next = blocks;
  blocks = b;
  used += n;
  *p = b->p;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  for (Block** q = &blocks; *q; q = &(*q)->next)
    if ((*q)->p == p) {
      Block* b = *q;
      *q = b->next;
      used -= b->n;
      free(b->p);
      free(b);
      return hipSuccess;
    }
  return p ? hipErrorInvalidValue : hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
  *f = limit - used;
  *t = limit;
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned f) {
  (void)f;
  *p = calloc(1, n ? n : 1);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void* p) {
  free(p);
  return hipSuccess;
}
static hipError_t clear(void* p, int v, size_t n) {
  if (fail_clear && --fail_clear == 0) return hipErrorUnknown;
  memset(p, v, n);
  if (nclears < 4096) clears[nclears++] = n;
  return hipSuccess;
}
hipError_t hipMemset(void* p, int v, size_t n) { return clear(p, v, n); }
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t s) {
  (void)s;
  return clear(p, v, n);
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind k) {
  (void)k;
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t t) {
  (void)t;
  return hipMemcpy(d, s, n, k);
}
hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int d) {
  (void)d;
  memset(p, 0, sizeof *p);
  p->multiProcessorCount = 256;
  p->totalGlobalMem = limit;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int d) {
  (void)a;
  (void)d;
  *v = 100000;
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void* f, int b, size_t m) {
  (void)f;
  (void)b;
  (void)m;
  *n = 4;
  return hipSuccess;
}
static int handle;
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned f) { (void)f; *s = (hipStream_t)&handle; return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)&handle; return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) { (void)a; (void)b; *ms = 1.f; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned f) { (void)s; (void)e; (void)f; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { (void)e; (void)s; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t e) { (void)e; return "fake"; }
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void** a, size_t m, hipStream_t s) {
  (void)f; (void)g; (void)b; (void)a; (void)m; (void)s; return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t m, hipStream_t s) { (void)g; (void)b; (void)m; (void)s; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* m, hipStream_t* s) {
  (void)g; (void)b; (void)m; (void)s; return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode m) { (void)s; (void)m; return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* g) { (void)s; *g = (hipGraph_t)&handle; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, hipGraphNode_t* n, char* l, size_t k) {
  (void)g; (void)n; (void)l; (void)k;
  *e = (hipGraphExec_t)&handle;
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t s) { (void)e; (void)s; return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) { (void)g; return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { (void)e; return hipSuccess; }
