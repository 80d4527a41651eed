/* A stand-in for the HIP runtime calls libkq4.so makes, for tests of its host logic without a GPU:
 * memory is addresses nobody reads, a launch is a line in a log. Loaded with RTLD_GLOBAL before
 * libkq4.so, whose calls then bind here. Errors follow ROCm 7: hipGetLastError returns the thread's
 * last error, whatever succeeded since, and clears it. */
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>
#include <stdio.h>
#include <string.h>

#define EXPORT __attribute__((visibility("default")))

static struct { const void *fn; const char *name; } kern[1024];
static int nkern;
static char logbuf[1 << 16];
static size_t loglen, limit = (size_t)1 << 40, used, next = (size_t)1 << 32;
static struct { char *p; size_t n; } mem[256];
static int capturing, mallocs;
static hipError_t last = hipSuccess;

static hipError_t err(hipError_t e) {
  if (e != hipSuccess) last = e;
  return e;
}

/* ---- for the test ---- */
EXPORT void standin_limit(size_t bytes) { limit = bytes; }     /* of memory allocated at once */
EXPORT void standin_capture(int on) { capturing = on; }        /* every stream asked about */
EXPORT int standin_mallocs(void) { return mallocs; }           /* hipMalloc calls so far */
EXPORT size_t standin_used(void) { return used; }
EXPORT const char *standin_log(void) { return logbuf; }        /* launched kernels, a line each */
EXPORT void standin_clear(void) { logbuf[loglen = 0] = 0; }

/* ---- HIP ---- */
EXPORT void **__hipRegisterFatBinary(const void *data) { (void)data; static void *h; return &h; }
EXPORT void __hipUnregisterFatBinary(void **h) { (void)h; }
EXPORT void __hipRegisterFunction(void **h, const void *fn, char *dev, const char *name, unsigned lim,
                                  void *tid, void *bid, void *bd, void *gd, int *ws) {
  (void)h; (void)dev; (void)lim; (void)tid; (void)bid; (void)bd; (void)gd; (void)ws;
  if (nkern < 1024) { kern[nkern].fn = fn; kern[nkern++].name = name; }
}
EXPORT void __hipRegisterVar(void **h, void *var, char *host, char *dev, int ext, size_t size, int con,
                             int glob) {
  (void)h; (void)var; (void)host; (void)dev; (void)ext; (void)size; (void)con; (void)glob;
}
static struct { dim3 g, b; size_t lds; hipStream_t s; } cfg;
EXPORT hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
  cfg.g = g; cfg.b = b; cfg.lds = lds; cfg.s = s;
  return hipSuccess;
}
EXPORT hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s) {
  *g = cfg.g; *b = cfg.b; *lds = cfg.lds; *s = cfg.s;
  return hipSuccess;
}
EXPORT hipError_t hipLaunchKernel(const void *fn, dim3 g, dim3 b, void **args, size_t lds,
                                  hipStream_t s) {
  (void)args; (void)lds; (void)s;
  const char *name = "?";
  for (int i = 0; i < nkern; ++i)
    if (kern[i].fn == fn) name = kern[i].name;
  if (loglen + strlen(name) + 32 < sizeof logbuf)
    loglen += (size_t)sprintf(logbuf + loglen, "%s %u %u\n", name, g.x, b.x);
  return hipSuccess;
}
EXPORT hipError_t hipFuncSetAttribute(const void *fn, hipFuncAttribute a, int v) {
  (void)fn; (void)a; (void)v;
  return hipSuccess;
}
EXPORT hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
EXPORT hipError_t hipSetDevice(int d) { return err(d ? hipErrorInvalidDevice : hipSuccess); }
EXPORT hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
EXPORT hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int d) {
  (void)d;
  memset(p, 0, sizeof *p);
  strcpy(p->gcnArchName, "gfx950:sramecc+:xnack-");
  p->multiProcessorCount = 256;
  return hipSuccess;
}
EXPORT hipError_t hipGetSymbolAddress(void **p, const void *sym) {
  (void)sym;
  *p = (void *)((size_t)1 << 31);
  return hipSuccess;
}
EXPORT hipError_t hipMalloc(void **p, size_t n) {
  ++mallocs;
  if (capturing) return err(hipErrorStreamCaptureUnsupported);
  if (n > limit - used || used > limit) return err(hipErrorOutOfMemory);
  for (int i = 0; i < 256; ++i)
    if (!mem[i].p) {
      mem[i].p = *p = (char *)next;
      mem[i].n = n;
      next += (n + 4095) & ~(size_t)4095;
      used += n;
      return hipSuccess;
    }
  return err(hipErrorOutOfMemory);
}
EXPORT hipError_t hipFree(void *p) {
  for (int i = 0; i < 256; ++i)
    if (p && mem[i].p == p) {
      used -= mem[i].n;
      mem[i].p = 0;
      return hipSuccess;
    }
  return err(p ? hipErrorInvalidValue : hipSuccess);
}
EXPORT hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) {
  (void)d; (void)s; (void)n; (void)k;
  return hipSuccess;
}
EXPORT hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st) {
  (void)d; (void)s; (void)n; (void)k; (void)st;
  return hipSuccess;
}
EXPORT hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
EXPORT hipError_t hipStreamSynchronize(hipStream_t s) { (void)s; return hipSuccess; }
EXPORT hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *st) {
  (void)s;
  *st = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
EXPORT hipError_t hipGetLastError(void) {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
EXPORT const char *hipGetErrorString(hipError_t e) {
  return e == hipErrorOutOfMemory ? "out of memory" : "error";
}
