/*
 * A HIP runtime and kernel launchers without a GPU, for the host code's own
 * paths (test_host_paths.py): device memory is host memory, launches count
 * themselves and do nothing.  Allocation `fail_at` (counted from 1, by
 * stub_reset) and any of more than `fail_above` bytes are refused, and
 * the synchronous copies while another thread captures (stub_capturing), as HIP
 * refuses them; as in HIP too, the error of a failed call stays the thread's
 * last error until hipGetLastError takes it, and a launcher reports it.
 */
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>
#include <stdlib.h>
#include <string.h>

#include "awefd.h"
#include "awefd_internal.h"
#include "res_adj.h"

long stub_allocs, stub_fail_at, stub_bytes, stub_resident, stub_adjoint, stub_steps, stub_rows, stub_max_rows, stub_recomputed;
size_t stub_fail_above;
int stub_launch_error, stub_give_up, stub_capturing;
static hipError_t last;

void stub_reset(long fail_at, size_t fail_above)
{
    stub_allocs = stub_resident = stub_adjoint = stub_steps = stub_rows = stub_max_rows = stub_recomputed = 0;
    stub_fail_at = fail_at;
    stub_fail_above = fail_above;
    stub_launch_error = stub_give_up = stub_capturing = 0;
    last = hipSuccess;
}

static hipError_t take(void **p, size_t n)
{
    stub_allocs++;
    if (stub_allocs == stub_fail_at || (stub_fail_above && n > stub_fail_above)) return last = hipErrorOutOfMemory;
    char *b = calloc(1, n + 64);
    if (!b) return last = hipErrorOutOfMemory;
    memcpy(b, &n, sizeof n);                           /* its size ahead of it */
    *p = b + 64;
    stub_bytes += (long)n;
    return hipSuccess;
}

hipError_t hipGetLastError(void)
{
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : e ? "other error" : "no error"; }
hipError_t hipMalloc(void **p, size_t n) { return take(p, n); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned f) { (void)f; return take(p, n); }
hipError_t hipFree(void *p)
{
    size_t n;
    if (!p) return hipSuccess;
    memcpy(&n, (char *)p - 64, sizeof n);
    stub_bytes -= (long)n;
    free((char *)p - 64);
    return hipSuccess;
}
hipError_t hipHostFree(void *p) { return hipFree(p); }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st)
{
    (void)k; (void)st;
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k)
{
    return stub_capturing ? (last = hipErrorStreamCaptureImplicit) : hipMemcpyAsync(d, s, n, k, NULL);
}
hipError_t hipMemcpy2D(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, hipMemcpyKind k)
{
    hipError_t e = hipSuccess;
    for (size_t i = 0; i < h && e == hipSuccess; i++) e = hipMemcpy((char *)d + i * dp, (const char *)s + i * sp, w, k);
    return e;
}
hipError_t hipMemGetInfo(size_t *f, size_t *t) { *f = *t = (size_t)288 << 30; return hipSuccess; }
hipError_t hipSetDevice(int d) { return d == 0 ? hipSuccess : (last = hipErrorInvalidDevice); }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int d)
{
    (void)d;
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 1;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned f) { (void)f; *s = (hipStream_t)malloc(1); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { free(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode m) { (void)s; (void)m; return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t *g) { (void)s; *g = (hipGraph_t)malloc(1); return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t g, hipGraphNode_t *n, char *l, size_t z)
{
    (void)g; (void)n; (void)l; (void)z;
    *x = (hipGraphExec_t)malloc(1);
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t s) { (void)x; (void)s; return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t x) { free(x); return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) { free(g); return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)malloc(1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { (void)e; (void)s; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b) { (void)a; (void)b; *ms = 1.f; return hipSuccess; }

/* launchers: the argument lists are the headers' */
static int launched(void) { return (int)hipGetLastError(); }

int awefd_launch_fill(float *p, long n, float v, void *s)
{
    (void)s;
    for (long i = 0; i < n; i++) p[i] = v;
    return launched();
}
int awefd_launch_cart_step(const awefd_cart_args *a, int nop, int ndim, int sse, int vd, void *s)
{
    (void)nop; (void)ndim; (void)sse; (void)vd; (void)s;
    stub_steps++;
    if (a->Pn) a->Pn[0] = (float)(a->it + 1);          /* marks the field a step writes out of place */
    return launched();
}
int awefd_launch_cart_traces(const awefd_cart_args *a, const float *c0, const float *seg, long nal, int nt, float *tr, void *s)
{
    (void)s;
    if (nt > stub_max_rows) stub_max_rows = nt;
    /* the mark of the field each row is read from, as the first trace */
    for (int n = 0; n < nt && a->nr > 0; n++) tr[(long)n * a->nr] = n == 0 ? *c0 : seg[(long)(n - 1) * nal];
    stub_rows += nt;
    return launched();
}
static int resident(const awefd_res_args *a)
{
    stub_resident++;
    if (stub_give_up) *a->stop = 1;
    return stub_launch_error;
}
#define RES(n) \
    int awefd__res_launch##n(const awefd_res_args *a, int nblk, int rx, int S, int vd, void *s) \
    { (void)nblk; (void)rx; (void)S; (void)vd; (void)s; return resident(a); } \
    int awefd__res_blocks##n(int rx, int S, int vd) { (void)rx; (void)S; (void)vd; return 1; }
RES(1) RES(2) RES(3) RES(4)
int awefd__polar_launch(const awefd_polar_args *a, int nblk, int rx, int S, void *s)
{
    (void)nblk; (void)rx; (void)S; (void)s;
    stub_resident++;
    if (stub_give_up) *a->stop = 1;
    return stub_launch_error;
}
int awefd__polar_blocks(int rx, int S) { (void)rx; (void)S; return 1; }
int awefd__resadj_launch(const awefd_resadj_args *a, int nblk, int nop, int rx, void *s)
{
    (void)nblk; (void)nop; (void)rx; (void)s;
    stub_adjoint++;
    if (stub_give_up) *a->stop = 1;
    return stub_launch_error;
}
int awefd__resadj_blocks(int nop, int rx) { (void)nop; (void)rx; return 1; }
int awefd__scratch(int dev, float **out)
{
    static float scratch[AWEFD_NOALLOC_TRACE_BYTES / 4];
    (void)dev;
    *out = scratch;
    return 0;
}
int awefd_cart_step_occupancy(int nop, int ndim, int sse) { (void)nop; (void)ndim; (void)sse; return 4; }
int awefd_spher_step_occupancy(int ndim) { (void)ndim; return 4; }

int awefd_launch_adj2d_step(const awefd_adj2d_args *a, int n, int nop, void *s)
{ (void)a; (void)n; (void)nop; (void)s; return launched(); }
int awefd_launch_adj2d_batch(const awefd_adj2d_args *a, const int *b, int nblk, int n, int nop, void *s)
{ (void)a; (void)b; (void)nblk; (void)n; (void)nop; (void)s; return launched(); }
int awefd_launch_adj2d_batch2(const awefd_adj2d_args *a, const int *b, int nblk, int n, int nop, void *s)
{ (void)a; (void)b; (void)nblk; (void)n; (void)nop; (void)s; return launched(); }
int awefd_launch_adj2d_chain(const awefd_adj2d_args *h, const awefd_adj2d_args *a, int nshot, float *g, void *s)
{ (void)h; (void)a; (void)nshot; (void)g; (void)s; return launched(); }
int awefd_launch_copy_jobs(const awefd_copy_job *j, const long *c, int n, long m, void *s)
{ (void)j; (void)c; (void)n; (void)m; (void)s; return launched(); }
int awefd_launch_set_vel(const float *d, float *v, const int n[3], const int nbs[3], int ld, float dt2, int fsnb, void *s)
{ (void)d; (void)v; (void)n; (void)nbs; (void)ld; (void)dt2; (void)fsnb; (void)s; return launched(); }
int awefd_launch_cart_abc_xy(const awefd_cart_args *a, int nop, void *s)
{ (void)a; (void)nop; (void)s; return launched(); }
int awefd_launch_cart_hybrid(const awefd_cart_args *a, int nop, int ndim, void *s)
{ (void)a; (void)nop; (void)ndim; (void)s; return launched(); }
int awefd_launch_cart_batch_t2(const awefd_cart_args *a, const int *b, int nblk, int it, int roles, int two, int nop, int sse, int rx, void *s)
{ (void)a; (void)b; (void)nblk; (void)it; (void)roles; (void)two; (void)nop; (void)sse; (void)rx; (void)s; return launched(); }
int awefd_launch_cart_batch_t3(const awefd_cart_args *a, const int *b, int nblk, int it, int roles, int nst, int nop, int sse, int rx, void *s)
{ (void)a; (void)b; (void)nblk; (void)it; (void)roles; (void)nst; (void)nop; (void)sse; (void)rx; (void)s; return launched(); }
int awefd_launch_cart_batch_rc(const awefd_cart_args *a, const int *b, int nblk, int n, int nop, int sse, int rx, void *s)
{ (void)a; (void)b; (void)nblk; (void)n; (void)nop; (void)sse; (void)rx; (void)s; stub_recomputed++; return launched(); }
int awefd_launch_cart_batch_t3rc(const awefd_cart_args *a, const int *b, int nblk, int n, int nop, int sse, int rx, void *s)
{ (void)a; (void)b; (void)nblk; (void)n; (void)nop; (void)sse; (void)rx; (void)s; stub_recomputed += 3; return launched(); }
int awefd_launch_cart_batch2(const awefd_cart_args *a, const int *b, int nblk, int it, int nop, int sse, int rx, void *s)
{ (void)a; (void)b; (void)nblk; (void)it; (void)nop; (void)sse; (void)rx; (void)s; return launched(); }
#define SPHER(n) int awefd_launch_spher_##n(const awefd_spher_args *a, void *s) { (void)a; (void)s; return launched(); }
SPHER(inject) SPHER(step) SPHER(shell) SPHER(extract) SPHER(points)
