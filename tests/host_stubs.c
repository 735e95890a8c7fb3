/* A device that is host memory, for the host code's plan decisions on the CPU:
 * allocations come from calloc, copies are copies, and a kernel launch adds a
 * planted duration to a clock that the events read.  Entry points not defined
 * here are generated by the test and return 0. */
#include <hip/hip_runtime_api.h>
#include <stdlib.h>
#include <string.h>

#include "vnec_hip.h"

size_t stub_largest = (size_t)-1; /* a larger allocation fails */
int stub_layout_error;            /* returned by the layout builders */
int stub_choice;                  /* the learned selector's pick */
double stub_win_us = 1, stub_tiles_us = 1, stub_merge_us[16], stub_other_us = 1;
int stub_win_launches, stub_other_launches;
int stub_x_changes;               /* windowed launches on another x than the one before */

static double now_us, captured_us;
static int capturing;

static int launch(double us, int win)
{
    if (win) stub_win_launches++;
    else stub_other_launches++;
    if (capturing) captured_us += us;
    else now_us += us;
    return 0;
}

hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned f) { *s = (hipStream_t)&now_us; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int d) { *v = 256; return hipSuccess; }
const char *hipGetErrorString(hipError_t e) { return "planted"; }
hipError_t hipMalloc(void **p, size_t n)
{
    *p = n <= stub_largest ? calloc(1, n) : NULL;
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void *p) { free(p); return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t t)
{
    return hipMemcpy(d, s, n, k);
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t t) { memset(d, v, n); return hipSuccess; }

hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)calloc(1, sizeof(double)); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { *(double *)e = now_us; return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b)
{
    *ms = (float)((*(double *)b - *(double *)a) / 1e3);
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode m)
{
    capturing = 1;
    captured_us = 0;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t *g)
{
    double *us = (double *)malloc(sizeof *us);
    capturing = 0;
    *us = captured_us;
    *g = (hipGraph_t)us;
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t g, hipGraphNode_t *n, char *log, size_t size)
{
    double *us = (double *)malloc(sizeof *us);
    *us = *(double *)g;
    *e = (hipGraphExec_t)us;
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { free(g); return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { free(e); return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t s) { now_us += *(double *)e; return hipSuccess; }

int vnec_hip_merge_supported(int variant, int ipt, int enc, int nrhs) { return 1; }
int vnec_hip_stream_supported(int variant, int ipt, int enc, int block) { return 1; }
int vnec_hip_strided_supported(int variant, int ipt, int enc, int block, int gather) { return 1; }
int vnec_hip_d_supported(int ipt, int lanes) { return 1; }
int vnec_hip_stream_grid(int variant, int ipt, int enc, int block, int *nwg) { *nwg = 8; return 0; }
int vnec_hip_strided_grid(int variant, int ipt, int enc, int block, int gather, int *nwg) { *nwg = 8; return 0; }
int vnec_hip_scan_excl_i32(const int32_t *in, int32_t *out, int64_t n, int64_t *total, void *s)
{
    *total = 0;
    return 0;
}
int vnec_hip_max_tile_nnz(const int32_t *co, int64_t n, int32_t *mx, void *s) { *mx = 0; return 0; }
int vnec_hip_mlp_select(const float *p, const float *mu, const float *sd, const float *f, const uint32_t *mask,
                        int64_t n, int32_t *choice, void *s)
{
    *choice = stub_choice;
    return 0;
}
int vnec_hip_win_layout(const int32_t *ptr, const double *val, const uint16_t *lcol, const int32_t *co, int64_t n,
                        int ipt, int enc, double *wv, float *whi, float *wlo, uint16_t *wl, uint32_t *wt,
                        uint64_t *rmask, uint16_t *rbase, const int32_t *nec, int32_t *nsum, int32_t *mx, void *slot,
                        void *s)
{
    return stub_layout_error;
}
int vnec_hip_spmm_layout(const int32_t *ptr, const int32_t *col, const double *val, const int32_t *co, int64_t n,
                         int k, int run, double *sv, int32_t *sc, uint32_t *sf, uint64_t *rmask, int32_t *rbase,
                         int32_t *nsum, int32_t *mx, double *slot, void *s)
{
    return stub_layout_error;
}

int vnec_hip_spmv_win(const vnec_win_args *a, void *s)
{
    static const double *last;
    stub_x_changes += last != a->x;
    last = a->x;
    return launch(stub_win_us, 1);
}
int vnec_hip_spmm_tiles(const vnec_spmm_args *a, void *s) { return launch(stub_tiles_us, 1); }
int vnec_hip_spmv_merge(const vnec_merge_args *m, void *s)
{
    return launch(m->nrhs > 1 ? stub_merge_us[m->ipt] : stub_other_us, 0);
}
int vnec_hip_spmv_stream(const vnec_merge_args *m, int nwg, int32_t *row, double *carry, void *s)
{
    return launch(stub_other_us, 0);
}
int vnec_hip_spmv_strided(const vnec_merge_args *m, int nwg, void *s) { return launch(stub_other_us, 0); }
int vnec_hip_spmv_slice(const vnec_slice_args *a, void *s) { return launch(stub_other_us, 0); }
int vnec_hip_spmv_pattern(const vnec_pattern_args *a, void *s) { return launch(stub_other_us, 0); }
int vnec_hip_spmv_d(const vnec_d_args *a, void *s) { return launch(stub_other_us, 0); }
