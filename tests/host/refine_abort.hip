// Host-only build of the refined solve's host side (no device code, no GPU).  Device memory is host memory;
// of the kernels only the residual's contract is played: iterate number k is x = k everywhere (the first is
// 1), with a residual that never passes, unless solve number `abort_at` (from 1) was aborted.
#include "../../sparse-operator-graph-lu_amd/csrc/device/factor.hip"
#undef HIP_TRY
#include "../../sparse-operator-graph-lu_amd/csrc/device/solve.hip"
#undef HIP_TRY
#include "../../sparse-operator-graph-lu_amd/csrc/device/refine.hip"
#include "no_device.h"

static int abort_at = 0, solves = 0;
static size_t refuse = 0;  // allocations of this many bytes fail

extern "C" {
hipError_t hipMalloc(void** p, size_t bytes) {
    if (bytes == refuse) return hipErrorOutOfMemory;
    *p = malloc(bytes);
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) { return hipMalloc(p, bytes); }
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipHostGetDevicePointer(void** d, void* p, unsigned) {
    *d = p;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
    *ms = 1;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t bytes, hipMemcpyKind, hipStream_t) {
    memmove(d, s, bytes);
    return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* s, hipStream_t* st) {
    *g = *b = dim3(1);
    *s = 0;
    *st = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* k, dim3, dim3, void** a, size_t, hipStream_t) {
    if (k == (const void*)k_solve_begin) solves++;
    if (k != (const void*)k_residual<1>) return hipSuccess;
    double *xo = *(double**)a[6], *xold = *(double**)a[7], *norms = *(double**)a[15];
    const int n = *(int32_t*)a[9];
    const bool aborted = solves == abort_at;
    for (int i = 0; i < n && !aborted; i++) {
        if (xold) xold[i] = xo[i];
        xo[i] = solves;
    }
    for (int v = 0; v < NORM_VALUES; v++) norms[v] = 1;
    norms[NORM_VALUES] = aborted;
    return hipSuccess;
}
}

// x after a refined solve of up to max_iter corrections into an x of -1 whose solve number `at` times out
// (0: none), without room for a copy of x (`full`); the return code in rc.
extern "C" double x_after_abort(int at, int max_iter, int full, int* rc) {
    refuse = full ? 100 * sizeof(double) : 0;
    sogl_ctx x;
    Factor f;
    f.block_rows = 2;
    f.n = 100;
    f.elem = 8;
    f.has_refine = true;
    f.a_fro = f.a_inf = 1;
    x.c.num_cu = 1;
    x.c.factors[1] = &f;
    abort_at = at;
    solves = 0;
    std::vector<double> b(100, 1.0), xv(100, -1.0);
    int32_t it = 0;
    double resid = 0;
    *rc = sogl_solve_refined_device(&x, 1, b.data(), xv.data(), 1, 1e-12, max_iter, &it, &resid);
    for (double v : xv)
        if (v != xv[0]) return -2;
    return xv[0];
}
