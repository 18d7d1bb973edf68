// Host-only build of the solve's buffer handling (no device code, no GPU): device allocations come from
// malloc, the n-th of them fails.
#include "../../sparse-operator-graph-lu_amd/csrc/device/factor.hip"
#undef HIP_TRY
#include "../../sparse-operator-graph-lu_amd/csrc/device/solve.hip"
#include "no_device.h"

static int fail_at = -1, calls = 0;

extern "C" {
hipError_t hipMalloc(void** p, size_t bytes) {
    if (calls++ == fail_at) return hipErrorOutOfMemory;
    *p = malloc(bytes);
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    free(p);
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
}

// Buffers for 1 column, then for 4 with allocation `fail` of that growth failing, then for `again`: 0 if
// the last call succeeds and every buffer has room for its columns, 1 if it fails, 2 if one has not.
extern "C" int grow_after_failure(int fail, int again) {
    sogl_dev::Context c;
    sogl_dev::Factor f;
    f.block_rows = 2;
    if (sogl_dev::ensure_vectors(&c, &f, 1) != SOGL_OK) return -1;
    fail_at = calls + fail;
    if (sogl_dev::ensure_vectors(&c, &f, 4) == SOGL_OK) return -2;
    fail_at = -1;
    const int rc = sogl_dev::ensure_vectors(&c, &f, again);
    int out = rc != SOGL_OK;
    for (sogl_dev::DevBuf* b : {&f.vec_b, &f.vec_x, &f.vec_y}) {
        if (!rc && (!b->p || b->bytes < (size_t)again * 128 * 8)) out = 2;
        sogl_dev::dev_free(*b);
    }
    return out;
}
