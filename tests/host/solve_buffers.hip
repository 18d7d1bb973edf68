// Host-only build of the solve's buffer handling and of its choice of kernel (no device code, no GPU):
// device allocations come from malloc, the n-th of them fails.
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

// Whether an FP64 solve of a band of `rows` block rows, `half` of them to either side, then padding up to
// `block_rows`, loads whole steps ahead.
extern "C" int steps_ahead(int rows, int half, int block_rows, double zero_blocks) {
    sogl_dev::Factor f;
    sogl_dev::HostGraph hg;
    f.block_rows = block_rows;
    f.zero_blocks = zero_blocks;
    hg.lp.assign(1, 0);
    hg.up.assign(1, 0);
    for (int i = 0; i < block_rows; i++) {
        for (int j = std::max(0, i - half); i < rows && j < std::min(rows, i + half + 1); j++)
            if (j != i) (j < i ? hg.lc : hg.uc).push_back(j);
        hg.lp.push_back((int32_t)hg.lc.size());
        hg.up.push_back((int32_t)hg.uc.size());
    }
    sogl_dev::count_solve_tiles(&f, hg);
    return sogl_dev::whole_steps_ahead(&f);
}
