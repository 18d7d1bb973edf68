// Mixed precision: an FP32 (or bf16-GEMM) factor is corrected by FP64
// iterative refinement against the original matrix,
//     x_0 = solve(b);  repeat  r = b - A x (FP64 CSR SpMV);  x += solve(r)
// until the normwise backward error is <= tol in both of its usual forms,
//     ||r||_inf / (||A||_inf ||x||_inf + ||b||_inf)  and
//     ||r||_2 / (||A||_F ||x||_2 + ||b||_2).
// (The second alone is about sqrt(n) looser at large n, since ||A||_F grows with
// sqrt(n) where ||A||_inf, a row sum, does not.)  FP64 lives only in the
// residual, the correction accumulation and the solve's vector sums; the
// factor tiles stay in their low precision.  The reference has no
// counterpart (it factors in FP64 only); its residual check is the max-abs
// mtx::checkResult (mtx.cpp:183-215).
//
// Also the drop-in sogl_solveLU, which mirrors SOGLU::solveLU (solver.h:24).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <mutex>
#include <vector>

#include "device.h"
#include "tile_ops.h"

using namespace sogl_dev;

namespace {

#define HIP_TRY(ctx, expr)                                       \
    do {                                                         \
        int _rc = check_hip((ctx), (expr), #expr);               \
        if (_rc != SOGL_OK) return _rc;                          \
    } while (0)

constexpr int RED_BLOCKS = 256;  // blocks of a column group in the residual kernel

// bp[i] = b[new_order[i]] for i < n, 1 on the padding rows (solver.cpp:155-161 + GPSOrder.cpp:433-447);
// also zeroes the residual kernel's block counters
__global__ void k_permute_in(const double* b, const int32_t* new_order, double* bp, int32_t n, int64_t N,
                             int nrhs, int* count, int ncount) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (blockIdx.y == 0)
        for (int64_t k = i; k < ncount; k += (int64_t)gridDim.x * blockDim.x) count[k] = 0;
    if (i >= N) return;
    const int64_t o = i < n ? new_order[i] : 0;
    for (int c = blockIdx.y; c < nrhs; c += gridDim.y) bp[i + c * N] = i < n ? b[o + (int64_t)c * n] : 1.0;
}

__global__ void k_axpy(double* x, const double* d, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] += d[i];
}

// All that follows a solve, in one launch: r = b - A x on the permuted padded system; x in
// the caller's order, xo[new_order[i]] = x[i] (GOrder::reOrderResult, GPSOrder.cpp:41-53);
// per column, over the first n rows, {||r||_2^2, ||x||_2^2, ||b||_2^2, ||r||_inf, ||x||_inf,
// ||b||_inf} and, after the columns, whether a pass of the solve was aborted, to pinned host
// memory `norms`, so that the host's one wait brings everything it decides by.  Where a pass was
// aborted, xo is left as it is; with xold, what xo held goes there first.  (As a
// residual, norm, copy and output kernel with a copy of the control words and three waits,
// and with every column in turn in one thread per row, it was half of a resident solve:
// random band 4,099 x 100 columns 3.1 of 3.6 ms, 2D 64^2 0.13 of 0.24.)
// A block takes CW columns (the matrix entries are read once for them); its sums go to
// part[(column * NORM_VALUES + v) * blocks + block], and the last block of a column group
// adds them up in block order, so a result does not depend on the blocks' timing.  A NaN
// reaches the maxima's reader through the sums (fmax drops NaN; the host checks the sums).
constexpr int NORM_VALUES = 6;
constexpr int RES_CW = 4;  // columns of a group (one column: 1)
constexpr int RES_NT = 256;

template <bool MAX>
__device__ inline double wave_reduce(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const double u = __shfl_xor(v, o);
        v = MAX ? fmax(v, u) : v + u;
    }
    return v;
}

template <int CW>
__global__ __launch_bounds__(RES_NT) void k_residual(const int64_t* ptr, const int32_t* col, const double* val,
                                                     const double* b, const double* x, double* r, double* xo,
                                                     double* xold, const int32_t* new_order, int32_t n, int64_t N, int nrhs,
                                                     double* part, int* count, const int* ctrl, double* norms) {
    __shared__ double s_w[RES_NT / 64][CW * NORM_VALUES];
    __shared__ int s_last;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, nb = gridDim.x;
    const int c0 = blockIdx.y * CW, cw = min(CW, nrhs - c0);
    const bool aborted = ctrl[1] || ctrl[5];
    const double* xc[CW];  // a column past the last repeats it and is not stored
#pragma unroll
    for (int c = 0; c < CW; c++) xc[c] = x + (int64_t)(c0 + min(c, cw - 1)) * N;
    double acc[CW][NORM_VALUES];
#pragma unroll
    for (int c = 0; c < CW; c++)
#pragma unroll
        for (int v = 0; v < NORM_VALUES; v++) acc[c][v] = 0;
    for (int64_t i = (int64_t)blockIdx.x * RES_NT + tid; i < N; i += (int64_t)nb * RES_NT) {
        double s[CW];
#pragma unroll
        for (int c = 0; c < CW; c++) s[c] = 0;
        int64_t e = ptr[i];
        const int64_t e1 = ptr[i + 1];
        for (; e + 4 <= e1; e += 4) {  // four entries' loads in flight
            double v[4], xv[4][CW];
            int32_t j[4];
#pragma unroll
            for (int k = 0; k < 4; k++) j[k] = col[e + k];
#pragma unroll
            for (int k = 0; k < 4; k++) v[k] = val[e + k];
#pragma unroll
            for (int k = 0; k < 4; k++)
#pragma unroll
                for (int c = 0; c < CW; c++) xv[k][c] = xc[c][j[k]];
#pragma unroll
            for (int k = 0; k < 4; k++)
#pragma unroll
                for (int c = 0; c < CW; c++) s[c] = fma(v[k], xv[k][c], s[c]);
        }
        for (; e < e1; e++) {
            const double v = val[e];
            const int32_t j = col[e];
#pragma unroll
            for (int c = 0; c < CW; c++) s[c] = fma(v, xc[c][j], s[c]);
        }
        const int64_t o = i < n ? new_order[i] : 0;
#pragma unroll
        for (int c = 0; c < CW; c++) {
            if (c >= cw) continue;
            const double bv = b[i + (int64_t)(c0 + c) * N], xv = xc[c][i], rv = bv - s[c];
            r[i + (int64_t)(c0 + c) * N] = rv;
            if (i < n) {
                if (!aborted) {
                    const int64_t q = o + (int64_t)(c0 + c) * n;
                    if (xold) xold[q] = xo[q];
                    xo[q] = xv;
                }
                acc[c][0] += rv * rv;
                acc[c][1] += xv * xv;
                acc[c][2] += bv * bv;
                acc[c][3] = fmax(acc[c][3], fabs(rv));
                acc[c][4] = fmax(acc[c][4], fabs(xv));
                acc[c][5] = fmax(acc[c][5], fabs(bv));
            }
        }
    }
#pragma unroll
    for (int c = 0; c < CW; c++)
#pragma unroll
        for (int v = 0; v < NORM_VALUES; v++) {
            const double t = v < 3 ? wave_reduce<false>(acc[c][v]) : wave_reduce<true>(acc[c][v]);
            if (lane == 0) s_w[w][c * NORM_VALUES + v] = t;
        }
    __syncthreads();
    if (tid < cw * NORM_VALUES) {
        double t = s_w[0][tid];
        for (int k = 1; k < RES_NT / 64; k++) t = tid % NORM_VALUES < 3 ? t + s_w[k][tid] : fmax(t, s_w[k][tid]);
        __hip_atomic_store(part + ((int64_t)c0 * NORM_VALUES + tid) * nb + blockIdx.x, t, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
    wave_stores_done();  // the partials are at the coherence point before the count
    __syncthreads();
    if (tid == 0)
        s_last = __hip_atomic_fetch_add(count + blockIdx.y, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == nb - 1;
    __syncthreads();
    if (!s_last) return;
    if (tid == 0) {
        count[blockIdx.y] = 0;  // for the next launch
        if (blockIdx.y == 0) norms[(int64_t)nrhs * NORM_VALUES] = aborted ? 1.0 : 0.0;
    }
    for (int v = w; v < cw * NORM_VALUES; v += RES_NT / 64) {
        const double* q = part + ((int64_t)c0 * NORM_VALUES + v) * nb;
        const bool sum = v % NORM_VALUES < 3;
        double t = 0;  // (maxima of magnitudes start at 0 too)
        for (int k = lane; k < nb; k += 64) {
            const double u = __hip_atomic_load(q + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            t = sum ? t + u : fmax(t, u);
        }
        t = sum ? wave_reduce<false>(t) : wave_reduce<true>(t);
        if (lane == 0) norms[(int64_t)c0 * NORM_VALUES + v] = t;
    }
}

}  // namespace

namespace sogl {
void set_last_error(const std::string& s);
}  // namespace sogl

extern "C" int sogl_refine_attach(sogl_ctx* x, int32_t factor_id, const sogl_plan* plan) {
    if (!x || !plan) return set_error(x ? &x->c : nullptr, SOGL_ERR_ARG, "null argument");
    Context* c = &x->c;
    std::lock_guard<std::mutex> g(c->mu);
    Factor* f = find_factor(c, factor_id);
    if (!f) return set_error(c, SOGL_ERR_ARG, "unknown factor id");
    sogl::PlanView v;
    if (!sogl::plan_view(plan, &v)) return set_error(c, SOGL_ERR_ARG, "bad plan");
    if (v.N != (int64_t)f->block_rows * TS) return set_error(c, SOGL_ERR_ARG, "plan does not match factor");
    HIP_TRY(c, hipSetDevice(c->device));
    // CSR of the permuted padded matrix, taken from the input tiles' cells so that the
    // residual uses the matrix the factor holds (where the COO repeats a position, the
    // tiles keep one value; the rows >= n hold the padding diagonal only)
    const int64_t nc = v.n_inputs ? v.cell_begin[v.n_inputs] : 0;
    std::vector<int64_t> ptr((size_t)v.N + 1, 0);
    for (int64_t t = 0; t < v.n_inputs; t++)
        for (int64_t q = v.cell_begin[t]; q < v.cell_begin[t + 1]; q++)
            ptr[(size_t)((int64_t)v.in_bi[t] * TS + (v.cell_pos[q] >> 6)) + 1]++;
    for (int64_t i = 0; i < v.N; i++) ptr[(size_t)i + 1] += ptr[(size_t)i];
    std::vector<int32_t> col((size_t)nc);
    std::vector<double> val((size_t)nc);
    std::vector<int64_t> pos(ptr.begin(), ptr.end() - 1);
    for (int64_t t = 0; t < v.n_inputs; t++)
        for (int64_t q = v.cell_begin[t]; q < v.cell_begin[t + 1]; q++) {
            const int64_t r = (int64_t)v.in_bi[t] * TS + (v.cell_pos[q] >> 6);
            const int64_t p = pos[(size_t)r]++;
            col[(size_t)p] = v.in_bj[t] * TS + (v.cell_pos[q] & 63);
            val[(size_t)p] = v.cell_val[q];
        }
    // each row by column, and the Frobenius and infinity norms over the rows of the
    // original matrix
    double fro = 0, inf = 0;
    std::vector<std::pair<int32_t, double>> row;
    for (int64_t i = 0; i < v.N; i++) {
        const int64_t b = ptr[(size_t)i], e = ptr[(size_t)i + 1];
        row.clear();
        for (int64_t p = b; p < e; p++) row.emplace_back(col[(size_t)p], val[(size_t)p]);
        std::sort(row.begin(), row.end(), [](const auto& x, const auto& y) { return x.first < y.first; });
        double rsum = 0;
        for (int64_t p = b; p < e; p++) {
            col[(size_t)p] = row[(size_t)(p - b)].first;
            val[(size_t)p] = row[(size_t)(p - b)].second;
            if (i < v.n) {
                fro += val[(size_t)p] * val[(size_t)p];
                rsum += std::fabs(val[(size_t)p]);
            }
        }
        inf = std::max(inf, rsum);
    }
    int rc;
    if ((rc = dev_alloc(c, f->csr_ptr, ptr.size() * 8, "csr ptr")) ||
        (rc = dev_alloc(c, f->csr_col, std::max<size_t>(col.size(), 1) * 4, "csr col")) ||
        (rc = dev_alloc(c, f->csr_val, std::max<size_t>(val.size(), 1) * 8, "csr val")))
        return rc;
    HIP_TRY(c, hipMemcpy(f->csr_ptr.p, ptr.data(), ptr.size() * 8, hipMemcpyHostToDevice));
    if (!col.empty()) {
        HIP_TRY(c, hipMemcpy(f->csr_col.p, col.data(), col.size() * 4, hipMemcpyHostToDevice));
        HIP_TRY(c, hipMemcpy(f->csr_val.p, val.data(), val.size() * 8, hipMemcpyHostToDevice));
    }
    f->n = v.n;
    f->nnz = nc;
    f->new_order.assign(v.new_order, v.new_order + v.n);
    if ((rc = dev_alloc(c, f->perm_d, (size_t)v.n * 4, "permutation"))) return rc;
    HIP_TRY(c, hipMemcpy(f->perm_d.p, v.new_order, (size_t)v.n * 4, hipMemcpyHostToDevice));
    f->a_fro = std::sqrt(fro);
    f->a_inf = inf;
    f->has_refine = true;
    return SOGL_OK;
}

// d_old (n x nrhs): takes what d_x held, which gets it back where a correction's solve fails;
// null: d_x may be left with an earlier iterate then.
static int refined_core(Context* c, Factor* f, const double* d_b, double* d_x, double* d_old, int32_t nrhs, double tol,
                        int32_t max_iter, int32_t* iters, double* resid) {
    const int32_t n = f->n;
    const int64_t N = (int64_t)f->block_rows * TS;
    int rc;
    const int cw = nrhs == 1 ? 1 : RES_CW, groups = (nrhs + cw - 1) / cw;
    const int nb = (int)std::min<int64_t>((N + RES_NT - 1) / RES_NT, RED_BLOCKS);
    const size_t part_bytes = (size_t)nrhs * NORM_VALUES * RED_BLOCKS * 8, norms = (size_t)nrhs * NORM_VALUES + 1;
    SolveWork w;
    if ((rc = ensure_vectors(c, f, nrhs)) || (rc = solve_work(c, f, w))) return rc;
    if ((rc = dev_alloc(c, f->vec_r, (size_t)N * nrhs * 8, "residual")) ||
        (rc = dev_alloc(c, f->vec_d, (size_t)N * nrhs * 8, "correction")) ||
        (rc = dev_alloc(c, f->red, part_bytes + (size_t)groups * sizeof(int), "norms")))
        return rc;
    if (c->norms_cap < norms) {
        if (c->norms_h) (void)hipHostFree(c->norms_h);
        c->norms_h = nullptr;
        c->norms_cap = 0;
        HIP_TRY(c, hipHostMalloc((void**)&c->norms_h, norms * 8, hipHostMallocDefault));
        c->norms_cap = norms;
    }
    double* d_norms = nullptr;
    HIP_TRY(c, hipHostGetDevicePointer((void**)&d_norms, c->norms_h, 0));
    double* db = (double*)f->vec_b.p;
    double* dx = (double*)f->vec_x.p;
    double* dr = (double*)f->vec_r.p;
    double* dd = (double*)f->vec_d.p;
    int* count = (int*)((char*)f->red.p + part_bytes);
    const unsigned gN = (unsigned)((N + 255) / 256);
    const unsigned gA = (unsigned)((N * nrhs + 255) / 256);
    hipLaunchKernelGGL(k_permute_in, dim3(gN, (unsigned)std::min(nrhs, 65535)), dim3(256), 0, c->stream, d_b,
                       (const int32_t*)f->perm_d.p, db, n, N, nrhs, count, groups);
    HIP_TRY(c, hipGetLastError());
    if ((rc = solve_launch(c, f, w, db, dx, nrhs))) return rc;
    double solve_ms = 0;
    int it = 0;
    double worst = 0;
    auto fail = [&](int code) {
        if (it > 0 && d_old) {
            HIP_TRY(c, hipMemcpyAsync(d_x, d_old, (size_t)n * nrhs * 8, hipMemcpyDeviceToDevice, c->stream));
            HIP_TRY(c, hipStreamSynchronize(c->stream));
        }
        return code;
    };
    for (;;) {
        auto kern = cw == 1 ? k_residual<1> : k_residual<RES_CW>;
        hipLaunchKernelGGL(kern, dim3(nb, groups), dim3(RES_NT), 0, c->stream, (const int64_t*)f->csr_ptr.p,
                           (const int32_t*)f->csr_col.p, (const double*)f->csr_val.p, (const double*)db,
                           (const double*)dx, dr, d_x, it == 0 ? d_old : nullptr, (const int32_t*)f->perm_d.p, n, N, nrhs,
                           (double*)f->red.p, count, (const int*)w.ctrl, d_norms);
        HIP_TRY(c, hipGetLastError());
        HIP_TRY(c, hipStreamSynchronize(c->stream));
        float ms = 0;
        HIP_TRY(c, hipEventElapsedTime(&ms, c->ev0, c->ev1));
        solve_ms += ms;
        if (c->norms_h[norms - 1] != 0) return fail(solve_timeout(c));
        worst = 0;
        for (int32_t r = 0; r < nrhs; r++) {
            const double* v = c->norms_h + (size_t)r * NORM_VALUES;
            const double den2 = f->a_fro * std::sqrt(v[1]) + std::sqrt(v[2]);
            const double rel2 = den2 > 0 ? std::sqrt(v[0]) / den2 : std::sqrt(v[0]);
            const double deni = f->a_inf * v[4] + v[5];
            const double reli = deni > 0 ? v[3] / deni : v[3];
            const double rel = std::isnan(rel2) ? rel2 : std::max(rel2, reli);
            if (!(rel <= worst)) worst = rel;  // NaN propagates
        }
        if (worst <= tol || it >= max_iter || std::isnan(worst)) break;
        it++;
        if ((rc = solve_launch(c, f, w, dr, dd, nrhs))) return fail(rc);
        hipLaunchKernelGGL(k_axpy, dim3(gA), dim3(256), 0, c->stream, dx, (const double*)dd, N * nrhs);
        HIP_TRY(c, hipGetLastError());
    }
    f->solve_ms = solve_ms;
    if (iters) *iters = it;
    if (resid) *resid = worst;
    if (std::isnan(worst)) return set_error(c, SOGL_ERR_NAN, "refinement: NaN in the residual");
    if (!(worst <= tol)) return set_error(c, SOGL_ERR_NOT_CONVERGED, "refinement did not reach the tolerance");
    return SOGL_OK;
}

extern "C" int sogl_solve_refined_device(sogl_ctx* x, int32_t factor_id, const double* d_b, double* d_x,
                                         int32_t nrhs, double tol, int32_t max_iter, int32_t* iters,
                                         double* resid) {
    if (!x || !d_b || !d_x || nrhs <= 0) return set_error(x ? &x->c : nullptr, SOGL_ERR_ARG, "bad argument");
    Context* c = &x->c;
    std::lock_guard<std::mutex> g(c->mu);
    Factor* f = find_factor(c, factor_id);
    if (!f) return set_error(c, SOGL_ERR_ARG, "unknown factor id");
    if (!f->has_refine) return set_error(c, SOGL_ERR_ARG, "sogl_refine_attach was not called");
    HIP_TRY(c, hipSetDevice(c->device));
    // (no room for what d_x holds is no reason to refuse the solve)
    const bool old = max_iter > 0 && dev_alloc(c, f->vec_io, (size_t)f->n * nrhs * 8, "earlier x") == SOGL_OK;
    return refined_core(c, f, d_b, d_x, old ? (double*)f->vec_io.p : nullptr, nrhs, tol, max_iter, iters, resid);
}

extern "C" int sogl_solve_refined(sogl_ctx* x, int32_t factor_id, const double* b, double* xo,
                                  int32_t nrhs, double tol, int32_t max_iter, int32_t* iters,
                                  double* resid) {
    if (!x || !b || !xo || nrhs <= 0) return set_error(x ? &x->c : nullptr, SOGL_ERR_ARG, "bad argument");
    Context* c = &x->c;
    std::lock_guard<std::mutex> g(c->mu);
    Factor* f = find_factor(c, factor_id);
    if (!f) return set_error(c, SOGL_ERR_ARG, "unknown factor id");
    if (!f->has_refine) return set_error(c, SOGL_ERR_ARG, "sogl_refine_attach was not called");
    HIP_TRY(c, hipSetDevice(c->device));
    const size_t bytes = (size_t)f->n * nrhs * 8;
    int rc;
    if ((rc = dev_alloc(c, f->vec_io, 2 * bytes, "refine io"))) return rc;
    double* db = (double*)f->vec_io.p;
    double* dx = db + (size_t)f->n * nrhs;
    HIP_TRY(c, hipMemcpyAsync(db, b, bytes, hipMemcpyHostToDevice, c->stream));
    int rc2 = refined_core(c, f, db, dx, nullptr, nrhs, tol, max_iter, iters, resid);
    if (rc2 != SOGL_OK && rc2 != SOGL_ERR_NOT_CONVERGED && rc2 != SOGL_ERR_NAN) return rc2;
    HIP_TRY(c, hipMemcpyAsync(xo, dx, bytes, hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(c, hipStreamSynchronize(c->stream));
    return rc2;
}

// ------------------------------------------------------------------ drop-in solveLU
extern "C" int sogl_factor_load_plan(sogl_ctx* x, const sogl_plan* plan, int32_t precision,
                                     int32_t* factor_id);

extern "C" int sogl_solveLU(int32_t dim, int64_t valcount, int32_t symmetric, const int32_t* index_i,
                            const int32_t* index_j, const double* vals, const double* b, double* xo) {
    static std::mutex mu;
    static sogl_ctx* ctx = nullptr;
    std::lock_guard<std::mutex> g(mu);
    if (!xo || !b) return set_error(nullptr, SOGL_ERR_ARG, "null b or x");
    sogl_plan* plan = nullptr;
    int rc = sogl_plan_create(dim, valcount, symmetric, index_i, index_j, vals, b, 0, &plan);
    if (rc) return rc;
    if (!ctx && (rc = sogl_ctx_create(0, &ctx))) {
        sogl_plan_destroy(plan);
        return rc;
    }
    int32_t fid = 0;
    if ((rc = sogl_factor_load_plan(ctx, plan, SOGL_FP64, &fid))) {
        sogl_plan_destroy(plan);
        return rc;
    }
    sogl_plan_info info;
    sogl_plan_get_info(plan, &info);
    const int64_t N = (int64_t)info.block_rows * 64;
    std::vector<double> bp((size_t)N), xp((size_t)N);
    rc = sogl_factor_run(ctx, fid, SOGL_EXEC_PERSISTENT);
    if (!rc) rc = sogl_plan_permute_rhs(plan, b, 1, dim, bp.data());
    if (!rc) rc = sogl_solve(ctx, fid, bp.data(), xp.data(), nullptr, 1);
    if (!rc) rc = sogl_plan_unpermute(plan, xp.data(), 1, xo, dim);
    sogl_factor_release(ctx, fid);
    sogl_plan_destroy(plan);
    if (!rc)
        for (int32_t i = 0; i < dim; i++)
            if (std::isnan(xo[i])) return set_error(nullptr, SOGL_ERR_NAN, "NaN in the solution");
    return rc;
}

// ------------------------------------------------------------------ device memory helpers
extern "C" int sogl_device_alloc(sogl_ctx* x, size_t bytes, void** ptr) {
    if (!x || !ptr) return set_error(nullptr, SOGL_ERR_ARG, "null argument");
    Context* c = &x->c;
    HIP_TRY(c, hipSetDevice(c->device));
    HIP_TRY(c, hipMalloc(ptr, bytes));
    return SOGL_OK;
}

extern "C" int sogl_device_free(sogl_ctx* x, void* ptr) {
    if (!x) return set_error(nullptr, SOGL_ERR_ARG, "null context");
    Context* c = &x->c;
    HIP_TRY(c, hipSetDevice(c->device));
    if (ptr) HIP_TRY(c, hipFree(ptr));
    return SOGL_OK;
}

extern "C" int sogl_device_copy(sogl_ctx* x, void* dst, const void* src, size_t bytes, int32_t to_device) {
    if (!x || (bytes && (!dst || !src))) return set_error(nullptr, SOGL_ERR_ARG, "null argument");
    Context* c = &x->c;
    HIP_TRY(c, hipSetDevice(c->device));
    HIP_TRY(c, hipMemcpyAsync(dst, src, bytes, to_device ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(c, hipStreamSynchronize(c->stream));
    return SOGL_OK;
}
