// Block triangular solve with many right-hand sides: replaces
// BlockPlanner::solve / lowerSolver / upperSolver / updateVector
// (BlockPlanner.cpp:669-862), which recurse over the L and U quadtrees with
// one right-hand side, serially.
//
// Here a persistent kernel solves, forward,
//     y_I = Linv_II (b_I - sum_{J<I} L_IJ y_J)
// backward,
//     x_I = Uinv_II (y_I - sum_{J>I} U_IJ x_J)
// with the inverses of the diagonal tiles and the off-diagonal block of each row pair's 2x2
// diagonal block's inverse made once per factor.  Tasks are pairs of block rows, taken in
// dependency order (ascending / descending); a task waits only for the rows it reads, on the
// stored values themselves (a pending marker until stored), so independent rows overlap and
// the chain only serialises where the factor's block structure does.  With 1-15 right-hand
// sides every column is a chain of tasks of its own, from 16 on every panel of 16 columns is
// (on MFMA).  Sums run in FP64 for every tile precision.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "device.h"
#include "tile_ops.h"

namespace sogl_dev {

constexpr long long SOLVE_SPIN_LIMIT = 20LL * 100 * 1000 * 1000;
constexpr int TRSM_MIN_RHS = 16;   // from this many right-hand sides the block-row sums run on MFMA
// FP64 solves of 1-15 columns: off-diagonal tiles of L and U together per block row that has one
// (padding rows have none), less the share of zero blocks, from which the kernel that loads a
// whole step ahead (KEEP) is taken.  A solve of one column without / with it, ms, by that
// number: 1.6 (2D 64^2) 0.093 / 0.112, 3.3 (2D convection-diffusion 300^2) 1.89 / 2.15, 4.2
// (2D 200^2) 0.99 / 1.07, 4.6 (3D 16^3) 0.122 / 0.126, 4.75 (2D 230^2) 1.48 / 1.42, 5.4 (2D
// 256^2) 2.21 / 1.78, 6.8 (3D 20^3) 0.308 / 0.234, 8.2 (2D 400^2) 7.78 / 5.08, 16 (3D 31^3)
// 1.82 / 1.39.
constexpr double KEEP_TILES = 4.7;
constexpr int MAX_RHS = 1024;      // columns per launch: pairs x panels fit the 32-bit task counter

struct SolveArgs {
    const void* pool;
    const int32_t* rowptr;
    const int32_t* col;
    const int32_t* slot;
    const int32_t* dinv;  // per block row: slot of the inverted diagonal tile
    const double* in;
    double* out;
    int64_t ld;           // column stride of in/out (padded n)
    int32_t nrhs;
    int32_t nbr;
    int32_t forward;
    int* ctrl;            // the pass's: [0] task counter, [1] abort
    const uint32_t* mask; // per slot: the factor's 16x16 block masks (a zero tile is skipped)
    const int32_t* prow;     // the many-RHS form's steps (pair_steps): per row pair, its steps'
    const int32_t* pcol;     // block column pairs
    const int4* pslot;       // and tiles
    const int32_t* pairinv;  // per row pair: slot of the 2x2 diagonal block's inverse's
                             // off-diagonal block, -1: zero
};

// The abort word and the wall clock are looked at every SOLVE_SPIN_CHECK polls only, so
// that each poll costs one round trip to the device coherence point.
constexpr int SOLVE_SPIN_CHECK = 64;

// Rows of the output that a pass has not stored yet hold this signalling NaN, written before
// the pass (k_solve_begin; k_fill_pending for an x that shares memory with b).  FP arithmetic
// never produces a signalling NaN (a NaN result is quiet), so a stored value is never mistaken
// for it.  A task polls the values it reads themselves, with agent-scope atomic loads, until
// none is the marker, and stores its rows with agent-scope atomic stores, which reach the
// coherence point without a release.
constexpr unsigned long long SOLVE_PENDING = 0x7FF4C0DE5EED0001ull;

// Before the two passes: the outputs of both pending (x null: y alone), the task counters of
// both (ctrl[0], ctrl[4]) at zero and, before the first columns, their abort words (ctrl[1],
// ctrl[5]).
__global__ void k_solve_begin(int* ctrl, int first, double* y, double* x, int64_t n) {
    if (blockIdx.x == 0 && threadIdx.x < SOLVE_CTRL_WORDS && (first || threadIdx.x % 4 == 0)) ctrl[threadIdx.x] = 0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        reinterpret_cast<unsigned long long*>(y)[i] = SOLVE_PENDING;
        if (x) reinterpret_cast<unsigned long long*>(x)[i] = SOLVE_PENDING;
    }
}
__global__ void k_fill_pending(double* x, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        reinterpret_cast<unsigned long long*>(x)[i] = SOLVE_PENDING;
}

// A wait has exceeded its bound: every task ends.  A release, so that whoever sees the word
// sees all that this wave stored before it.
__device__ inline void raise_abort(const SolveArgs& a) {
    release_agent();
    __hip_atomic_store(a.ctrl + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The 64 values of one column of row J, which another task stores, into this wave's
// LDS slot ls once all are stored: lane l polls value l (one coalesced load per spin
// for the wave), the wave's ballot says when none is pending.  NC = 2 polls the same
// column of a second row (col + step) in the same spin, into ls[64 ..]: the two rows a
// row-pair task stores together cost one wait.  On the wait bound (or an abort
// elsewhere) it raises the abort flag and leaves zeros.  The caller reads ls after it
// (LDS accesses of one wave complete in order).
template <int NC = 1>
__device__ inline void load_row_stored(const double* col, double* ls, int lane, const SolveArgs& a,
                                       int64_t step = 0) {
    const unsigned long long* q = reinterpret_cast<const unsigned long long*>(col) + lane;
    long long t0 = 0;
    unsigned long long u[NC];
    for (int spin = 0;; spin++) {
        bool pend = false;
#pragma unroll
        for (int i = 0; i < NC; i++) {
            u[i] = __hip_atomic_load(q + i * step, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            pend |= u[i] == SOLVE_PENDING;
        }
        if (!__ballot(pend)) break;
        if (spin == 0) {
            t0 = wall_clock64();
        } else if (spin % SOLVE_SPIN_CHECK == 0 &&
                   (__hip_atomic_load(a.ctrl + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ||
                    wall_clock64() - t0 > SOLVE_SPIN_LIMIT)) {
            raise_abort(a);
#pragma unroll
            for (int i = 0; i < NC; i++) u[i] = 0;  // the bit pattern of 0.0
            break;
        }
        __builtin_amdgcn_s_sleep(2);
    }
#pragma unroll
    for (int i = 0; i < NC; i++) ls[i * TS + lane] = __longlong_as_double((long long)u[i]);
    __builtin_amdgcn_wave_barrier();
}

// Two block rows per task (a row pair p: rows 2p, 2p+1), pairs taken in dependency
// order, so each hand-off along the chain serves two rows.  With A the pair's row solved
// first (forward 2p, backward 2p+1) and B the other, and r_A, r_B the right-hand sides
// less the products of every earlier row (B's entry in column A left out):
//     x_A = D_A^-1 r_A,   x_B = D_B^-1 r_B + C_p r_A,
// where C_p is the off-diagonal block of the inverse of the pair's 2x2 diagonal block
// (forward X_p = -L_BB^-1 L_BA L_AA^-1, backward Y_p = -U_BB^-1 U_BA U_AA^-1; pairinv,
// -1 when L_BA / U_BA is absent and the block is zero), made by two GEMM tasks of the
// factor.  Waves 0-3 (group 0) sum row A, waves 4-7 (group 1) row B, each over its own
// row's entries in dependency order (oldest first), independently up to one barrier
// before the diagonal products.  The entries' columns, slots and masks are read 64 at a
// time, one per lane, and taken from their lane (readlane), so no load chain runs
// between two waits; the next nonzero tile is loaded while the current one's column is
// polled; two consecutive entries stored by the same pair task (the usual last two) are
// polled in one spin.  So once the newest dependency lands only its tile products and
// the diagonal products remain on the chain.  A tile whose masks are all zero is
// skipped with no wait, and every thread skips the 16x16 blocks the factor's masks mark
// zero.  CW right-hand sides per pass over the pair.  An odd last row is a pair of its
// own (B absent).
constexpr int NTP = 2 * NT;  // threads of a row-pair task

// one thread's 16 elements of a tile row.  Callers branch around it rather than
// select per element: a select makes the compiler wait for each load in turn.
template <typename T>
__device__ inline void seg16(const T* p, T* v) {
#pragma unroll
    for (int k = 0; k < 16; k++) v[k] = p[k];
}

// Sum over the 4 lanes of a quad (lanes 4i .. 4i+3) in every lane, by two DPP quad
// permutes (lane ^ 1, then lane ^ 2); every lane of the wave must be active.
template <int CTRL>
__device__ inline double dpp_f64(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xF, 0xF, false);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
__device__ inline double quad_sum(double v) {
    v += dpp_f64<0xB1>(v);
    return v + dpp_f64<0x4E>(v);
}

//
// KEEP (FP64 tiles, rows of many entries): a task there is bound by walking its entries, each
// a load of two or four tiles, so the whole next step's tiles and a first read of its x are
// loaded ahead, and the blocks of the diagonal products wait in LDS for want of registers.
// Where rows have few entries the hand-off from pair to pair bounds the pass; it is shorter
// with those blocks in registers.
template <typename T, bool KEEP>
__global__ __launch_bounds__(NTP) void k_trsv_persistent(SolveArgs a) {
    constexpr int VE = 16 / sizeof(T);  // elements of a 16-byte vector
    __shared__ __attribute__((aligned(16))) T kept_d[KEEP ? NTP / 64 : 1][16 / VE][64 * VE];
    __shared__ __attribute__((aligned(16))) T kept_c[KEEP ? NT / 64 : 1][16 / VE][64 * VE];  // group 1
    __shared__ double vec[2][TS];
    __shared__ double rowls[NTP / 64][2 * TS];  // per wave: one column of one or two polled rows
    __shared__ int s_row;
    const int tid = threadIdx.x, g = tid / NT, tg = tid % NT;
    const int r = tg >> 2, kp = tg & 3, lane = tid & 63, w = tid >> 6;
    const int bsh = 4 * (r >> 4) + kp;  // this thread's 16x16 block in a tile's mask
    double* ls = rowls[tid >> 6];
    const T* pool = reinterpret_cast<const T*>(a.pool);
    const int ntask = (a.nbr + 1) / 2 * a.nrhs;
    const int rowoff = r * TS + kp * 16;
    for (;;) {
        if (tid == 0) {
            const int abort = __hip_atomic_load(a.ctrl + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            s_row = abort ? ntask : atomicAdd(a.ctrl, 1);
        }
        __syncthreads();
        const int q = __builtin_amdgcn_readfirstlane(s_row);  // wave-uniform loop control
        if (q >= ntask) break;
        const int qp = q / a.nrhs, c = q - qp * a.nrhs;
        const int p = a.forward ? qp : (a.nbr + 1) / 2 - 1 - qp;
        const double* in = a.in + (int64_t)c * a.ld;
        double* out = a.out + (int64_t)c * a.ld;
        const int I0 = 2 * p, I1 = 2 * p + 1 < a.nbr ? 2 * p + 1 : -1;
        const int IA = a.forward || I1 < 0 ? I0 : I1;
        const int IB = I1 < 0 ? -1 : (a.forward ? I1 : I0);
        const int I = g == 0 ? IA : IB;  // this group's row, -1: none
        const int cpl = g == 1 && IB >= 0 ? a.pairinv[p] : -1;
        // the diagonal inverse (and for row B the coupling block), loaded while the rows
        // wait; a group without a row or coupling block loads A's inverse and ignores it
        T dg[16], cb[16];
        const bool hcb = cpl >= 0;
        seg16(pool + (size_t)a.dinv[I >= 0 ? I : IA] * TE + rowoff, dg);
        seg16(pool + (size_t)(hcb ? cpl : a.dinv[IA]) * TE + rowoff, cb);
        if constexpr (KEEP) {  // each thread its own
#pragma unroll
            for (int k = 0; k < 16; k++) kept_d[w][k / VE][lane * VE + k % VE] = dg[k];
            if (g == 1) {
#pragma unroll
                for (int k = 0; k < 16; k++) kept_c[w - NT / 64][k / VE][lane * VE + k % VE] = cb[k];
            }
        }
        const int e0 = I >= 0 ? a.rowptr[I] : 0, e1 = I >= 0 ? a.rowptr[I + 1] : 0;
        // entries in dependency order: forward e0, e0+1, ..; backward e1-1, e1-2, ..; row
        // B's last one (column IA: forward the largest column, backward the smallest) is
        // the coupling block's
        int n = e1 - e0;
        if (g == 1 && n > 0 && a.col[a.forward ? e1 - 1 : e0] == IA) n--;
        const int64_t rowI = (int64_t)(I >= 0 ? I : 0) * TS;
        double acc = (I >= 0 && kp == 0) ? in[rowI + r] : 0.0;
        for (int base = 0; base < n; base += 64) {  // group-uniform
            const int m = min(64, n - base);
            int Jv = 0, sv = 0;
            uint32_t mv = 0;
            if (lane < m) {
                const int e = a.forward ? e0 + base + lane : e1 - 1 - base - lane;
                Jv = a.col[e];
                sv = a.slot[e];
                mv = a.mask[sv];
            }
            uint64_t rem = __ballot(mv != 0u);  // entries with a nonzero tile, in order
            if (!rem) continue;
            // one step: entry J (tile t0), or J and J1 stored by one pair task (t1),
            // their columns polled in one spin, then the tiles' products
            auto consume = [&](const double* xj, int64_t off, bool poll, bool both, bool b0, bool b1, const T* u0,
                               const T* u1) {
                if (poll) {
                    if (both)  // the whole wave
                        load_row_stored<2>(xj, ls, lane, a, off);
                    else
                        load_row_stored<1>(xj, ls, lane, a);
                }
                // the column into registers first (one batch of LDS reads),
                // then one branch per tile
                double xc[16], s = 0;
#pragma unroll
                for (int k = 0; k < 16; k++) xc[k] = ls[kp * 16 + k];
                if (b0) {
#pragma unroll
                    for (int k = 0; k < 16; k++) s += (double)u0[k] * xc[k];
                }
                if (both) {
#pragma unroll
                    for (int k = 0; k < 16; k++) xc[k] = ls[TS + kp * 16 + k];
                    if (b1) {
#pragma unroll
                        for (int k = 0; k < 16; k++) s += (double)u1[k] * xc[k];
                    }
                }
                __builtin_amdgcn_wave_barrier();  // ls is rewritten for the next column
                acc -= s;
            };
            auto on = [&](int j) { return (__builtin_amdgcn_readlane(mv, j) >> bsh) & 1u; };
            auto tile = [&](int j) { return pool + (size_t)__builtin_amdgcn_readlane(sv, j) * TE + rowoff; };
            if constexpr (KEEP) {
                struct Step {
                    T t0[16], t1[16];  // (an element of a zero block: anything)
                    const double* xj;
                    int64_t off;       // of the second entry's row from the first's
                    unsigned long long u[2];
                    bool both, on0, on1;
                };
                // Every path issues the same loads (a zero block's threads read `idle`, which
                // is in the cache): behind a branch the compiler cannot count them, and waits
                // for them before the step before.
                const T* idle = pool + (size_t)a.dinv[IA] * TE + rowoff;
                auto fetch = [&](Step& s) {
                    const int ja = __builtin_ctzll(rem);
                    rem &= rem - 1;
                    int jb = ja;
                    s.both = false;
                    if (rem) {
                        const int j = __builtin_ctzll(rem);
                        if ((__builtin_amdgcn_readlane(Jv, j) >> 1) == (__builtin_amdgcn_readlane(Jv, ja) >> 1)) {
                            jb = j;
                            s.both = true;
                            rem &= rem - 1;
                        }
                    }
                    s.on0 = on(ja);
                    s.on1 = s.both && on(jb);
                    seg16(s.on0 ? tile(ja) : idle, s.t0);
                    seg16(s.on1 ? tile(jb) : idle, s.t1);
                    const int J = __builtin_amdgcn_readlane(Jv, ja), J1 = __builtin_amdgcn_readlane(Jv, jb);
                    s.xj = out + (int64_t)J * TS;
                    s.off = (int64_t)(J1 - J) * TS;
                    const unsigned long long* x = reinterpret_cast<const unsigned long long*>(s.xj) + lane;
                    s.u[0] = __hip_atomic_load(x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    s.u[1] = __hip_atomic_load(x + s.off, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                };
                auto use = [&](Step& s) {
                    const bool there = !__ballot(s.u[0] == SOLVE_PENDING || s.u[1] == SOLVE_PENDING);
                    if (there) {
                        ls[lane] = __longlong_as_double((long long)s.u[0]);
                        ls[TS + lane] = __longlong_as_double((long long)s.u[1]);
                        __builtin_amdgcn_wave_barrier();
                    }
                    consume(s.xj, s.off, !there, s.both, s.on0, s.on1, s.t0, s.t1);
                };
                Step b0, b1;
                fetch(b0);
                for (;;) {
                    if (!rem) {
                        use(b0);
                        break;
                    }
                    fetch(b1);
                    use(b0);
                    if (!rem) {
                        use(b1);
                        break;
                    }
                    fetch(b0);
                    use(b1);
                }
            } else if constexpr (sizeof(T) == 4) {
                // FP32 tiles: whole steps, the next step's tiles loaded while the
                // current step's columns are polled (a step that takes two entries
                // leaves no tile of its own to load during its wait)
                auto next_step = [&](uint64_t& r, int& ja, int& jb) {
                    if (!r) return false;
                    ja = __builtin_ctzll(r);
                    r &= r - 1;
                    jb = -1;
                    if (r) {
                        const int c = __builtin_ctzll(r);
                        if ((__builtin_amdgcn_readlane(Jv, c) >> 1) == (__builtin_amdgcn_readlane(Jv, ja) >> 1)) {
                            jb = c;
                            r &= r - 1;
                        }
                    }
                    return true;
                };
                T t0[16], t1[16], n0[16], n1[16];  // loaded only where the block is nonzero
                int ja, jb;
                next_step(rem, ja, jb);
                if (on(ja)) seg16(tile(ja), t0);
                if (jb >= 0 && on(jb)) seg16(tile(jb), t1);
                for (;;) {
                    int na = 0, nb = -1;
                    const bool more = next_step(rem, na, nb);
                    if (more && on(na)) seg16(tile(na), n0);
                    if (more && nb >= 0 && on(nb)) seg16(tile(nb), n1);
                    const bool both = jb >= 0;
                    const int J = __builtin_amdgcn_readlane(Jv, ja);
                    const int J1 = __builtin_amdgcn_readlane(Jv, both ? jb : ja);
                    consume(out + (int64_t)J * TS, (int64_t)(J1 - J) * TS, true, both, on(ja), both && on(jb), t0, t1);
                    if (!more) break;
                    ja = na;
                    jb = nb;
#pragma unroll
                    for (int k = 0; k < 16; k++) {
                        t0[k] = n0[k];
                        t1[k] = n1[k];
                    }
                }
            } else {
                // FP64 tiles (no registers for a second step): the next entry's tile
                // is loaded while the current one's column is polled
                int j = __builtin_ctzll(rem);
                rem &= rem - 1;
                T t0[16], t1[16];
                if (on(j)) seg16(tile(j), t0);
                for (;;) {
                    const int J = __builtin_amdgcn_readlane(Jv, j);
                    const bool has1 = rem != 0;
                    const int j1 = has1 ? __builtin_ctzll(rem) : 0;
                    const int J1 = __builtin_amdgcn_readlane(Jv, j1);
                    const bool on1 = has1 && on(j1);
                    if (on1) seg16(tile(j1), t1);  // the next tile, loaded while J's column is polled
                    const bool both = has1 && (J1 >> 1) == (J >> 1);  // stored by one pair task
                    consume(out + (int64_t)J * TS, (int64_t)(J1 - J) * TS, true, both, on(j), both && on1, t0, t1);
                    if (!has1) break;
                    rem &= rem - 1;
                    if (both) {  // both consumed: the one after is loaded now
                        if (!rem) break;
                        j = __builtin_ctzll(rem);
                        rem &= rem - 1;
                        if (on(j)) seg16(tile(j), t0);
                    } else {
                        j = j1;
#pragma unroll
                        for (int k = 0; k < 16; k++) t0[k] = t1[k];
                    }
                }
            }
        }
        acc = quad_sum(acc);
        if (kp == 0) vec[g][r] = acc;
        __syncthreads();
        double v[16], s = 0;
#pragma unroll
        for (int k = 0; k < 16; k++) v[k] = vec[g][kp * 16 + k];
#pragma unroll
        for (int k = 0; k < 16; k++) s += (double)(KEEP ? kept_d[w][k / VE][lane * VE + k % VE] : dg[k]) * v[k];
        if (g == 1 && hcb) {
#pragma unroll
            for (int k = 0; k < 16; k++) v[k] = vec[0][kp * 16 + k];
#pragma unroll
            for (int k = 0; k < 16; k++) s += (double)(KEEP ? kept_c[w - NT / 64][k / VE][lane * VE + k % VE] : cb[k]) * v[k];
        }
        s = quad_sum(s);
        if (kp == 0 && I >= 0)
            __hip_atomic_store(reinterpret_cast<unsigned long long*>(out) + rowI + r,
                               (unsigned long long)__double_as_longlong(s), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();  // vec is reused by the next task
    }
}

// Many right-hand sides (16 and more): the same pair tasks with the sums on MFMA, one task
// per pair and panel of 16 columns (panels are chains of their own: 128 columns are 8
// chains, which fill the chip where one chain of block rows leaves it idle).  Waves 0-3 sum
// row A, waves 4-7 row B, wave w rows 16 (w % 4) .. + 15 of it: the products are formed
// transposed (X^T L^T), so that a lane holds one row and its loads of the right-hand sides
// and stores of x are whole lines.  A step takes two block columns 2P, 2P+1, which one pair
// task stores, and the up to four tiles there (pcol, pslot).  Its x (128 x 16) is read, and
// polled where still pending, once per workgroup, a quarter KB per wave and eighth, and goes
// through LDS; polled by every wave for itself it was 8 times the traffic, and the polls
// of the waiting tasks held up the chain (3D 31^3, 16 columns: 8.0 ms a solve).  The
// tiles' elements come from memory straight into registers: contraction step 4 j + i takes
// k = 16 j + 4 (lane / 16) + i, so that a lane's operands are runs of four consecutive
// elements.  The next step's tiles and x are loaded before the current one is waited for.  x
// is read ahead by ordinary loads while other workgroups store it.  What that rests on: a line
// cached while pending is seen to be pending and polled, and the caches are invalidated at the
// kernel's start, so no older pass's values are read; a value is one aligned 8-byte store and
// lies in one aligned 16-byte part of a lane's load, which does not tear it; and the loaded
// registers, not the memory, are looked at and handed on.  Relaxed atomic loads, 8 bytes each,
// would state that in the language: a random band of 16,384 x 128 columns takes 2.95 ms so,
// 3.12 with wavefront scope and 3.27 with agent scope (FP64; 3D 48^3 x 16 10.0 / 10.2 / 10.6).
constexpr int PC = 16;          // columns of a panel
constexpr int XLD = 2 * TS + 2; // LDS strides of a column: 16-byte reads of 16 columns on distinct banks
constexpr int PLD = TS + 2;

template <typename T>
__global__ __launch_bounds__(NTP) void k_trsm_persistent(SolveArgs a) {
    constexpr int VE = 16 / sizeof(T);  // elements of a 16-byte vector
    __shared__ __attribute__((aligned(16))) double xs[2][PC * XLD];
    __shared__ __attribute__((aligned(16))) double vec[2][PC * PLD];
    __shared__ __attribute__((aligned(16))) T kept_d[NTP / 64][16 / VE][64 * VE];
    __shared__ __attribute__((aligned(16))) T kept_c[NT / 64][16 / VE][64 * VE];  // group 1
    __shared__ int s_row;
    typedef MfmaOp<double> M;
    typedef M::acc_t acc_t;
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), g = w >> 2, rb = w & 3;
    const T* pool = reinterpret_cast<const T*>(a.pool);
    const int strip = (rb * 16 + li) * TS + 4 * lk;  // this lane's row of a tile
    const int npan = (a.nrhs + PC - 1) / PC, npair = (a.nbr + 1) / 2;
    auto load_strip = [&](const T* t, T* v) {
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int i = 0; i < 4; i++) v[4 * j + i] = t[strip + 16 * j + i];
    };
    const int xc = tid >> 5, xr = 4 * (tid & 31);  // this thread's part of a step's x
    struct Step {
        T t0[16], t1[16];  // the strips of the row's tiles in block columns 2P, 2P+1
        double x[4];
        const double* xp;
        uint32_t b0, b1;   // their nonzero 16x16 blocks
    };
    acquire_agent();  // every wave: lines left from earlier passes
    for (;;) {
        if (tid == 0) {
            const int abort = __hip_atomic_load(a.ctrl + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            s_row = abort ? npair * npan : atomicAdd(a.ctrl, 1);
        }
        __syncthreads();
        const int q = __builtin_amdgcn_readfirstlane(s_row);  // wave-uniform loop control
        if (q >= npair * npan) break;
        const int qp = q / npan, c0 = (q - qp * npan) * PC;
        const int p = a.forward ? qp : npair - 1 - qp;
        const int I0 = 2 * p, I1 = 2 * p + 1 < a.nbr ? 2 * p + 1 : -1;
        const int IA = a.forward || I1 < 0 ? I0 : I1;
        const int IB = I1 < 0 ? -1 : (a.forward ? I1 : I0);
        const int I = g == 0 ? IA : IB;  // this group's row, -1: none
        const int cpl = g == 1 && IB >= 0 ? a.pairinv[p] : -1;
        const int idle = a.dinv[IA];  // read in the place of an absent tile
        // the strips of the diagonal inverse and of row B's coupling block, loaded before the
        // waits and kept in LDS, each lane its own
        {
            T dg[16], cb[16];
            load_strip(pool + (size_t)a.dinv[I >= 0 ? I : IA] * TE, dg);
            if (cpl >= 0) load_strip(pool + (size_t)cpl * TE, cb);
#pragma unroll
            for (int k = 0; k < 16; k++) kept_d[w][k / VE][lane * VE + k % VE] = dg[k];
            if (cpl >= 0) {
#pragma unroll
                for (int k = 0; k < 16; k++) kept_c[w - NT / 64][k / VE][lane * VE + k % VE] = cb[k];
            }
        }
        const int e0 = a.prow[p], n = a.prow[p + 1] - e0;
        const int64_t rowI = (int64_t)(I >= 0 ? I : 0) * TS + rb * 16 + li;
        // the right-hand sides wait in the lane's own places of vec
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int c = c0 + M::row(li, lk, r);
            vec[g][M::row(li, lk, r) * PLD + rb * 16 + li] = c < a.nrhs ? a.in[rowI + (int64_t)c * a.ld] : 0.0;
        }
        // a column past nrhs repeats the last one and is not stored
        const double* xcol = a.out + (int64_t)min(c0 + xc, a.nrhs - 1) * a.ld;
        acc_t s0 = {0, 0, 0, 0}, s1 = {0, 0, 0, 0};
        // the pair's steps in dependency order, 64 at a time, one per lane; every wave walks
        // the same ones (a step whose tiles are all zero is skipped, with no wait)
        int base = -64, Pv = 0, sv0 = 0, sv1 = 0;
        uint32_t mv0 = 0, mv1 = 0;
        uint64_t rem = 0;
        auto more = [&]() {
            while (!rem) {
                base += 64;
                if (base >= n) return false;
                bool any = false;
                if (lane < n - base) {
                    const int e = a.forward ? e0 + base + lane : e0 + n - 1 - base - lane;
                    Pv = a.pcol[e];
                    const int4 s = a.pslot[e];
                    const uint32_t m0 = s.x >= 0 ? a.mask[s.x] : 0, m1 = s.y >= 0 ? a.mask[s.y] : 0;
                    const uint32_t m2 = s.z >= 0 ? a.mask[s.z] : 0, m3 = s.w >= 0 ? a.mask[s.w] : 0;
                    any = (m0 | m1 | m2 | m3) != 0;
                    const bool odd = (I & 1) != 0;
                    sv0 = odd ? s.z : s.x;
                    sv1 = odd ? s.w : s.y;
                    mv0 = I < 0 ? 0 : (odd ? m2 : m0) >> (4 * rb);
                    mv1 = I < 0 ? 0 : (odd ? m3 : m1) >> (4 * rb);
                }
                rem = __ballot(any);
            }
            return true;
        };
        // every path issues the same loads, so that waits can count them
        auto fetch = [&](Step& s) {
            const int j = __builtin_ctzll(rem);
            rem &= rem - 1;
            s.b0 = __builtin_amdgcn_readlane(mv0, j) & 0xFu;
            s.b1 = __builtin_amdgcn_readlane(mv1, j) & 0xFu;
            const int P = __builtin_amdgcn_readlane(Pv, j);
            const int t0 = __builtin_amdgcn_readlane(sv0, j), t1 = __builtin_amdgcn_readlane(sv1, j);
            load_strip(pool + (size_t)(s.b0 ? t0 : idle) * TE, s.t0);
            load_strip(pool + (size_t)(s.b1 ? t1 : idle) * TE, s.t1);
            // (an odd last block row has no second: its own is read in its place)
            s.xp = xcol + (int64_t)2 * P * TS + (2 * P + 1 < a.nbr ? xr : xr & (TS - 1));
#pragma unroll
            for (int i = 0; i < 4; i++) s.x[i] = s.xp[i];
        };
        auto pending = [&](const Step& s) {
            bool pend = false;
#pragma unroll
            for (int i = 0; i < 4; i++) pend |= (unsigned long long)__double_as_longlong(s.x[i]) == SOLVE_PENDING;
            return __ballot(pend) != 0;
        };
        int buf = 0;
        auto consume = [&](Step& s) {
            if (pending(s)) {
                const unsigned long long* u = reinterpret_cast<const unsigned long long*>(s.xp);
                const long long t0 = wall_clock64();
                for (int spin = 1;; spin++) {
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        s.x[i] = __longlong_as_double(
                            (long long)__hip_atomic_load(u + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
                    if (!pending(s)) break;
                    if (spin % SOLVE_SPIN_CHECK == 0 &&
                        (__hip_atomic_load(a.ctrl + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ||
                         wall_clock64() - t0 > SOLVE_SPIN_LIMIT)) {
                        raise_abort(a);
#pragma unroll
                        for (int i = 0; i < 4; i++) s.x[i] = 0.0;
                        break;
                    }
                    __builtin_amdgcn_s_sleep(1);
                }
            }
            // two buffers: every wave has read this one two steps ago, before the last barrier
            double* xb = xs[buf];
            buf ^= 1;
#pragma unroll
            for (int i = 0; i < 4; i++) xb[xc * XLD + xr + i] = s.x[i];
            __syncthreads();
            auto mul = [&](const T* t, uint32_t bits, const double* x) {
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    if (!((bits >> j) & 1u)) continue;  // a zero block
                    double v[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) v[i] = x[li * XLD + 16 * j + 4 * lk + i];
                    s0 = M::mma(v[0], (double)t[4 * j], s0);
                    s1 = M::mma(v[1], (double)t[4 * j + 1], s1);
                    s0 = M::mma(v[2], (double)t[4 * j + 2], s0);
                    s1 = M::mma(v[3], (double)t[4 * j + 3], s1);
                }
            };
            mul(s.t0, s.b0, xb);
            mul(s.t1, s.b1, xb + TS);
        };
        Step b0, b1;
        if (more()) {
            fetch(b0);
            for (;;) {
                if (!more()) {
                    consume(b0);
                    break;
                }
                fetch(b1);
                consume(b0);
                if (!more()) {
                    consume(b1);
                    break;
                }
                fetch(b0);
                consume(b1);
            }
        }
        // r = b - sum, in LDS by columns for the diagonal products
#pragma unroll
        for (int r = 0; r < 4; r++) vec[g][M::row(li, lk, r) * PLD + rb * 16 + li] -= s0[r] + s1[r];
        __syncthreads();
        s0 = acc_t{0, 0, 0, 0};
        s1 = acc_t{0, 0, 0, 0};
        auto diag = [&](const double* v, const T* kept) {
#pragma unroll
            for (int k = 0; k < 16; k++) {
                const double x = v[li * PLD + 4 * lk + 16 * (k / 4) + k % 4];
                const double d = (double)kept[(k / VE) * 64 * VE + lane * VE + k % VE];
                if (k % 2) s1 = M::mma(x, d, s1);
                else s0 = M::mma(x, d, s0);
            }
        };
        diag(vec[g], &kept_d[w][0][0]);
        if (cpl >= 0) diag(vec[0], &kept_c[w - NT / 64][0][0]);  // wave-uniform
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int c = c0 + M::row(li, lk, r);
            // a NaN is stored quiet: never the pending marker
            if (I >= 0 && c < a.nrhs)
                __hip_atomic_store(reinterpret_cast<unsigned long long*>(a.out) + rowI + (int64_t)c * a.ld,
                                   (unsigned long long)__double_as_longlong(__builtin_canonicalize(s0[r] + s1[r])),
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();  // vec and xs are reused by the next task
    }
}

// out = diag(L) y over the padded rows, every column: the forward result as the
// reference's lowerSolver leaves it in its right-hand side, b_i = l_ii y_i (for a
// unit-diagonal L that is y itself).
template <typename T>
__global__ void k_scale_by_ldiag(const T* __restrict__ pool, const int32_t* __restrict__ l_diag,
                                 const double* __restrict__ y, double* __restrict__ out, int64_t ld, int64_t n) {
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = e % ld;
        const int64_t i = r / TS, q = r % TS;
        out[e] = (double)pool[(size_t)l_diag[i] * TE + q * TS + q] * y[e];
    }
}

namespace {

#define HIP_TRY(ctx, expr)                                       \
    do {                                                         \
        int _rc = check_hip((ctx), (expr), #expr);               \
        if (_rc != SOGL_OK) return _rc;                          \
    } while (0)

bool whole_steps_ahead(const Factor* f) {
    return (1 - f->zero_blocks) * (double)f->solve_entries >= KEEP_TILES * (double)f->solve_rows;
}

template <typename T>
int launch_pass(Context* c, Factor* f, const SolveWork& w, bool mfma, bool forward, const double* in, double* out,
                int nrhs) {
    SolveArgs a{};
    a.pool = f->pool.p;
    a.rowptr = (const int32_t*)(forward ? f->l_rowptr.p : f->u_rowptr.p);
    a.col = (const int32_t*)(forward ? f->l_col.p : f->u_col.p);
    a.slot = (const int32_t*)(forward ? f->l_slot.p : f->u_slot.p);
    a.dinv = (const int32_t*)(forward ? f->linv_d.p : f->uinv_d.p);
    a.in = in;
    a.out = out;
    a.ld = (int64_t)f->block_rows * TS;
    a.nrhs = nrhs;
    a.nbr = f->block_rows;
    a.forward = forward ? 1 : 0;
    a.ctrl = w.ctrl + (forward ? 0 : 4);
    a.mask = (const uint32_t*)f->mask_d.p;
    a.prow = (const int32_t*)(forward ? f->lstep_ptr.p : f->ustep_ptr.p);
    a.pcol = (const int32_t*)(forward ? f->lstep_col.p : f->ustep_col.p);
    a.pslot = (const int4*)(forward ? f->lstep_slot.p : f->ustep_slot.p);
    a.pairinv = (const int32_t*)(forward ? f->pairx_d.p : f->pairy_d.p);
    const int64_t ntask = (int64_t)((a.nbr + 1) / 2) * (mfma ? (nrhs + PC - 1) / PC : nrhs);
    auto kern = mfma ? k_trsm_persistent<T> : k_trsv_persistent<T, false>;
    if constexpr (sizeof(T) == 8)
        if (!mfma && whole_steps_ahead(f)) kern = k_trsv_persistent<T, true>;
    int per_cu = 0;
    HIP_TRY(c, hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, NTP, 0));
    if (per_cu < 1) per_cu = 1;
    const int grid = (int)std::max<int64_t>(1, std::min<int64_t>(ntask, (int64_t)c->num_cu * per_cu));
    hipLaunchKernelGGL(kern, dim3(grid), dim3(NTP), 0, c->stream, a);
    HIP_TRY(c, hipGetLastError());
    return SOGL_OK;
}

}  // namespace

// Both passes over nrhs columns, enqueued on the context stream between the events ev0 and
// ev1.  d_x may be d_b: the forward pass reads b and writes y, and an x that shares memory
// with b is marked pending only after it (one launch more).  solve_finish waits and looks at
// the outcome.
int solve_launch(Context* c, Factor* f, const SolveWork& w, const double* d_b, double* d_x, int nrhs) {
    const int R = f->block_rows;
    int rc;
    HIP_TRY(c, hipEventRecord(c->ev0, c->stream));
    const int64_t ld = (int64_t)R * TS;
    const bool mfma = nrhs >= TRSM_MIN_RHS;
    const uintptr_t b0 = (uintptr_t)d_b, x0 = (uintptr_t)d_x, bytes = (uintptr_t)ld * (uintptr_t)nrhs * sizeof(double);
    const bool shared = b0 < x0 + bytes && x0 < b0 + bytes;
    for (int c0 = 0; c0 < nrhs; c0 += MAX_RHS) {
        const int m = std::min(MAX_RHS, nrhs - c0);
        const int64_t off = (int64_t)c0 * ld, n = ld * m;
        const unsigned grid = (unsigned)std::max<int64_t>(1, std::min<int64_t>((n + 255) / 256, 2048));
        auto pass = [&](bool forward, const double* in, double* out) {
            return f->elem == 8 ? launch_pass<double>(c, f, w, mfma, forward, in, out, m)
                                : launch_pass<float>(c, f, w, mfma, forward, in, out, m);
        };
        hipLaunchKernelGGL(k_solve_begin, dim3(grid), dim3(256), 0, c->stream, w.ctrl, c0 == 0, w.y + off,
                           shared ? nullptr : d_x + off, n);
        if ((rc = pass(true, d_b + off, w.y + off))) return rc;
        if (shared) hipLaunchKernelGGL(k_fill_pending, dim3(grid), dim3(256), 0, c->stream, d_x + off, n);
        if ((rc = pass(false, w.y + off, d_x + off))) return rc;
    }
    HIP_TRY(c, hipEventRecord(c->ev1, c->stream));
    return SOGL_OK;
}

int solve_timeout(Context* c) {
    return set_error(c, SOGL_ERR_TIMEOUT, "solve: a dependency wait exceeded its bound");
}

int solve_finish(Context* c, Factor* f, const SolveWork& w) {
    HIP_TRY(c, hipEventSynchronize(c->ev1));
    float ms = 0;
    HIP_TRY(c, hipEventElapsedTime(&ms, c->ev0, c->ev1));
    f->solve_ms = ms;
    int ctrl[SOLVE_CTRL_WORDS];
    HIP_TRY(c, hipMemcpy(ctrl, w.ctrl, sizeof(ctrl), hipMemcpyDeviceToHost));
    return ctrl[1] || ctrl[5] ? solve_timeout(c) : SOGL_OK;
}

int solve_core(Context* c, Factor* f, const SolveWork& w, const double* d_b, double* d_x, int nrhs) {
    const int rc = solve_launch(c, f, w, d_b, d_x, nrhs);
    return rc ? rc : solve_finish(c, f, w);
}

// With the factor's own control words (allocated on first use) and y.
int solve_work(Context* c, Factor* f, SolveWork& w) {
    int rc;
    if ((rc = dev_alloc(c, f->solve_ctrl, SOLVE_CTRL_WORDS * sizeof(int), "solve control"))) return rc;
    w = SolveWork{(double*)f->vec_y.p, (int*)f->solve_ctrl.p};
    return SOGL_OK;
}

int solve_device(Context* c, Factor* f, const double* d_b, double* d_x, int nrhs) {
    SolveWork w;
    int rc;
    if ((rc = solve_work(c, f, w))) return rc;
    return solve_core(c, f, w, d_b, d_x, nrhs);
}

int ensure_vectors(Context* c, Factor* f, int nrhs) {
    const size_t need = (size_t)f->block_rows * TS * (size_t)nrhs;
    if (f->vec_cap >= need) return SOGL_OK;
    f->vec_cap = 0;  // a growth that fails leaves a vector freed
    int rc;
    if ((rc = dev_alloc(c, f->vec_b, need * 8, "rhs")) || (rc = dev_alloc(c, f->vec_x, need * 8, "x")) ||
        (rc = dev_alloc(c, f->vec_y, need * 8, "y")))
        return rc;
    f->vec_cap = need;
    return SOGL_OK;
}

}  // namespace sogl_dev

using namespace sogl_dev;

extern "C" int sogl_solve(sogl_ctx* x, int32_t factor_id, const double* bp, double* xp, double* y,
                          int32_t nrhs) {
    if (!x || !bp || !xp || nrhs <= 0) return set_error(x ? &x->c : nullptr, SOGL_ERR_ARG, "bad argument");
    Context* c = &x->c;
    std::lock_guard<std::mutex> g(c->mu);
    Factor* f = find_factor(c, factor_id);
    if (!f) return set_error(c, SOGL_ERR_ARG, "unknown factor id");
    HIP_TRY(c, hipSetDevice(c->device));
    int rc;
    if ((rc = ensure_vectors(c, f, nrhs))) return rc;
    const size_t bytes = (size_t)f->block_rows * TS * nrhs * 8;
    HIP_TRY(c, hipMemcpyAsync(f->vec_b.p, bp, bytes, hipMemcpyHostToDevice, c->stream));
    if ((rc = solve_device(c, f, (const double*)f->vec_b.p, (double*)f->vec_x.p, nrhs)))
        return rc;
    HIP_TRY(c, hipMemcpyAsync(xp, f->vec_x.p, bytes, hipMemcpyDeviceToHost, c->stream));
    if (y && f->llt) {
        // L L^T: the reference's right-hand side ends as diag(L) y (the input b in
        // vec_b is no longer needed)
        const int64_t ld = (int64_t)f->block_rows * TS, n = ld * nrhs;
        const unsigned grid = (unsigned)std::min<int64_t>((n + 255) / 256, 4096);
        if (f->elem == 8)
            hipLaunchKernelGGL(k_scale_by_ldiag<double>, dim3(grid), dim3(256), 0, c->stream, (const double*)f->pool.p,
                               (const int32_t*)f->l_diag_d.p, (const double*)f->vec_y.p, (double*)f->vec_b.p, ld, n);
        else
            hipLaunchKernelGGL(k_scale_by_ldiag<float>, dim3(grid), dim3(256), 0, c->stream, (const float*)f->pool.p,
                               (const int32_t*)f->l_diag_d.p, (const double*)f->vec_y.p, (double*)f->vec_b.p, ld, n);
        HIP_TRY(c, hipGetLastError());
        HIP_TRY(c, hipMemcpyAsync(y, f->vec_b.p, bytes, hipMemcpyDeviceToHost, c->stream));
    } else if (y) {
        HIP_TRY(c, hipMemcpyAsync(y, f->vec_y.p, bytes, hipMemcpyDeviceToHost, c->stream));
    }
    HIP_TRY(c, hipStreamSynchronize(c->stream));
    return SOGL_OK;
}

extern "C" int sogl_solve_device(sogl_ctx* x, int32_t factor_id, const double* d_bp, double* d_xp,
                                 int32_t nrhs) {
    if (!x || !d_bp || !d_xp || nrhs <= 0) return set_error(x ? &x->c : nullptr, SOGL_ERR_ARG, "bad argument");
    Context* c = &x->c;
    std::lock_guard<std::mutex> g(c->mu);
    Factor* f = find_factor(c, factor_id);
    if (!f) return set_error(c, SOGL_ERR_ARG, "unknown factor id");
    HIP_TRY(c, hipSetDevice(c->device));
    int rc;
    if ((rc = ensure_vectors(c, f, nrhs))) return rc;
    return solve_device(c, f, d_bp, d_xp, nrhs);
}

// ------------------------------------------------------------------ solve without allocation
// The solve's work buffers (y, control) in one fixed array per GPU, for callers
// that cannot allocate device memory.  In host code `scratch` names a host-side stand-in
// for the array, never its device address: the address each GPU gives its own copy is
// looked up once per device, when the first context on it is created, and only that
// address is handed to kernels and copies.
namespace sogl_dev {
namespace {

static __device__ __align__(256) unsigned char scratch[SOGL_NOALLOC_SCRATCH_BYTES];

constexpr int SCRATCH_MAX_DEVICES = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[SCRATCH_MAX_DEVICES];       // device address of `scratch` on each GPU
hipError_t g_scratch_rc[SCRATCH_MAX_DEVICES];   // result of the lookup (valid when looked up)
bool g_scratch_done[SCRATCH_MAX_DEVICES];

constexpr size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

// Layout inside the array: control words, 4 bytes per block row that sogl.h counts in (not
// used any more; what fits stays the same), then y.
struct ScratchLayout {
    size_t ctrl, y, end;
};
ScratchLayout scratch_layout(int32_t rows, int32_t nrhs) {
    ScratchLayout l;
    l.ctrl = 0;
    l.y = 256 + align256((size_t)rows * 4);
    l.end = l.y + (size_t)rows * TS * (size_t)nrhs * 8;
    return l;
}

}  // namespace

// Looks up this GPU's address of `scratch`, once per device (the device is current).
void noalloc_scratch_init(int device) {
    if (device < 0 || device >= SCRATCH_MAX_DEVICES) return;
    std::lock_guard<std::mutex> g(g_scratch_mu);
    if (g_scratch_done[device]) return;
    void* p = nullptr;
    g_scratch_rc[device] = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (g_scratch_rc[device] != hipSuccess) {
        (void)hipGetLastError();
        p = nullptr;
    }
    g_scratch_ptr[device] = p;
    g_scratch_done[device] = true;
}

}  // namespace sogl_dev

extern "C" int sogl_solve_device_noalloc(sogl_ctx* x, int32_t factor_id, const double* d_bp, double* d_xp,
                                         int32_t nrhs) {
    if (!x || !d_bp || !d_xp || nrhs <= 0) return set_error(x ? &x->c : nullptr, SOGL_ERR_ARG, "bad argument");
    Context* c = &x->c;
    std::lock_guard<std::mutex> g(c->mu);
    Factor* f = find_factor(c, factor_id);
    if (!f) return set_error(c, SOGL_ERR_ARG, "unknown factor id");
    const int dev = c->device;
    void* base = nullptr;
    hipError_t lookup = hipErrorNotInitialized;
    {
        std::lock_guard<std::mutex> sg(g_scratch_mu);
        if (dev >= 0 && dev < SCRATCH_MAX_DEVICES && g_scratch_done[dev]) {
            base = g_scratch_ptr[dev];
            lookup = g_scratch_rc[dev];
        }
    }
    if (!base)
        return set_error(c, SOGL_ERR_DEVICE, std::string("solve without allocation: no scratch address for this "
                                                         "device: ") + hipGetErrorString(lookup));
    const ScratchLayout l = scratch_layout(f->block_rows, nrhs);
    if (l.end > (size_t)SOGL_NOALLOC_SCRATCH_BYTES)
        return set_error(c, SOGL_ERR_ARG, "solve without allocation: " + std::to_string(f->block_rows) +
                                              " block rows x " + std::to_string(nrhs) + " right-hand sides need " +
                                              std::to_string(l.end) + " bytes of scratch, more than its " +
                                              std::to_string((size_t)SOGL_NOALLOC_SCRATCH_BYTES));
    HIP_TRY(c, hipSetDevice(dev));
    char* s = (char*)base;
    const SolveWork w{(double*)(s + l.y), (int*)(s + l.ctrl)};
    return solve_core(c, f, w, d_bp, d_xp, nrhs);
}
