// The unit ops of a plan's factorisation in tile-column order: for every block row k
//     S_kk = A_kk - sum_{j<k} L_kj U_jk,   lu(S_kk) -> L_kk, U_kk (and their inverses)
//     L_ik = (A_ik - sum_{j<k} L_ij U_jk) U_kk^-1,   U_ki = L_kk^-1 (A_ki - sum_j L_kj U_ji)
// (L L^T: L_ik = (A_ik - sum_j L_ij L_kj^T) L_kk^-T).  The factor is the one the plan's own
// op list makes (L and U are unique; the sums are grouped differently), tile for tile in
// the plan's ids.  The plan's list follows the reference's recursion over 2x2 blocks
// (BlockPlanner.cpp:865-1092), which multiplies by the explicit inverses of growing
// diagonal blocks.  Both are bound by the chain of tasks through the diagonal: there 4.9
// tasks per block row on the critical path (C2; C5 4.7), here 3 (the sum, the lu, a
// panel), and 10 to 50% fewer tile products.  Factor alone, plan's list -> this one, same
// box: C5 (2D convection-diffusion 1000^2) FP32 348 -> 285 ms; C2 (3D 48^3) FP32 51.9 ->
// 37.8, FP64 79.2 -> 50.7; symmetric 3D 37^3 FP64 38.1 -> 25.9; C3 (random band, n =
// 16,384) FP32 41.4 -> 38.3; 2D 128^2 FP64 8.4 -> 7.4.
#pragma once

#include <algorithm>
#include <cstdint>
#include <utility>
#include <vector>

#include "../../../include/sogl.h"

namespace sogl_dev {

// Block columns per partial sum.  A GEMM task holds its workgroup while it waits for its last
// update, and one that starts late multiplies all of them on the spot: parts bound that
// work, and are made, as tasks of their own, as soon as their operands are.  A part of tile
// (i, k) begins where i + k + j is a multiple of SUM_PAIRS (an update by that column j there
// is), so that the parts of a block row's tiles do not all become ready at once: a dense sum
// has parts of SUM_PAIRS updates, a sparse one more or fewer in each.  Measured: C3 FP32 (sums of up to 255) 48.8 ms whole, 37.3 in
// parts of 64, 38.3 of 32, 45.4 of 16; C2 FP32 (up to 27) 39.2, 39.2, 37.8, 35.4.
constexpr int32_t SUM_PAIRS = 32;

struct TileOrderOps {
    std::vector<sogl_op> ops;
    int32_t n_ids = 0;
};

// The list above for a plan's description (its input tiles at block in_bi, in_bj).  False
// where the description is not the factorisation of one matrix in closed form -- a tile of
// the inputs or an update outside the L / U lists, a missing diagonal tile, an id used
// twice -- which keeps its own op list.
inline bool tile_order_ops(const sogl_factor_desc* d, const int32_t* in_bi, const int32_t* in_bj, TileOrderOps& out) {
    typedef std::pair<int32_t, int32_t> Ent;  // (block row or column, tile id)
    const int32_t R = d->block_rows;
    bool llt = false, lu = false;
    for (int64_t k = 0; k < d->n_ops; k++) {
        llt |= d->ops[k].op == SOGL_OP_LLT;
        lu |= d->ops[k].op == SOGL_OP_LU;
    }
    if (llt == lu || (llt && d->n_u)) return false;
    std::vector<char> used((size_t)d->n_ids, 0);
    auto take = [&](int32_t id) {
        if (id <= 0 || id >= d->n_ids || used[(size_t)id]) return false;
        used[(size_t)id] = 1;
        return true;
    };
    std::vector<std::vector<Ent>> lrow((size_t)R), lcol((size_t)R), urow((size_t)R), ucol((size_t)R);
    std::vector<std::vector<Ent>> arow((size_t)R);
    std::vector<int32_t> ldiag((size_t)R, 0), udiag((size_t)R, 0);
    for (int64_t k = 0; k < d->n_inputs; k++) {
        if (!take(d->input_ids[k]) || in_bi[k] < 0 || in_bi[k] >= R || in_bj[k] < 0 || in_bj[k] >= R) return false;
        if (llt && in_bi[k] < in_bj[k]) continue;  // L L^T reads the lower triangle
        arow[(size_t)in_bi[k]].push_back({in_bj[k], d->input_ids[k]});
    }
    for (int which = 0; which < 2; which++) {
        const int64_t cnt = which == 0 ? d->n_l : d->n_u;
        const int32_t* bi = which == 0 ? d->l_bi : d->u_bi;
        const int32_t* bj = which == 0 ? d->l_bj : d->u_bj;
        const int32_t* id = which == 0 ? d->l_ids : d->u_ids;
        for (int64_t k = 0; k < cnt; k++) {
            const int32_t i = bi[k], j = bj[k];
            if (i < 0 || i >= R || j < 0 || j >= R || !take(id[k])) return false;
            if (i == j) {
                (which == 0 ? ldiag : udiag)[(size_t)i] = id[k];
            } else if (which == 0) {
                if (i < j) return false;
                lrow[(size_t)i].push_back({j, id[k]});
                lcol[(size_t)j].push_back({i, id[k]});
            } else {
                if (i > j) return false;
                urow[(size_t)i].push_back({j, id[k]});
                ucol[(size_t)j].push_back({i, id[k]});
            }
        }
    }
    int64_t want = 0, found = 0;  // updates L_ij U_jk, and those that land in a listed tile
    for (int32_t k = 0; k < R; k++) {
        if (!ldiag[(size_t)k] || (!llt && !udiag[(size_t)k])) return false;
        for (auto* v : {&lrow, &lcol, &urow, &ucol, &arow}) {
            auto& e = (*v)[(size_t)k];
            std::sort(e.begin(), e.end());
            for (size_t q = 1; q < e.size(); q++)
                if (e[q].first == e[q - 1].first) return false;
        }
        const int64_t nl = (int64_t)lcol[(size_t)k].size();
        want += llt ? nl * (nl + 1) / 2 : nl * (int64_t)urow[(size_t)k].size();
    }
    if (want > (int64_t)INT32_MAX / 2) return false;
    out.ops.clear();
    out.ops.reserve((size_t)(want + 3 * (d->n_l + d->n_u) + 3 * (int64_t)R));
    int32_t next = d->n_ids, seq = 0, n_in = 0;
    auto emit = [&](int32_t code, int32_t src, int32_t src2, int32_t res, int32_t res2, int32_t stage) {
        out.ops.push_back(sogl_op{src, src2, code, res, res2, stage, seq++, 0});
    };
    // S_ik: the input tile (i, k) less its updates by block columns before min(i, k); 0: none
    // (products at stage st, part p's sum at st + 1 + p; most: the parts of the longest sum so far)
    int32_t most = 0;
    auto sum = [&](int32_t i, int32_t k, int32_t st) {
        int32_t a = 0;
        const auto& ar = arow[(size_t)i];
        auto it = std::lower_bound(ar.begin(), ar.end(), Ent{k, 0});
        if (it != ar.end() && it->first == k) {
            a = it->second;
            n_in++;
        }
        const int32_t m = std::min(i, k);
        const auto& lr = lrow[(size_t)i];
        const auto& uc = llt ? lrow[(size_t)k] : ucol[(size_t)k];
        // a sum of more than SUM_PAIRS updates is made in parts, each adding to the one before
        int32_t acc = 0, part = 0;
        auto close = [&]() {
            const int32_t r = next++;
            emit(SOGL_OP_SUB, acc, a, r, 0, st + 1 + part++);
            a = r;
            acc = 0;
        };
        for (size_t p = 0, q = 0; p < lr.size() && q < uc.size() && lr[p].first < m && uc[q].first < m;) {
            if (lr[p].first < uc[q].first) p++;
            else if (lr[p].first > uc[q].first) q++;
            else {
                const int32_t j = lr[p].first;
                // the diagonal's last update, by the block column before it, is a part of its
                // own: the lu / llt of that column runs it (diagonal chains in factor.hip)
                if (acc && ((i + k + j) % SUM_PAIRS == 0 || (i == k && j == k - 1))) close();
                if (!acc) acc = next++;
                emit(llt ? SOGL_OP_MULT : SOGL_OP_MUL, lr[p].second, uc[q].second, acc, 0, st);
                found++;
                p++, q++;
            }
        }
        if (acc) close();
        most = std::max(most, part);
        return a;
    };
    // an op that follows the sums of its step: its stage, counted from the end of theirs, is made
    // absolute when the step's sums are all there
    std::vector<size_t> after;
    auto emit_after = [&](int32_t code, int32_t src, int32_t src2, int32_t res, int32_t res2, int32_t stage) {
        after.push_back(out.ops.size());
        emit(code, src, src2, res, res2, stage);
    };
    int32_t stage = 1;
    for (int32_t k = 0; k < R; k++) {
        const auto& lc = lcol[(size_t)k];
        const auto& ur = urow[(size_t)k];
        std::vector<int32_t> s_l(lc.size(), -1), s_u(ur.size(), -1);
        most = 0;
        after.clear();
        const int32_t x = next++, z = llt ? 0 : next++;
        bool ok = true;
        auto panel_l = [&](size_t q) {
            if (s_l[q] < 0) s_l[q] = sum(lc[q].first, k, stage);
            ok &= s_l[q] != 0;  // else: a listed tile that nothing fills
            emit_after(llt ? SOGL_OP_MULT : SOGL_OP_MUL, s_l[q], llt ? x : z, lc[q].second, 0, 2);
        };
        auto panel_u = [&](size_t q) {
            if (s_u[q] < 0) s_u[q] = sum(k, ur[q].first, stage);
            ok &= s_u[q] != 0;
            emit_after(SOGL_OP_MUL, x, s_u[q], ur[q].second, 0, 2);
        };
        // the sums of the two panels next to the diagonal come before the diagonal's own:
        // the lu that runs those panels itself then finds them handed out earlier
        if (!lc.empty() && lc[0].first == k + 1) s_l[0] = sum(k + 1, k, stage);
        if (!ur.empty() && ur[0].first == k + 1) s_u[0] = sum(k, k + 1, stage);
        const int32_t s = sum(k, k, stage);
        if (!s) return false;
        emit_after(llt ? SOGL_OP_LLT : SOGL_OP_LU, s, 0, ldiag[(size_t)k], llt ? 0 : udiag[(size_t)k], 0);
        emit_after(SOGL_OP_LOWER_INV, ldiag[(size_t)k], 0, x, 0, 1);
        if (!llt) emit_after(SOGL_OP_UPPER_INV, udiag[(size_t)k], 0, z, 0, 1);
        for (size_t q = 0; q < std::max(lc.size(), ur.size()); q++) {
            if (q < lc.size()) panel_l(q);
            if (q < ur.size()) panel_u(q);
        }
        if (!ok) return false;
        stage += most + 1;
        for (size_t o : after) out.ops[o].stage += stage;
        stage += 3;
    }
    int64_t inputs = 0;
    for (const auto& e : arow) inputs += (int64_t)e.size();
    if (found != want || n_in != inputs) return false;  // an update or an input outside the lists
    out.n_ids = next;
    return true;
}

}  // namespace sogl_dev
