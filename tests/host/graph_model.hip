// Host-only build of the executor's graph code (no device code, no GPU) with an untimed model of
// the persistent kernels' queue: which tasks a given number of workgroups can finish.
#include "../../sparse-operator-graph-lu_amd/csrc/device/factor.hip"
#include "no_device.h"

using namespace sogl_dev;

namespace sogl_dev {
void noalloc_scratch_init(int) {}
}

namespace {

struct Graph {
    Factor f;
    HostGraph hg;
    TileOrderOps to;
    sogl_factor_desc d;
};

int build(const sogl_factor_desc* desc, const int32_t* in_bi, const int32_t* in_bj, Graph& g) {
    g.d = *desc;
    if (in_bi) {
        if (!tile_order_ops(desc, in_bi, in_bj, g.to)) return -1;
        g.d.ops = g.to.ops.data();
        g.d.n_ops = (int64_t)g.to.ops.size();
        g.d.n_ids = g.to.n_ids;
        g.f.tile_order = true;
    }
    g.f.precision = g.d.precision;
    g.f.elem = g.d.precision == SOGL_FP64 ? 8 : 4;
    g.f.n_inputs = g.d.n_inputs;
    g.f.absorb_panels = true;
    return build_host_graph(nullptr, &g.d, &g.f, g.hg);
}

struct Model {
    Factor& f;
    HostGraph& hg;
    bool chains;  // a diagonal chain's step inside its lu; else its tasks come from the queue
    int claims;   // dynamic chaining
    const std::vector<int32_t>& queue;
    std::vector<int32_t> maker;
    std::vector<char> done, claimed;
    size_t taken = 0, finished = 0;
    struct Wg {
        int32_t t = -1, mode = 0, pend = -1;
        std::deque<int32_t> ring;
    };

    Model(Graph& g, bool chains_, int claims_)
        : f(g.f), hg(g.hg), chains(chains_), claims(claims_), queue(chains || !f.n_diag_chains ? f.queue : f.queue_all) {
        maker.assign((size_t)f.n_slots, -1);
        for (size_t t = 0; t < f.tasks.size(); t++)
            for (int32_t o : {f.tasks[t].out0, f.tasks[t].out1, f.tasks[t].out2, f.tasks[t].out3})
                if (o >= 0) maker[(size_t)o] = (int32_t)t;
        done.assign(f.tasks.size(), 0);
        claimed.assign(f.tasks.size(), 0);
    }
    bool there(int32_t slot) const { return slot < 0 || maker[(size_t)slot] < 0 || done[(size_t)maker[(size_t)slot]]; }
    bool ready(int32_t t, int32_t but = -1) const {  // every operand there, but those that task `but` makes
        const DevTask& k = f.tasks[(size_t)t];
        for (int32_t q = k.dep_begin; q < k.dep_begin + k.dep_count; q++) {
            const int32_t s = hg.deps[(size_t)q];
            if (!(but >= 0 && maker[(size_t)s] == but) && !there(s)) return false;
        }
        return true;
    }
    void finish(int32_t t) {
        done[(size_t)t] = 1;
        finished++;
    }
    // One turn of a workgroup; false: it waits (or the queue is empty).
    bool turn(Wg& w) {
        if (w.t < 0) {
            if (taken >= queue.size()) return false;
            w.t = queue[taken++];
            w.mode = 0;
            if (claimed[(size_t)w.t]) w.t = -1;
            return true;
        }
        const DevTask& k = f.tasks[(size_t)w.t];
        if (claimed[(size_t)w.t] && w.mode == 0) return w.t = -1, true;  // dropped
        if (w.mode != 1 && !ready(w.t)) return false;
        if (chains && k.dia >= 0) {  // the lu waits for what its panels and the update read as well
            const DevTask& d = f.tasks[(size_t)k.dia];
            for (int32_t p : {k.pan_l, k.pan_u})
                if (p >= 0 && !ready(p, w.t)) return false;
            if (!there(d.add)) return false;
            for (int32_t p : {w.t, k.pan_l, k.pan_u, k.dia})
                if (p >= 0) finish(p);
            w.t = d.next;
            w.mode = 1;
            return true;
        }
        finish(w.t);
        if (k.next < 0)
            for (int32_t q = k.chk_begin, n = 0; claims && q < k.chk_begin + k.chk_count && n < claims; q++) {
                const int32_t c = f.chk[(size_t)q].task;
                if (claimed[(size_t)c] || done[(size_t)c] || !ready(c)) continue;
                claimed[(size_t)c] = 1;
                w.ring.push_back(c);
                n++;
            }
        auto go = [&](int32_t t, int mode) { w.t = t, w.mode = mode; };
        if (k.next >= 0) go(k.next, 1);
        else if (k.dia < 0 && (k.pan_l >= 0 || k.pan_u >= 0)) {
            go(k.pan_l >= 0 ? k.pan_l : k.pan_u, 3);
            w.pend = k.pan_l >= 0 ? k.pan_u : -1;
        } else if (w.pend >= 0) go(w.pend, 3), w.pend = -1;
        else if (!w.ring.empty()) go(w.ring.front(), 2), w.ring.pop_front();
        else w.t = -1;
        return true;
    }
    size_t run(int workgroups) {
        std::vector<Wg> wg((size_t)workgroups);
        for (bool any = true; any;) {
            any = false;
            for (Wg& w : wg)
                while (turn(w)) any = true;
        }
        return finished;
    }
};

}  // namespace

// out: tasks, those that `workgroups` workgroups finish, diagonal chains' steps, chains
extern "C" int model(const sogl_factor_desc* desc, const int32_t* in_bi, const int32_t* in_bj, int workgroups, int chains,
                     int claims, int64_t* out) {
    Graph g;
    int rc = build(desc, in_bi, in_bj, g);
    if (rc == SOGL_OK) rc = validate_graph(nullptr, &g.d, &g.f, g.hg);
    if (rc) return rc;
    int64_t steps = 0;
    for (const DevTask& k : g.f.tasks) steps += k.dia >= 0;
    Model m(g, chains != 0, claims);
    out[0] = (int64_t)g.f.tasks.size();
    out[1] = (int64_t)m.run(workgroups);
    out[2] = steps;
    out[3] = g.f.n_diag_chains;
    return SOGL_OK;
}

// A chain's update whose added tile is made planted to be a tile made after the chain's lu (and before
// the update): 0 if the check lets it pass, -1 if there is no such tile.
extern "C" int plant_late_sum(const sogl_factor_desc* desc, const int32_t* in_bi, const int32_t* in_bj) {
    Graph g;
    int rc = build(desc, in_bi, in_bj, g);
    if (rc) return -1;
    Model m(g, true, 0);
    for (size_t t = 0; t < g.f.tasks.size(); t++) {
        if (g.f.tasks[t].dia < 0) continue;
        DevTask& d = g.f.tasks[(size_t)g.f.tasks[t].dia];
        for (size_t q = t + 1; q < g.f.tasks.size() && g.f.tasks[q].level < d.level; q++) {
            const DevTask& k = g.f.tasks[q];
            if (k.kind != TK_GEMM || k.next >= 0 || (int32_t)q == g.f.tasks[t].pan_l || (int32_t)q == g.f.tasks[t].pan_u)
                continue;
            for (int32_t e = d.dep_begin; e < d.dep_begin + d.dep_count; e++)
                if (g.hg.deps[(size_t)e] == d.add) g.hg.deps[(size_t)e] = k.out0;
            d.add = k.out0;
            return validate_graph(nullptr, &g.d, &g.f, g.hg);
        }
    }
    return -1;
}

// The tile-column op list of a description (ops may be null): its length, -1 where there is none.
extern "C" int64_t tile_ops(const sogl_factor_desc* desc, const int32_t* in_bi, const int32_t* in_bj, sogl_op* ops) {
    TileOrderOps to;
    if (!tile_order_ops(desc, in_bi, in_bj, to)) return -1;
    if (ops) std::copy(to.ops.begin(), to.ops.end(), ops);
    return (int64_t)to.ops.size();
}
