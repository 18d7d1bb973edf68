"""The order in which the persistent executor's workgroups can run a task graph with diagonal chains, on
the CPU: host/graph_model.hip builds the graph with the executor's own code and plays the queue without
times.  Every number of workgroups above the number of chains has to finish every task with the chains'
steps inside their lus, and any number without (two workgroups per CU, dynamic chaining)."""
import ctypes as C

import numpy as np
import pytest

import host_lib
import sogl


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    return host_lib.build("graph_model", str(tmp_path_factory.mktemp("graph_model")))


def fill(n, pairs):
    """Block rows of L (strictly lower) of a symmetric block pattern after elimination in order."""
    rows = [set() for _ in range(n)]
    for i, j in pairs:
        rows[max(i, j)].add(min(i, j))
    cols = [set() for _ in range(n)]
    for i in range(n):
        for j in rows[i]:
            cols[j].add(i)
    for j in range(n):
        c = sorted(cols[j])
        for a, i in enumerate(c):
            for k in c[a + 1:]:
                rows[k].add(i)
                cols[i].add(k)
    return rows


def leaf_beside_chain(depth, width):
    """A tridiagonal chain of `depth` block rows, then a block coupled to none of them, then `width` rows
    coupled to it, the first of them to the chain's end as well: that row's diagonal has an update from
    the chain that is made long after the leaf's lu could be."""
    leaf = depth
    pairs = [(i, i + 1) for i in range(depth - 1)] + [(leaf, leaf + 1 + k) for k in range(width)] + [(depth - 1, leaf + 1)]
    return depth + 1 + width, pairs


def band(n, half):
    return n, [(i, j) for i in range(n) for j in range(max(0, i - half), i)]


LU, LLT = 1, 10


def describe(n, pairs, symmetric, precision):
    """A factor description of the block pattern (one op, which says LU or L L^T; the tile-column list takes its
    place) and its inputs' block coordinates."""
    at = [(i, i) for i in range(n)] + [(max(p), min(p)) for p in pairs]
    if not symmetric:
        at += [(j, i) for i, j in at if i != j]
    ids = np.arange(1, len(at) + 1, dtype=np.int32)
    nid = len(at) + 1
    rows = fill(n, pairs)
    lt, ut = [], []
    for i in range(n):
        for j in sorted(rows[i]) + [i]:
            lt.append([i, j, nid])
            nid += 1
            if not symmetric:
                ut.append([j, i, nid])
                nid += 1
    op = [[1, 0, LLT if symmetric else LU, lt[0][2], 0 if symmetric else ut[0][2], 1, 0, 0]]
    d, keep = sogl.make_desc(nid, op, ids, np.zeros((1, 1)), lt, ut if ut else np.zeros((0, 3)), n, precision)
    bi, bj = (np.array([a[k] for a in at], np.int32) for k in range(2))
    return d, (keep, bi, bj), bi.ctypes.data_as(C.c_void_p), bj.ctypes.data_as(C.c_void_p)


def play(lib, desc, workgroups, chains, claims):
    d, _, bi, bj = desc
    out = np.zeros(4, np.int64)
    assert lib.model(C.byref(d), bi, bj, workgroups, chains, claims, out.ctypes.data_as(C.c_void_p)) == sogl.OK
    return dict(zip(("tasks", "finished", "steps", "chains"), (int(v) for v in out)))


PATTERNS = {
    "leaf_beside_chain": lambda: leaf_beside_chain(12, 8),
    "wide_leaf_beside_chain": lambda: leaf_beside_chain(40, 30),
    "band_3": lambda: band(14, 3),
    "tridiagonal": lambda: band(20, 1),
}


# a row coupled to every 32nd: each of its diagonal's updates is a part of its own
STAGED = dict(PATTERNS, band_40=lambda: band(90, 40), every_32nd=lambda: (641, [(640, 32 * q) for q in range(20)]),
              every_32nd_beside_a_band=lambda: (200, band(200, 2)[1] + [(160, 32 * q) for q in range(5)]))


@pytest.mark.parametrize("symmetric", [False, True])
@pytest.mark.parametrize("name", sorted(STAGED))
def test_stages_follow_their_operands(lib, name, symmetric):
    """The tile-column list's stages are a schedule: an op comes after the ops that make what it reads, and
    the products of one sum share a stage."""
    d, _, bi, bj = describe(*STAGED[name](), symmetric, sogl.FP64)
    lib.tile_ops.restype = C.c_int64
    ops = np.zeros((lib.tile_ops(C.byref(d), bi, bj, None), 8), np.int32)
    lib.tile_ops(C.byref(d), bi, bj, ops.ctypes.data_as(C.c_void_p))
    made = {}
    for src, src2, _, res, res2, stage, _, _ in ops.tolist():
        for r in (res, res2):
            if r:
                assert made.setdefault(r, stage) == stage
    for src, src2, _, res, _, stage, _, _ in ops.tolist():
        assert all(stage > made.get(a, 0) for a in (src, src2) if a), (src, src2, res, stage)


@pytest.mark.parametrize("symmetric", [False, True])
@pytest.mark.parametrize("name", sorted(PATTERNS))
@pytest.mark.parametrize("chains,claims", [(1, 0), (0, 0), (0, 4)])
def test_every_task_finishes(lib, name, symmetric, chains, claims):
    desc = describe(*PATTERNS[name](), symmetric, sogl.FP64)
    least = play(lib, desc, 64, chains, claims)["chains"] if chains else 0
    for workgroups in range(least + 1, least + 8):
        r = play(lib, desc, workgroups, chains, claims)
        assert r["finished"] == r["tasks"], (workgroups, r)


def test_bands_are_chains(lib):
    for half in (1, 3):  # every diagonal but the first comes from a chain's step
        r = play(lib, describe(*band(14, half), False, sogl.FP32), 4, 1, 0)
        assert (r["chains"], r["steps"]) == (1, 13)


@pytest.mark.parametrize("symmetric", [False, True])
def test_late_sum_breaks_the_chain(lib, symmetric):
    """The leaf's step is not linked (the row's other updates come long after the leaf's lu), and a graph
    with such a link is refused."""
    desc = describe(*leaf_beside_chain(12, 8), symmetric, sogl.FP64)
    assert play(lib, desc, 4, 1, 0)["steps"] == 11 + 7  # along the chain, and along the leaf's rows
    d, _, bi, bj = describe(*band(14, 3), symmetric, sogl.FP64)
    assert lib.plant_late_sum(C.byref(d), bi, bj) > 0


class Ops:
    """An op list over new ids, kept by stage."""
    LINV, UINV, SUB, MUL = 2, 3, 4, 8

    def __init__(self, inputs):
        self.inputs = {key: k + 1 for k, key in enumerate(inputs)}
        self.n_ids = len(self.inputs) + 1
        self.rows, self.lt, self.ut = [], [], []

    def __getitem__(self, key):
        return self.inputs[key]

    def op(self, code, src, src2, stage, res=None):
        if res is None:
            res, self.n_ids = self.n_ids, self.n_ids + 1
        self.rows.append([src, src2, code, res, 0, stage, 0, 0])
        return res

    def less(self, a, products, stage):
        """a - sum of the products"""
        acc = None
        for x, y in products:
            acc = self.op(self.MUL, x, y, stage, acc)
        return self.op(self.SUB, acc, a, stage + 1)

    def lu(self, k, s, stage):
        low = self.op(LU, s, 0, stage)
        up, self.n_ids = self.n_ids, self.n_ids + 1
        self.rows[-1][4] = up
        self.lt.append([k, k, low])
        self.ut.append([k, k, up])
        return self.op(self.LINV, low, 0, stage + 1), self.op(self.UINV, up, 0, stage + 1)

    def panels(self, k, x, z, s_l, s_u, stage):
        pl, pu = self.op(self.MUL, s_l, z, stage), self.op(self.MUL, x, s_u, stage)
        self.lt.append([k + 1, k, pl])
        self.ut.append([k, k + 1, pu])
        return pl, pu

    def desc(self, n):
        rows = sorted(self.rows, key=lambda r: r[5])
        for k, r in enumerate(rows):
            r[6] = k
        ids = np.arange(1, len(self.inputs) + 1, dtype=np.int32)
        d, keep = sogl.make_desc(self.n_ids, rows, ids, np.zeros((1, 1)), self.lt, self.ut, n, sogl.FP64)
        return d, keep, None, None


def tridiagonal_inputs(n):
    return [(i, i) for i in range(n)] + [(i + 1, i) for i in range(n - 1)] + [(i, i + 1) for i in range(n - 1)] + ["v"]


def claims_inside_a_chain():
    """The first step's panel could claim a product that the third step's panel needs (a sum of 60 products
    follows the claimed one, so it is on the critical path)."""
    n = 4
    o = Ops(tridiagonal_inputs(n))
    s, first = o[0, 0], None
    for k in range(n):
        st = 10 * k + 1
        x, z = o.lu(k, s, st)
        if k == n - 1:
            break
        s_l, v = o[k + 1, k], o["v"]
        if k == 2:
            s_l = o.less(s_l, [(o.op(o.MUL, first, v, 5), v)] + [(v, v)] * 60, 6)
        pl, pu = o.panels(k, x, z, s_l, o[k, k + 1], st + 2)
        first = first or pl
        s = o.less(o[k + 1, k + 1], [(pl, pu)], st + 3)
    return o.desc(n)


def claims_before_a_chain():
    """A product outside any chain could claim the sum that a chain's first lu follows, and with it another
    that this lu's panel needs (a sum of 13 products follows that one: both are on the critical path)."""
    o = Ops(tridiagonal_inputs(2))
    v = o["v"]
    p = o.op(o.MUL, v, v, 1)
    s_l = o.less(o[1, 0], [(o.op(o.MUL, p, v, 2), v)] + [(v, v)] * 12, 3)
    x, z = o.lu(0, o.less(o[0, 0], [(p, v)], 2), 5)
    pl, pu = o.panels(0, x, z, s_l, o[0, 1], 7)
    o.lu(1, o.less(o[1, 1], [(pl, pu)], 8), 10)
    return o.desc(2)


@pytest.mark.parametrize("make", [claims_inside_a_chain, claims_before_a_chain])
def test_claims_beside_a_chain(lib, make):
    """Dynamic chaining: a workgroup runs the tasks it has claimed when its chain ends, so it runs no diagonal
    chain (one that waits for a task it holds never ends)."""
    desc = make()
    for workgroups in (2, 3, 8):
        for claims in (0, 1, 8):
            r = play(lib, desc, workgroups, int(claims == 0), claims)
            assert r["steps"] > 0 and r["finished"] == r["tasks"], (claims, workgroups, r)
