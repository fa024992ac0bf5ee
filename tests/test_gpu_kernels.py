"""Edges of single kernels' ranges (tile remainders, smallest and largest
sizes of a dispatch rule) against the checker, bit for bit (GPU)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _states(sim, T):
    st, died = sim._read_agents(T)
    st = np.ascontiguousarray(st)
    return st.view(np.uint8).reshape(len(st), st.dtype.itemsize), died


# rows of 16 cells (the shortest of the row kernel) and below, row lengths
# around its 8-cell groups and 512-cell waves, one to four dimensions, reaches
# 1, 2 and 7 (the largest) and 8 (past it), extents smaller than the reach
ROWS = [((16, 5), 1, "chebyshev"), ((15, 6), 1, "chebyshev"), ((17, 3), 2, "euclidean"), ((23, 9), 7, "manhattan"),
        ((50,), 8, "manhattan"), ((40,), 3, "chebyshev"), ((512, 4), 1, "chebyshev"), ((513, 7), 1, "manhattan"),
        ((519, 1), 2, "manhattan"), ((33, 6, 5), 1.5, "euclidean"), ((16, 3, 2, 4), 1, "chebyshev")]


@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("dims,dist,metric", ROWS, ids=lambda v: str(v).replace(" ", ""))
def test_diffuse_rows(vh, ora, gpu_ready, dims, dist, metric, periodic):
    """diffuse on a raster of one-byte cells; some active cells hold values
    other than 1 (any nonzero byte is true and becomes 1)."""
    n = int(np.prod(dims))
    rng = np.random.default_rng(n)
    raw = np.where(rng.random(n) < 2.0 / n, rng.choice([1, 2, 128, 255], n), 0).astype(np.uint8)
    raw[[0, n - 1]] = [255 if n % 2 else 0, 64]
    got = []
    for V in (vh, ora):
        Cell = V.struct("Cell", [("active", "?")])
        Adj = V.struct("Adj")
        model = (V.ModelTypes() | V.register_agenttype_(Cell, "Immortal")
                 | V.register_edgetype_(Adj, "Stateless", target=Cell) | V.create_model("rows"))
        sim = V.create_simulation(model)
        V.raster.add_raster_(sim, "r", dims, raw.view([("active", "?")]), T=Cell)
        V.raster.connect_raster_neighbors_(sim, "r", Adj(), distance=dist, metric=metric, periodic=periodic,
                                           device=None if V is vh else False)
        V.finish_init_(sim)
        out = []
        for _ in range(3):
            V.apply_(sim, V.transitions.diffuse(Adj, Cell), Cell, [Cell, Adj], Cell)
            out.append(_states(sim, Cell)[0].copy())
        got.append(out)
    for k, (a, b) in enumerate(zip(*got)):
        assert np.array_equal(a, b), k


def _ragged_edges(n, seed):
    """In-degrees 0, 1, ..., 9, 0, 1, ... (every remainder of the bodies'
    groups of four), uniform sources, edges in no order."""
    rng = np.random.default_rng(seed)
    to = np.repeat(np.arange(1, n + 1), np.arange(n) % 10)
    to = rng.permutation(to).astype(np.uint64)
    tid = np.uint64(1) << np.uint64(56)
    return tid | rng.integers(1, n + 1, len(to)).astype(np.uint64), tid | to


@pytest.mark.parametrize("n", [1, 63, 1025])
@pytest.mark.parametrize("hints", [(), ("Immortal",)], ids=["mortal", "immortal"])
def test_sum_neighbors_ragged(vh, ora, gpu_ready, hints, n):
    """Int64 sums that wrap, over rows of 0 to 9 in-edges; with mortal agents
    a third dies first (their edges go)."""
    fr, to = _ragged_edges(n, n)
    got = []
    for V in (vh, ora):
        A, E = V.struct("A", [("foo", "<i8")]), V.struct("E")
        model = (V.ModelTypes() | V.register_agenttype_(A, *hints) | V.register_edgetype_(E, "Stateless", target=A)
                 | V.create_model("sum"))
        sim = V.create_simulation(model)
        st = np.zeros(n, dtype=A.dtype)
        st["foo"] = np.arange(n) * 0x1234567812345 + (1 << 62)
        sim._add_agents_array(A, st)
        if len(to):
            sim._add_edges_array(E, fr, to)
        V.finish_init_(sim)
        if not hints:
            V.apply_(sim, V.transitions.die_if("odd"), A, [A], A)
        for _ in range(2):
            V.apply_(sim, V.transitions.sum_neighbors(E), A, [A, E], A)
        raw, died = _states(sim, A)
        got.append((raw[~died], died))
    assert np.array_equal(got[0][1], got[1][1]) and np.array_equal(got[0][0], got[1][0])


@pytest.mark.parametrize("n", [2, 64, 1025])
@pytest.mark.parametrize("fields", [[("foo", "<i8")], []], ids=["state", "stateless"])
def test_added_edges_ragged(vh, ora, gpu_ready, fields, n):
    """neighbor_foo_edges adds 0 to 18 edges per agent: targets, sources in
    insertion order and states as the checker has them."""
    fr, to = _ragged_edges(n, n + 7)
    got = []
    for V in (vh, ora):
        A, E, F = V.struct("A", [("foo", "<i8")]), V.struct("E"), V.struct("F", fields)
        model = (V.ModelTypes() | V.register_agenttype_(A, "Immortal") | V.register_edgetype_(E, "Stateless", target=A)
                 | V.register_edgetype_(F, *([] if fields else ["Stateless"]), target=A) | V.create_model("add"))
        sim = V.create_simulation(model)
        st = np.zeros(n, dtype=A.dtype)
        st["foo"] = np.arange(n)
        sim._add_agents_array(A, st)
        sim._add_edges_array(E, fr, to)
        V.finish_init_(sim)
        out = []
        for _ in range(2):
            V.apply_(sim, V.transitions.neighbor_foo_edges(E, F, -1), A, [A, E], F)
            t, f, s = sim._read_edges(F)
            out += [t.copy(), f.copy(), np.ascontiguousarray(s).view(np.uint8) if fields else np.zeros(0)]
        got.append(out)
    assert len(got[0][0]) == 2 * len(to)
    for a, b in zip(*got):
        assert np.array_equal(a, b)


# one record, partial blocks, one block per tail group and more, a second tail
# level, and more block results than the tail takes (a level of its own first)
@pytest.mark.parametrize("n", [1, 2047, 2049, 9 * 2048 + 5, 2048 * 2048 + 1, 32768 * 2048 + 2049])
def test_mapreduce_levels(vh, ora, gpu_ready, n):
    """Field and computed maps: every level's order is the checker's tree."""
    small = n < 1 << 22
    rng = np.random.default_rng(n)
    fields = [("x", "<f8"), ("g", "u1")] if small else [("g", "u1")]
    st = None
    got = []
    for V in (vh, ora):
        A = V.struct("A", fields)
        sim = V.create_simulation(V.ModelTypes() | V.register_agenttype_(A, "Immortal") | V.create_model("levels"))
        if st is None:
            st = np.zeros(n, dtype=A.dtype)
            st["g"] = rng.integers(0, 5, n)
            if small:
                st["x"] = rng.normal(0, 1, n)
        sim._add_agents_array(A, st)
        V.finish_init_(sim)
        sim.order = 1
        f = V.expr.field
        out = [V.mapreduce(sim, "g", "+", A), V.mapreduce(sim, V.Field("g", 3), "+", A), V.mapreduce(sim, "g", "max", A),
               V.mapreduce(sim, f("g") * 2.5 - 1, "+", A)]
        if small:
            out += [V.mapreduce(sim, "x", op, A) for op in ("+", "max", "min")]
            out += [V.mapreduce(sim, f("x") * f("g"), "+", A)]
        got.append(out)
    assert [repr(v) for v in got[0]] == [repr(v) for v in got[1]]


@pytest.mark.parametrize("depth", [1, 3, 4, 5])
def test_expr_depth(vh, ora, gpu_ready, depth):
    """Programs of each stack depth around the one that fits the registers
    (4), the last operands on top: x op (x op (... select ...))."""
    n = 5000
    rng = np.random.default_rng(depth)
    got = []
    for V in (vh, ora):
        A = V.struct("A", [("x", "<f8"), ("k", "<i4"), ("b", "?")])
        sim = V.create_simulation(V.ModelTypes() | V.register_agenttype_(A) | V.create_model("depth"))
        st = np.zeros(n, dtype=A.dtype)
        r = np.random.default_rng(depth)
        st["x"], st["k"], st["b"] = r.normal(0, 1, n), r.integers(-9, 9, n), r.random(n) < 0.5
        sim._add_agents_array(A, st)
        V.finish_init_(sim)
        sim.order = 1
        f = V.expr.field
        out = []
        for leaf in (f("k"), f("x"), f("b")):
            e = V.expr.where(f("b"), leaf, f("k")) if depth >= 3 else leaf
            for _ in range(depth - 3 if depth >= 3 else depth - 1):
                e = f("k") - e
            out += [V.mapreduce(sim, e, op, A) for op in ("+", "max")] + [V.mapreduce(sim, e > 0, "+", A)]
        got.append(out)
    assert [repr(v) for v in got[0]] == [repr(v) for v in got[1]]


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("case", ["light", "heavy", "sparse"])
def test_opinion_one_pass_blocks(vh, ora, gpu_ready, case, f32):
    """Blocks of 256 agents around one and two tiles of slots: without heavy
    agents (rows of exactly 64 in-edges among them), with one (65), with long
    stretches of isolated agents; the last block partial."""
    n = 256 * 3 + 7
    deg = {"light": lambda i: np.where(i < 256, 12, np.where(i < 512, 13 - i % 3, 64 * (i % 5 == 0))),
           "heavy": lambda i: np.where(i == 300, 65, np.where(i == n - 1, 200, i % 9)),
           "sparse": lambda i: np.where(i % 251 == 0, 3, 0)}[case](np.arange(n))
    rng = np.random.default_rng(n)
    to = rng.permutation(np.repeat(np.arange(1, n + 1), deg)).astype(np.uint32)
    fr = rng.integers(1, n + 1, len(to)).astype(np.uint32)
    w = (rng.random(len(to)) * 0.9 + 0.05).astype(np.float32)
    g = vh.models.build_opinion(vh, n, seed=2, f32=f32, edges=(fr, to, w))
    c = vh.models.build_opinion(ora, n, seed=2, f32=f32, edges=(fr, to, w))
    for k in range(3):
        vh.models.step_opinion(vh, g)
        vh.models.step_opinion(ora, c)
        assert np.array_equal(_states(g.sim, g.T)[0], _states(c.sim, c.T)[0]), k


# contacts (a group of four and remainders, the 32 of a mask, past it),
# redraws, deaths, agents: one word, a partial block, and sizes at which the
# filter's groups hold 2 slots (its bits for single slots end at 1 310 720)
# and blocks of 1024 begin (262 144)
CONTACTS = [(1, 16, 0.05, 1), (3, 0, 0.1, 64), (4, 1, 0.5, 63), (5, 16, 0.3, 257), (31, 3, 0.1, 1000),
            (32, 16, 0.02, 777), (33, 16, 0.02, 777), (7, 16, 0.02, 262_144), (3, 16, 0.04, 1_310_721)]


@pytest.mark.parametrize("C,R,pd,n", CONTACTS)
def test_contact_masks(vh, ora, gpu_ready, C, R, pd, n):
    """States, died flags and contacts of three steps (two at the large
    sizes), newborn slots among them."""
    M = vh.models
    g, c = (M.build_contact(V, n, seed=9, n_init=max(1, n // 5)) for V in (vh, ora))
    for k in range(3 if n < 100_000 else 2):
        for V, m in ((vh, g), (ora, c)):
            M.step_contact(V, m, seed=9, beta=0.3, p_death=pd, n_contacts=C, max_redraw=R)
        (a, da), (b, db) = _states(g.sim, g.T), _states(c.sim, c.T)
        assert np.array_equal(da, db), k
        assert np.array_equal(a[~da], b[~db]), k
        for x, y in zip(g.sim._read_edges(g.E)[:2], c.sim._read_edges(c.E)[:2]):
            assert np.array_equal(x, y), k


@pytest.mark.parametrize("expose", [0, 1])
@pytest.mark.parametrize("block", [64, 256, 1024])
def test_ensemble_four_agents_per_thread(vh, ora, gpu_ready, opts, block, expose):
    """Members around a thread's four agents, a bitmap word and a tile (256 to
    4096 agents), against their solo runs on the checker."""
    opts(sir_expose=expose, sir_expose_min=0)
    E = vh.ensemble.Ensemble()
    E.set_config(block, False)
    E.set_tiles([4, 4, 4])
    sizes = [1, 3, 33, 255, 1023, 1025, 4097, 12345]
    ids = [E.add_sir(n, 6.0, 0.2, 50 + k, 60 + k, n_init=max(1, n // 60)) for k, n in enumerate(sizes)]
    E.step(9)
    E.step(3, use_graph=False)
    for k, (mid, n) in enumerate(zip(ids, sizes)):
        m = vh.models.build_sir(ora, n, seed=50 + k, n_init=max(1, n // 60), init="frac",
                                edges=vh.inputs.graph_gnp(n, 6.0, 60 + k))
        for _ in range(12):
            vh.models.step_sir(ora, m, p_inf=0.2, seed=50 + k, recovery=7)
        got, want = E.read(mid)[0], m.sim._read_agents(m.T)[0]
        assert np.array_equal(np.ascontiguousarray(got).view(np.uint8), np.ascontiguousarray(want).view(np.uint8)), n


# around a tile of 2048 pairs, several, and the switch to tiles of 8192
# (4 194 304) with and without a partial last tile; digits of 9 bits (17 and 26
# bits of rows) and 10 (10 and 20 bits)
@pytest.mark.parametrize("ne,n", [(1, 1), (63, 300), (2047, 5), (2048, 70_000), (2049, 256), (70_001, 66_000),
                                  (4_194_303, 100_000), (4_194_304, 257), (4_202_500, 17_000_000),
                                  (5000, 900), (300_000, 900_000), (4097, 40_000_000)])
def test_edges_sorted_stably(vh, gpu_ready, ne, n):
    """The CSR of edges added in random order: targets ascending, each
    target's edges (source, state) in the order they were added."""
    rng = np.random.default_rng(ne)
    A, E = vh.struct("A", [("x", "u1")]), vh.struct("E", [("k", "<u4")])
    sim = vh.create_simulation(vh.ModelTypes() | vh.register_agenttype_(A, "Immortal")
                               | vh.register_edgetype_(E, target=A) | vh.create_model("sort"))
    sim._add_agents_array(A, np.zeros(n, dtype=A.dtype))
    tid = np.uint64(1) << np.uint64(56)
    fr, to = (tid | rng.integers(1, n + 1, ne).astype(np.uint64) for _ in range(2))
    st = np.zeros(ne, dtype=E.dtype)
    st["k"] = np.arange(ne)
    sim._add_edges_array(E, fr, to, st)
    vh.finish_init_(sim)
    order = np.argsort(to, kind="stable")
    t, f, s = sim._read_edges(E)
    assert np.array_equal(t, to[order]) and np.array_equal(f, fr[order]) and np.array_equal(s["k"], order)


@pytest.mark.parametrize("late", [False, True])
def test_ensemble_out_edges_together(vh, ora, gpu_ready, opts, late):
    """Out-edges of several members from one sort: members without edges, of
    one agent, around 256 rows, and one whose 9 10^6 edges end a batch; the
    exposure pass on from the start, or only after the members were added."""
    opts(sir_expose=0 if late else 1, sir_expose_min=0)
    E = vh.ensemble.Ensemble()
    sizes = [(1, 0.0), (256, 4.0), (300, 0.0), (255, 9.0), (257, 1.0), (900_000, 10.0), (513, 3.0), (70_000, 12.0)]
    ids = [E.add_sir(n, d, 0.2, 70 + k, 80 + k, n_init=max(1, n // 60)) for k, (n, d) in enumerate(sizes)]
    if late:
        E.step(2)
        opts(sir_expose=1)
    E.step(6)
    for k, (mid, (n, d)) in enumerate(zip(ids, sizes)):
        m = vh.models.build_sir(ora, n, seed=70 + k, n_init=max(1, n // 60), init="frac",
                                edges=vh.inputs.graph_gnp(n, d, 80 + k))
        for _ in range(8 if late else 6):
            vh.models.step_sir(ora, m, p_inf=0.2, seed=70 + k, recovery=7)
        got, want = E.read(mid)[0], m.sim._read_agents(m.T)[0]
        assert np.array_equal(np.ascontiguousarray(got).view(np.uint8), np.ascontiguousarray(want).view(np.uint8)), n


# one target; around 256 targets; a block of several passes (256 x 40 > 4096
# edges); most agents a source, so that every list draws again; degrees of
# thousands
@pytest.mark.parametrize("n,deg", [(1, 0.0), (2, 1.0), (255, 16.0), (256, 17.5), (257, 100.0), (1000, 40.0), (40, 30.0),
                                   (2500, 2000.0), (100_001, 8.0)])
def test_gnp_sources(vh, gpu_ready, n, deg):
    """The device's G(n, p) against the host twin."""
    A, E = vh.struct("A", [("x", "u1")]), vh.struct("E", [])
    sim = vh.create_simulation(vh.ModelTypes() | vh.register_agenttype_(A, "Immortal")
                               | vh.register_edgetype_(E, "Stateless", target=A) | vh.create_model("gnp"))
    sim._add_agents_array(A, np.zeros(n, dtype=A.dtype))
    sim._add_edges_gnp(E, deg, 11)
    vh.finish_init_(sim)
    t, f, _ = sim._read_edges(E)
    fr, to = vh.inputs.graph_gnp(n, deg, 11)
    tid = np.uint64(1) << np.uint64(56)
    assert np.array_equal(t, tid | to.astype(np.uint64)) and np.array_equal(f, tid | fr.astype(np.uint64))


@pytest.mark.parametrize("f32", [False, True])
def test_opinion_batch_beyond_the_caches(vh, gpu_ready, f32):
    """Five simulations whose edges are more than 256 MB together, batched,
    against the same simulations one by one (72 MB of edges at most)."""
    sizes = [900_000, 750_000, 800_000, 700_001, 900_017]

    def build():
        s = C.c_void_p()
        vh._abi.lib().stream_create(C.byref(s))
        return [vh.models.build_opinion_gnp(vh, n, mean_deg=9.0, seed=k, graph_seed=20 + k, weight_seed=40 + k, f32=f32,
                                            stream=s) for k, n in enumerate(sizes)]
    ms, solo = build(), build()
    m0 = ms[0]
    vh.Batch().apply([m.sim for m in ms], vh.transitions.opinion(m0.E, 0.3, f32), m0.T, [m0.T, m0.E], m0.T, steps=3)
    for m, o in zip(ms, solo):
        for _ in range(3):
            vh.apply_(o.sim, vh.transitions.opinion(o.E, 0.3, f32), o.T, [o.T, o.E], o.T)
        assert np.array_equal(_states(m.sim, m.T)[0].view(np.uint8), _states(o.sim, o.T)[0].view(np.uint8))


# in-degrees around a wave's 64 lanes, the limits of the plan's classes (64,
# 65, 512, 513) and blocks of more than 2048 agents (most without in-edges)
@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("degs,n", [([0, 1, 2, 3, 63, 64, 65, 130, 512, 513, 700], 3000), ([64], 1025), ([65], 900),
                                    ([0] * 60 + [1, 7], 40_000), ([5, 5, 5, 6, 9, 70], 6000), ([1], 64)])
def test_opinion_plan_order(vh, ora, gpu_ready, opts, degs, n, f32):
    """The two-pass gather over blocks ordered by in-degree, three steps."""
    opts(opinion_plan_bytes=0, opinion_part_bytes=4096)
    rng = np.random.default_rng(n + f32)
    d = rng.choice(degs, n)
    d[0] = max(d[0], 1)
    to = np.repeat(np.arange(1, n + 1), d)
    fr = rng.integers(1, n + 1, len(to))
    dt = np.float32 if f32 else np.float64
    got = []
    for V in (vh, ora):
        A, E = V.struct("A", [("x", dt)]), V.struct("E", [("w", "<f4")])
        r = np.random.default_rng(n)
        sim = V.create_simulation(V.ModelTypes() | V.register_agenttype_(A, "Immortal")
                                  | V.register_edgetype_(E, target=A) | V.create_model("order"))
        st, ws = np.zeros(n, dtype=A.dtype), np.zeros(len(to), dtype=E.dtype)
        st["x"], ws["w"] = r.random(n), r.random(len(to)) + 0.01
        sim._add_agents_array(A, st)
        tid = np.uint64(1) << np.uint64(56)
        sim._add_edges_array(E, tid | fr.astype(np.uint64), tid | to.astype(np.uint64), ws)
        V.finish_init_(sim)
        for _ in range(3):
            V.apply_(sim, V.transitions.opinion(E, 0.3, f32), A, [A, E], A)
        got.append(_states(sim, A)[0])
    assert np.array_equal(*got)


@pytest.mark.parametrize("n", [1, 3, 33, 1023, 1026, 4100, 70_001])
def test_sir_exposure_two_launches(vh, ora, gpu_ready, opts, n):
    """Solo SIR with the exposure pass from few agents on, the pass left out in
    one step, around a lane's four agents and a block's 1024."""
    M = vh.models
    g, c = (M.build_sir(V, n, seed=3, n_init=max(1, n // 60), init="frac", edges=vh.inputs.graph_gnp(n, 6.0, 4))
            for V in (vh, ora))
    for k in range(8):
        opts(sir_expose=int(k != 4), sir_expose_min=0)
        for V, m in ((vh, g), (ora, c)):
            M.step_sir(V, m, p_inf=0.2, seed=3, recovery=5)
        assert np.array_equal(_states(g.sim, g.T)[0], _states(c.sim, c.T)[0]), k


@pytest.mark.parametrize("block,apt", [(64, 1), (64, 4), (128, 1), (256, 1)])
def test_ensemble_long_runs(vh, ora, gpu_ready, opts, block, apt):
    """Epidemics that are over, not yet everywhere, or nearly everywhere, over
    60 steps, in tiles from a quarter of a wave's four agents per lane on: with
    the exposure pass switched off and on between calls, members past
    their horizon and called on again after it."""
    opts(sir_expose=1, sir_expose_min=0)
    E = vh.ensemble.Ensemble()
    E.set_config(block, False)
    E.set_tiles([apt] * 3)
    sizes = [(3000, 3.0, 0.3, 1), (5000, 1.2, 0.3, 3), (20_000, 2.0, 0.2, 1), (4097, 6.0, 0.2, 60), (900, 0.5, 0.9, 2)]
    ids = [E.add_sir(n, d, p, 90 + k, 30 + k, recovery=4, n_init=i) for k, (n, d, p, i) in enumerate(sizes)]
    sims = [vh.models.build_sir(ora, n, seed=90 + k, n_init=i, init="frac", edges=vh.inputs.graph_gnp(n, d, 30 + k))
            for k, (n, d, p, i) in enumerate(sizes)]
    done = [0] * len(sizes)

    def check(upto):
        for k, (n, d, p, i) in enumerate(sizes):
            while done[k] < upto[k]:
                vh.models.step_sir(ora, sims[k], p_inf=p, seed=90 + k, recovery=4)
                done[k] += 1
            got, want = E.read(ids[k])[0], sims[k].sim._read_agents(sims[k].T)[0]
            assert np.array_equal(np.ascontiguousarray(got).view(np.uint8), np.ascontiguousarray(want).view(np.uint8)), k
    E.set_horizon(ids[2], 9)
    E.step(14)
    check([14, 14, 9, 14, 14])
    opts(sir_expose=0)
    E.step(3)
    opts(sir_expose=1)
    E.set_horizon(ids[2], 0)
    E.step(20, use_graph=False)
    check([37, 37, 29, 37, 37])
    E.step(23)
    check([60, 60, 52, 60, 60])


def _edge_list(sim, E, state):
    t, f, s = sim._read_edges(E)
    return [np.array(t), np.array(f), np.ascontiguousarray(s).view(np.uint8).copy() if state else np.zeros(0)]


@pytest.mark.parametrize("hints", [(), ("SingleEdge",)], ids=["plain", "single"])
def test_edge_rebuild_out_of_memory(vh, ora, gpu_ready, hints):
    """Each device allocation of a rebuild with more rows and edges fails
    once: the edges are then the old ones, or none where a buffer had grown,
    and the same call afterwards gives the oracle's edges."""
    n = 300
    fr, to = _ragged_edges(n, 5)

    def build(V):
        A, E, F = V.struct("A", [("foo", "<i8")]), V.struct("E"), V.struct("F", [("foo", "<i8")])
        kw = {} if "SingleEdge" in hints else {"target": A}
        model = (V.ModelTypes() | V.register_agenttype_(A) | V.register_edgetype_(E, "Stateless", target=A)
                 | V.register_edgetype_(F, *hints, **kw) | V.create_model("oom"))
        sim = V.create_simulation(model)
        st = np.zeros(n, dtype=A.dtype)
        st["foo"] = np.arange(n)
        sim._add_agents_array(A, st)
        sim._add_edges_array(E, fr, to)
        V.finish_init_(sim)
        V.apply_(sim, V.transitions.add_self_edge(F, state=np.array([7], "<i8")), A, A, F)
        V.apply_(sim, V.transitions.spawn(A, 4, E), A, [A, E], [A, E], add_existing=E)
        body = (V.transitions.add_self_edge(F, state=np.array([9], "<i8")) if hints
                else V.transitions.neighbor_foo_edges(E, F, -1))
        return sim, A, E, F, lambda: V.apply_(sim, body, A, [A, E], F)

    csim, _, _, cF, step = build(ora)
    step()
    want = _edge_list(csim, cF, True)
    lib, failed, emptied = vh._abi.lib(), 0, 0
    for after in range(100):
        sim, A, E, F, step = build(vh)
        old = _edge_list(sim, F, True)
        assert len(old[0]) == n
        lib.debug_fail_allocs_after(after, 1)
        try:
            step()
            break
        except vh.VahanaError as err:
            assert err.code == vh._abi.VH_ERR_OOM, after
        finally:
            lib.debug_fail_allocs(0)
        failed += 1
        now = _edge_list(sim, F, True)
        empty = len(now[0]) == 0
        emptied += empty
        assert empty or all(np.array_equal(a, b) for a, b in zip(now, old)), after
        step()
        for a, b in zip(_edge_list(sim, F, True), want):
            assert np.array_equal(a, b), after
    print(f"[gpu] {failed} allocations failed, {emptied} of them with the edges gone", flush=True)
    assert 0 < emptied < failed < 100


@pytest.mark.parametrize("C", [9, 40], ids=["masks", "log"])
def test_contact_rebuild_out_of_memory(vh, gpu_ready, C):
    """Each device allocation of a contact step with more contacts and newborn
    slots fails once: the contacts are the old ones or none."""
    M, lib = vh.models, vh._abi.lib()
    failed, emptied = 0, 0
    for after in range(100):
        m = M.build_contact(vh, 3000, seed=9, n_init=600)
        M.step_contact(vh, m, seed=9, beta=0.3, p_death=0.0, n_contacts=2)
        old = _edge_list(m.sim, m.E, False)
        lib.debug_fail_allocs_after(after, 1)
        try:
            M.step_contact(vh, m, seed=9, beta=0.3, p_death=0.3, n_contacts=C)
            break
        except vh.VahanaError as err:
            assert err.code == vh._abi.VH_ERR_OOM, after
        finally:
            lib.debug_fail_allocs(0)
        failed += 1
        now = _edge_list(m.sim, m.E, False)
        emptied += len(now[0]) == 0
        assert len(now[0]) == 0 or all(np.array_equal(a, b) for a, b in zip(now, old)), after
    print(f"[gpu] {failed} allocations failed, {emptied} of them with the contacts gone", flush=True)
    assert 0 < emptied < failed < 100


@pytest.mark.parametrize("n", [4999, 5120])
@pytest.mark.parametrize("shift", range(7))
def test_contact_filter_groups(vh, ora, gpu_ready, shift, n):
    """Filter groups of 1, 2, 4, ..., 32 slots and, past them, no filter: 20
    blocks of 256 slots (25 with newborns at most), whose bits fit the limit
    from that group size on. Many deaths, so that a group without its mark
    would keep dead partners."""
    M, lib = vh.models, vh._abi.lib()
    g, c = (M.build_contact(V, n, seed=4, n_init=n // 5) for V in (vh, ora))
    lib.debug_contact_filter(800 >> shift)
    try:
        for k in range(4):
            for V, m in ((vh, g), (ora, c)):
                M.step_contact(V, m, seed=4, beta=0.3, p_death=0.05, n_contacts=6)
            (a, da), (b, db) = _states(g.sim, g.T), _states(c.sim, c.T)
            assert np.array_equal(da, db), k
            assert np.array_equal(a[~da], b[~db]), k
            for x, y in zip(g.sim._read_edges(g.E)[:2], c.sim._read_edges(c.E)[:2]):
                assert np.array_equal(x, y), k
    finally:
        lib.debug_contact_filter(0)


@pytest.mark.parametrize("f32", [False, True])
def test_opinion_one_pass_beyond_the_caches(vh, gpu_ready, opts, f32):
    """One simulation whose edges are more than 256 MB, gathered in one pass
    (its edges read past the caches) against the two-pass gather."""
    got = []
    for plan in (-1, 0):
        opts(opinion_plan_bytes=plan)
        m = vh.models.build_opinion_gnp(vh, 3_800_001, mean_deg=9.0, seed=3, graph_seed=23, weight_seed=43, f32=f32)
        assert vh.num_edges(m.sim, m.E) * 8 > 256 << 20
        for _ in range(2):
            vh.models.step_opinion(vh, m, eps=0.3)
        got.append(_states(m.sim, m.T)[0].copy())
    assert np.array_equal(*got)


@pytest.mark.parametrize("body", ["sum", "foo_edges", "diffuse", "move_to"])
def test_bodies_need_sources(vh, gpu_ready, body):
    """A body that asks an :IgnoreFrom type for its neighbours fails with the
    reference's assertion (the type keeps no sources to look at)."""
    n = 64
    A, E, F = vh.struct("A", [("foo", "<i8"), ("active", "?")]), vh.struct("E"), vh.struct("F", [("foo", "<i8")])
    model = (vh.ModelTypes() | vh.register_agenttype_(A, "Immortal") | vh.register_edgetype_(E, "Stateless", "IgnoreFrom")
             | vh.register_edgetype_(F) | vh.create_model("sources"))
    sim = vh.create_simulation(model)
    st = np.zeros(n, dtype=A.dtype)
    st["foo"] = np.arange(n)
    vh.raster.add_raster_(sim, "r", (8, 8), st, T=A)
    ids = (np.uint64(1) << np.uint64(56)) | np.arange(1, n + 1, dtype=np.uint64)
    sim._add_edges_array(E, np.roll(ids, 1), ids)
    vh.finish_init_(sim)
    T = vh.transitions
    tr, write = {"sum": (T.sum_neighbors(E), A), "foo_edges": (T.neighbor_foo_edges(E, F, -1), F),
                 "diffuse": (T.diffuse(E, A), A), "move_to": (T.move_to_value(sim, "r", E), [A, E])}[body]
    with pytest.raises(AssertionError, match="hint combination"):
        vh.apply_(sim, tr, A, [A, E], write)
    assert vh.num_agents(sim, A) == n


def test_errors_of_replayed_steps(vh, gpu_ready):
    """A captured general transition that flags: each replay's error is
    reported by the next checked apply!, also by one whose own kernels can
    not flag, and only once."""
    import torch
    A, E = vh.struct("A", [("foo", "<i8")]), vh.struct("E")
    B, F = vh.struct("B", [("opinion", "<f8")]), vh.struct("F", [("w", "<f4")])
    model = (vh.ModelTypes() | vh.register_agenttype_(A, "Immortal", "Independent") | vh.register_agenttype_(B, "Immortal")
             | vh.register_edgetype_(E, "Stateless", target=A) | vh.register_edgetype_(F, target=B)
             | vh.create_model("replay"))
    sim = vh.create_simulation(model)
    stream = torch.cuda.Stream()
    sim._set_streams(stream.cuda_stream)
    sim._add_agents_array(A, np.zeros(100, dtype=A.dtype))
    sim._add_agents_array(B, np.full(50, 0.5).view(B.dtype))
    ids = (np.uint64(1) << np.uint64(56)) | np.arange(1, 101, dtype=np.uint64)
    sim._add_edges_array(E, np.roll(ids, 1), ids)
    vh.finish_init_(sim)

    def flag():   # A is not in `read`
        vh.apply_(sim, vh.transitions.sum_neighbors(E), A, [E], A)

    def checked():
        vh.apply_(sim, vh.transitions.opinion(F, 0.2, False), B, [B, F], B)
    vh.enable_asserts(False)
    try:
        flag()
    finally:
        vh.enable_asserts(True)
    with pytest.raises(AssertionError):
        checked()
    checked()   # (and B's buffers are where they were: the captured step needs the context it has)
    g = torch.cuda.CUDAGraph()
    vh.enable_asserts(False)
    try:
        with torch.cuda.graph(g, stream=stream, capture_error_mode="thread_local"):
            flag()
    finally:
        vh.enable_asserts(True)
    for _ in range(3):
        checked()
        with torch.cuda.stream(stream):
            g.replay()
        with pytest.raises(AssertionError, match="read"):
            checked()
    assert vh.num_agents(sim, A) == 100


@pytest.mark.parametrize("value", [1, 255])
@pytest.mark.parametrize("dims,dist", [((40, 9), 2), ((600, 5), 1), ((1100, 6), 5), ((24, 7, 6), 2)],
                         ids=lambda v: str(v).replace(" ", ""))
def test_diffuse_rows_filled(vh, ora, gpu_ready, dims, dist, value):
    """diffuse up to the raster where all cells are active but for holes that
    only some offsets reach, at which whole waves stop early or do not."""
    n = int(np.prod(dims))
    raw = np.full(n, value, dtype=np.uint8)
    hole = np.random.default_rng(n).integers(0, n)
    got = []
    for V in (vh, ora):
        Cell, Adj = V.struct("Cell", [("active", "?")]), V.struct("Adj")
        model = (V.ModelTypes() | V.register_agenttype_(Cell, "Immortal")
                 | V.register_edgetype_(Adj, "Stateless", target=Cell) | V.create_model("filled"))
        sim = V.create_simulation(model)
        cells = raw.reshape(dims, order="F").copy()
        at = np.unravel_index(hole, dims, order="F")
        box = tuple(slice(max(0, a - dist), a + dist + 1) for a in at)
        cells[box] = 0   # the hole's cells see active ones at its edge only
        V.raster.add_raster_(sim, "r", dims, cells.reshape(-1, order="F").view([("active", "?")]), T=Cell)
        V.raster.connect_raster_neighbors_(sim, "r", Adj(), distance=dist, periodic=False,
                                           device=None if V is vh else False)
        V.finish_init_(sim)
        out = []
        for _ in range(3):
            V.apply_(sim, V.transitions.diffuse(Adj, Cell), Cell, [Cell, Adj], Cell)
            out.append(_states(sim, Cell)[0].copy())
        got.append(out)
    for k, (a, b) in enumerate(zip(*got)):
        assert np.array_equal(a, b), k


@pytest.mark.parametrize("C,R,pd,n", [(8, 2, 0.5, 3001), (32, 16, 0.5, 5000), (20, 1, 0.5, 777), (6, 3, 0.9, 1000),
                                      (33, 2, 0.5, 777), (5, 16, 0.3, 8)])
def test_contact_many_deaths(vh, ora, gpu_ready, C, R, pd, n):
    """Most first draws fail: on dying slots (not kept), on dead ones and the
    slot itself (drawn again, up to the limit)."""
    M = vh.models
    g, c = (M.build_contact(V, n, seed=6, n_init=max(1, n // 3)) for V in (vh, ora))
    for k in range(5):
        for V, m in ((vh, g), (ora, c)):
            M.step_contact(V, m, seed=6, beta=0.3, p_death=pd, n_contacts=C, max_redraw=R)
        (a, da), (b, db) = _states(g.sim, g.T), _states(c.sim, c.T)
        assert np.array_equal(da, db), k
        assert np.array_equal(a[~da], b[~db]), k
        for x, y in zip(g.sim._read_edges(g.E)[:2], c.sim._read_edges(c.E)[:2]):
            assert np.array_equal(x, y), k
