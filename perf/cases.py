"""Performance cases: what programs have this framework do, through its public
entry points (the Python API and the C ABI it binds).

`listed()` names the cases, `draw(rng)` gives others of the same ranges,
`prepare(case, seed)` builds what a program has in hand before the call,
`run(state)` is one pass, `work(case)` the bytes and operations it cannot do
without, and `exact(case, seed)` the result in 64 bits by plain numpy.
"""
import ctypes as C
import importlib.util
import math
import os
import sys
import types

import numpy as np
import torch

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vahana.jl_amd")


def _package():
    """vahana.jl_amd/ as the module `vahana_amd` (the folder's name has a dot)."""
    if "vahana_amd" not in sys.modules:
        spec = importlib.util.spec_from_file_location(
            "vahana_amd", os.path.join(PKG, "__init__.py"), submodule_search_locations=[PKG])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["vahana_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["vahana_amd"]


vh = _package()
EPS = 0.2          # bounded confidence of every opinion case
TYPE1 = np.uint64(1) << np.uint64(56)


def listed():
    return [
        # the opinion benchmark: 10^7 agents on a Barabasi-Albert graph, one
        # apply! after the other in production mode (asserts off), then the
        # opinions are read
        {"name": "opinion_f64_ba_10m", "kind": "opinion", "n": 10_000_000, "m": 5, "graph": "ba", "f32": False,
         "steps": 10, "asserts": False},
        # its Float32 variant at a ragged size on a directed random graph, as
        # the serving loop builds them
        {"name": "opinion_f32_gnp_5m", "kind": "opinion", "n": 5_000_011, "deg": 8.0, "graph": "gnp", "f32": True,
         "steps": 10, "asserts": False},
        # an everyday model: a graph of the user's own, default settings
        # (asserts on), a state vector that one pass gathers
        {"name": "opinion_f64_200k", "kind": "opinion", "n": 200_003, "deg": 12.0, "graph": "host", "f32": False,
         "steps": 20, "asserts": True},
        # the smallest calls: a toy model stepped many times, where latency
        # and launches count
        {"name": "opinion_f32_small", "kind": "opinion", "n": 1_501, "deg": 10.0, "graph": "host", "f32": True,
         "steps": 100, "asserts": True},
        # a server's quantum of small opinion requests advanced together
        {"name": "opinion_batch_24", "kind": "batch", "sims": 24, "n_min": 10_000, "n_max": 1_000_000, "deg": 10.0,
         "sizes": 7, "f32": False, "steps": 20},
        # the SIR benchmark from start to end: agents and edges of a host
        # graph added, finish_init!, 100 days, the states read
        {"name": "sir_run_100k", "kind": "sir", "n": 100_000, "deg": 10.0, "p_inf": 0.05, "recovery": 7,
         "n_init": 100, "steps": 100, "asserts": True},
        # a parameter sweep: SIR replicas of uneven size on device graphs,
        # built, advanced 200 days and read
        {"name": "sir_sweep_48", "kind": "sweep", "members": 48, "n_min": 1_000, "n_max": 1_000_000, "sizes": 3,
         "steps": 200},
        # the dynamic contact network (births, deaths, 20 new partners per
        # agent and step) at its endemic state
        {"name": "contact_10m", "kind": "contact", "n": 10_000_000, "contacts": 20, "p_death": 0.02, "steps": 5,
         "asserts": False},
        # a raster scenario: a copy of the prepared simulation, 50 steps of
        # diffusion, the cells read
        {"name": "raster_3162", "kind": "raster", "nx": 3_162, "ny": 3_162, "periodic": True, "distance": 1,
         "frac": 1e-6, "steps": 50, "asserts": False},
        # a transition of the general form: every agent sums a field over its
        # neighbours (neighborstates), default settings
        {"name": "neighbors_1m", "kind": "neighbors", "n": 1_000_000, "deg": 10.0, "steps": 10, "asserts": True},
        # a network rebuilt in transitions: every agent adds edges to and from
        # its neighbours (add_edge!), the next transition reads them
        {"name": "rewire_200k", "kind": "rewire", "n": 200_000, "deg": 8.0, "steps": 5, "asserts": True},
        # the statistics that a program takes after a step: sum, mean of a
        # condition, extrema and counts over the agents of a type
        {"name": "stats_10m", "kind": "stats", "n": 10_000_000},
    ]


def _logu(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["opinion", "opinion", "opinion", "batch", "sir", "sweep", "contact", "raster", "neighbors",
                       "rewire", "stats"])
    if kind == "opinion":
        graph = rng.choice(["ba", "gnp", "host"])
        c = {"kind": kind, "graph": graph, "f32": rng.random() < 0.5, "steps": rng.randint(5, 20),
             "asserts": rng.random() < 0.5}
        if graph == "ba":
            return dict(c, n=_logu(rng, 20_000, 5_000_000), m=rng.randint(3, 6))
        if graph == "gnp":
            return dict(c, n=_logu(rng, 20_000, 5_000_000), deg=round(rng.uniform(4.0, 12.0), 2))
        return dict(c, n=_logu(rng, 500, 400_000), deg=round(rng.uniform(4.0, 20.0), 2))
    if kind == "batch":
        return {"kind": kind, "sims": rng.randint(4, 24), "n_min": 10_000, "n_max": 1_000_000,
                "deg": round(rng.uniform(4.0, 12.0), 2), "sizes": rng.randint(0, 1 << 20),
                "f32": rng.random() < 0.5, "steps": rng.randint(10, 20)}
    if kind == "sir":
        n = _logu(rng, 1_000, 300_000)
        return {"kind": kind, "n": n, "deg": round(rng.uniform(4.0, 16.0), 2), "p_inf": round(rng.uniform(0.01, 0.1), 4),
                "recovery": rng.randint(4, 14), "n_init": max(1, n // 1000), "steps": rng.randint(30, 100),
                "asserts": rng.random() < 0.5}
    if kind == "sweep":
        return {"kind": kind, "members": rng.randint(4, 48), "n_min": 1_000, "n_max": 1_000_000,
                "sizes": rng.randint(0, 1 << 20), "steps": rng.randint(50, 200)}
    if kind == "contact":
        return {"kind": kind, "n": _logu(rng, 10_000, 5_000_000), "contacts": rng.randint(5, 24),
                "p_death": round(rng.uniform(0.0, 0.04), 4), "steps": rng.randint(3, 6), "asserts": rng.random() < 0.5}
    if kind == "raster":
        return {"kind": kind, "nx": _logu(rng, 60, 3_162), "ny": _logu(rng, 60, 3_162),
                "periodic": rng.random() < 0.5, "distance": rng.randint(1, 2), "frac": 1e-4,
                "steps": rng.randint(10, 40), "asserts": rng.random() < 0.5}
    if kind == "neighbors":
        return {"kind": kind, "n": _logu(rng, 5_000, 1_000_000), "deg": round(rng.uniform(3.0, 16.0), 2),
                "steps": rng.randint(5, 10), "asserts": rng.random() < 0.5}
    if kind == "rewire":
        return {"kind": kind, "n": _logu(rng, 2_000, 300_000), "deg": round(rng.uniform(3.0, 10.0), 2),
                "steps": rng.randint(2, 5), "asserts": rng.random() < 0.5}
    return {"kind": kind, "n": _logu(rng, 10_000, 10_000_000)}


# ------------------------------------------------------------------ inputs
def _random_edges(n, deg, rng):
    """A user's edge list: round(n deg) edges between uniform agents, in no
    order (from, to as 1-based numbers)."""
    e = max(1, int(round(n * deg)))
    return rng.integers(1, n + 1, e), rng.integers(1, n + 1, e)


def _ids(nr):
    return TYPE1 | nr.astype(np.uint64)


def _opinion_inputs(case, seed):
    rng = np.random.default_rng(seed)
    n = case["n"]
    fr, to = _random_edges(n, case["deg"], rng)
    dt = np.float32 if case["f32"] else np.float64
    return rng.random(n).astype(dt), fr, to, (rng.random(len(fr)) * 0.998 + 0.001).astype(np.float32)


def _sizes(count, case):
    """Log-uniform sizes, mean degrees and infection probabilities of the
    members (the same for every seed, so that all inputs are the same work)."""
    rng = np.random.default_rng(case["sizes"])
    n = np.exp(rng.uniform(np.log(case["n_min"]), np.log(case["n_max"]), count))
    return [int(x) for x in n], rng.uniform(4.0, 20.0, count), rng.uniform(0.01, 0.1, count)


def _pinned(n, dtype):
    return torch.empty(max(n, 1), dtype=dtype, pin_memory=True)


def _read(sim, T, states, died=None):
    """vh_read_agents into the program's own buffers: the slots' states (and
    died flags)."""
    n = C.c_uint64()
    rc = sim.lib.read_agents(sim.handle, sim._aid(T), C.c_void_p(states.data_ptr()),
                             C.cast(died.data_ptr(), C.POINTER(C.c_uint8)) if died is not None else None,
                             states.numel(), C.byref(n))
    if rc:
        raise RuntimeError(sim.lib.last_error().decode())
    return n.value


def _opinion_types(f32):
    A = vh.struct("HK32", [("opinion", "<f4")]) if f32 else vh.struct("HK", [("opinion", "<f8")])
    E = vh.struct("Knows", [("w", "<f4")])
    model = (vh.ModelTypes() | vh.register_agenttype_(A, "Immortal") | vh.register_edgetype_(E, target=A)
             | vh.create_model("opinion"))
    return A, E, model


# ------------------------------------------------------------------ cases
class _Opinion:
    @staticmethod
    def prepare(case, seed):
        n, f32 = case["n"], case["f32"]
        if case["graph"] == "ba":
            m = vh.models.build_opinion(vh, n, m_ba=case["m"], seed=seed, f32=f32, device_graph=True)
        elif case["graph"] == "gnp":
            m = vh.models.build_opinion_gnp(vh, n, mean_deg=case["deg"], seed=seed, graph_seed=seed + 1,
                                            weight_seed=seed + 2, f32=f32)
        else:
            x, fr, to, w = _opinion_inputs(case, seed)
            A, E, model = _opinion_types(f32)
            sim = vh.create_simulation(model)
            st, ws = np.zeros(n, dtype=A.dtype), np.zeros(len(w), dtype=E.dtype)
            st["opinion"], ws["w"] = x, w
            sim._add_agents_array(A, st)
            sim._add_edges_array(E, _ids(fr), _ids(to), ws)
            vh.finish_init_(sim)
            m = types.SimpleNamespace(sim=sim, T=A, E=E, f32=f32)
        m.sim._opinion_prepare(m.T, m.E, f32)
        return types.SimpleNamespace(case=case, m=m, out=_pinned(n, torch.float32 if f32 else torch.float64))

    @staticmethod
    def run(s):
        m = s.m
        step = vh.transitions.opinion(m.E, EPS, m.f32)
        for _ in range(s.case["steps"]):
            vh.apply_(m.sim, step, m.T, [m.T, m.E], m.T)
        _read(m.sim, m.T, s.out)
        return s.out

    @staticmethod
    def work(case):
        n, sb = case["n"], 4 if case["f32"] else 8
        e = n * (2 * case["m"] if case["graph"] == "ba" else case["deg"])
        return {"bytes": case["steps"] * (2 * n * sb + 4 * n + 8 * e) + n * sb, "flops": case["steps"] * 5 * e}

    @staticmethod
    def exact(case, seed):
        # the device-generated graphs are not at hand without this
        # repository's generators
        if case["graph"] != "host":
            return None
        x, fr, to, w = _opinion_inputs(case, seed)
        x, w, n = x.astype(np.float64), w.astype(np.float64), case["n"]
        fr, to = fr - 1, to - 1
        for _ in range(case["steps"]):
            xf = x[fr]
            acc = np.where(np.abs(xf - x[to]) <= EPS, w, 0.0)
            den = np.bincount(to, weights=acc, minlength=n)
            num = np.bincount(to, weights=acc * xf, minlength=n)
            x = np.where(den > 0.0, num / np.where(den > 0.0, den, 1.0), x)
        return x


class _Batch:
    @staticmethod
    def prepare(case, seed):
        sizes, _, _ = _sizes(case["sims"], case)
        lib = vh._abi.lib()
        stream = C.c_void_p()
        lib.stream_create(C.byref(stream))
        f32 = case["f32"]
        ms = [vh.models.build_opinion_gnp(vh, n, mean_deg=case["deg"], seed=seed + k, graph_seed=seed + 100 + k,
                                          weight_seed=seed + 200 + k, f32=f32, stream=stream)
              for k, n in enumerate(sizes)]
        # one set of types for all (the batch takes the first simulation's)
        outs = [_pinned(n, torch.float32 if f32 else torch.float64) for n in sizes]
        return types.SimpleNamespace(case=case, ms=ms, outs=outs, batch=vh.Batch())

    @staticmethod
    def run(s):
        m0 = s.ms[0]
        vh.enable_asserts(False)   # as the serving loop runs them
        s.batch.apply([m.sim for m in s.ms], vh.transitions.opinion(m0.E, EPS, m0.f32), m0.T, [m0.T, m0.E], m0.T,
                      steps=s.case["steps"])
        for m, out in zip(s.ms, s.outs):
            _read(m.sim, m.T, out)
        return s.outs

    @staticmethod
    def work(case):
        n, sb = sum(_sizes(case["sims"], case)[0]), 4 if case["f32"] else 8
        e = n * case["deg"]
        return {"bytes": case["steps"] * (2 * n * sb + 4 * n + 8 * e) + n * sb, "flops": case["steps"] * 5 * e}


class _Sir:
    @staticmethod
    def prepare(case, seed):
        n = case["n"]
        rng = np.random.default_rng(seed)
        fr, to = _random_edges(n, case["deg"], rng)
        A = vh.struct("SIR", [("health", "u1"), ("pad", "u1"), ("days", "<u2")])
        E = vh.struct("Contact")
        st = np.zeros(n, dtype=A.dtype)
        st["health"][rng.choice(n, case["n_init"], replace=False)] = vh.I
        return types.SimpleNamespace(case=case, seed=seed, A=A, E=E, st=st, fr=_ids(fr), to=_ids(to),
                                     out=_pinned(n, torch.int32))

    @staticmethod
    def run(s):
        c = s.case
        model = (vh.ModelTypes() | vh.register_agenttype_(s.A, "Immortal")
                 | vh.register_edgetype_(s.E, "Stateless", target=s.A) | vh.create_model("sir"))
        sim = vh.create_simulation(model)
        sim._add_agents_array(s.A, s.st)
        sim._add_edges_array(s.E, s.fr, s.to)
        vh.finish_init_(sim)
        step = vh.transitions.sir(s.E, c["p_inf"], s.seed, c["recovery"])
        for _ in range(c["steps"]):
            vh.apply_(sim, step, s.A, [s.A, s.E], s.A)
        _read(sim, s.A, s.out)
        vh.finish_simulation_(sim)
        return s.out

    @staticmethod
    def work(case):
        n, e = case["n"], case["n"] * case["deg"]
        # the edge list read, its CSR written; every day the states; each edge
        # once while its source is infected
        return {"bytes": 4 * n + 16 * e + 4 * n + 4 * e + case["steps"] * 8 * n + 4 * e + 4 * n, "flops": 0}


class _Sweep:
    @staticmethod
    def prepare(case, seed):
        return types.SimpleNamespace(case=case, seed=seed, sizes=_sizes(case["members"], case))

    @staticmethod
    def run(s):
        ens = vh.ensemble.Ensemble()
        ids = [ens.add_sir(n, deg, p, s.seed + 3 * k, s.seed + 3 * k + 1, n_init=max(10, n // 1000))
               for k, (n, deg, p) in enumerate(zip(*s.sizes))]
        ens.step(s.case["steps"])
        outs = [ens.read(i)[0].view(np.int32) for i in ids]
        ens.close()
        return outs

    @staticmethod
    def work(case):
        sizes, deg, _ = _sizes(case["members"], case)
        n, e = sum(sizes), float(np.dot(sizes, deg))
        # the graphs written, every day the states, each edge once while its
        # source is infected
        return {"bytes": 8 * n + 4 * e + case["steps"] * 8 * n + 4 * e + 4 * n, "flops": 0}


class _Contact:
    @staticmethod
    def prepare(case, seed):
        n = case["n"]
        rng = np.random.default_rng(seed)
        A = vh.struct("Person", [("health", "u1"), ("susc", "<f4")])
        E = vh.struct("Met")
        model = (vh.ModelTypes() | vh.register_agenttype_(A) | vh.register_edgetype_(E, "Stateless", target=A)
                 | vh.create_model("contact"))
        sim = vh.create_simulation(model)
        st = np.zeros(n, dtype=A.dtype)
        # the endemic state: shares of susceptible, infected and recovered
        st["health"] = rng.choice(np.array([vh.S, vh.I, vh.R], np.uint8), n, p=[0.15, 0.15, 0.7])
        st["susc"] = 0.5 + 0.5 * rng.random(n, dtype=np.float32)
        sim._add_agents_array(A, st)
        vh.finish_init_(sim)
        # slots: the agents and the newborns that find no free slot
        cap = n + n // 8 + 64
        s = types.SimpleNamespace(case=case, seed=seed, sim=sim, A=A, E=E, out=_pinned(cap, torch.int64).zero_(),
                                  died=_pinned(cap, torch.uint8).zero_())
        _Contact.step(s)   # the first contacts
        return s

    @staticmethod
    def step(s):
        c = s.case
        body = vh.transitions.contact(s.E, 0.05, 0.1, c["p_death"], s.seed, c["contacts"])
        vh.apply_(s.sim, body, s.A, [s.A, s.E], [s.A, s.E])

    @staticmethod
    def run(s):
        for _ in range(s.case["steps"]):
            _Contact.step(s)
        n = _read(s.sim, s.A, s.out, s.died)
        return [s.out, s.died, n, vh.num_edges(s.sim, s.E)]

    @staticmethod
    def work(case):
        n, e = case["n"], case["n"] * case["contacts"]
        return {"bytes": case["steps"] * (17 * n + 8 * n + 8 * e) + 9 * n, "flops": 0}


class _Raster:
    @staticmethod
    def prepare(case, seed):
        nx, ny = case["nx"], case["ny"]
        rng = np.random.default_rng(seed)
        A = vh.struct("Cell", [("active", "?")])
        E = vh.struct("Adj")
        model = (vh.ModelTypes() | vh.register_agenttype_(A, "Immortal")
                 | vh.register_edgetype_(E, "Stateless", target=A) | vh.create_model("raster"))
        sim = vh.create_simulation(model)
        st = np.zeros(nx * ny, dtype=A.dtype)
        st["active"][rng.integers(0, nx * ny, max(1, int(nx * ny * case["frac"])))] = True
        vh.raster.add_raster_(sim, "grid", (nx, ny), st, T=A)
        vh.raster.connect_raster_neighbors_(sim, "grid", E(), distance=case["distance"], periodic=case["periodic"])
        vh.finish_init_(sim)
        return types.SimpleNamespace(case=case, sim=sim, A=A, E=E, out=_pinned(nx * ny, torch.uint8))

    @staticmethod
    def run(s):
        sim = vh.copy_simulation(s.sim)
        body = vh.transitions.diffuse(s.E, s.A)
        for _ in range(s.case["steps"]):
            vh.apply_(sim, body, s.A, [s.A, s.E], s.A)
        _read(sim, s.A, s.out)
        vh.finish_simulation_(sim)
        return s.out

    @staticmethod
    def work(case):
        n = case["nx"] * case["ny"]
        side = 2 * case["distance"] + 1
        # the copy (states, offsets, stencil edges read and written) and the steps
        return {"bytes": 2 * (n + 4 * n + 4 * n * (side * side - 1)) + case["steps"] * 2 * n + n, "flops": 0}


class _Neighbors:
    @staticmethod
    def prepare(case, seed):
        n = case["n"]
        rng = np.random.default_rng(seed)
        fr, to = _random_edges(n, case["deg"], rng)
        A = vh.struct("Agent", [("foo", "<i8")])
        E = vh.struct("Link")
        model = (vh.ModelTypes() | vh.register_agenttype_(A, "Immortal")
                 | vh.register_edgetype_(E, "Stateless", target=A) | vh.create_model("neighbors"))
        sim = vh.create_simulation(model)
        st = np.zeros(n, dtype=A.dtype)
        st["foo"] = rng.integers(0, 100, n)
        sim._add_agents_array(A, st)
        sim._add_edges_array(E, _ids(fr), _ids(to))
        vh.finish_init_(sim)
        return types.SimpleNamespace(case=case, sim=sim, A=A, E=E, out=_pinned(n, torch.int64))

    @staticmethod
    def run(s):
        body = vh.transitions.sum_neighbors(s.E)
        for _ in range(s.case["steps"]):
            vh.apply_(s.sim, body, s.A, [s.A, s.E], s.A)
        _read(s.sim, s.A, s.out)
        return s.out

    @staticmethod
    def work(case):
        n, e = case["n"], case["n"] * case["deg"]
        return {"bytes": case["steps"] * (16 * n + 4 * n + 4 * e) + 8 * n, "flops": case["steps"] * e}


class _Rewire:
    @staticmethod
    def prepare(case, seed):
        n = case["n"]
        rng = np.random.default_rng(seed)
        fr, to = _random_edges(n, case["deg"], rng)
        A = vh.struct("Agent", [("foo", "<i8")])
        E = vh.struct("Link")
        F = vh.struct("Message", [("foo", "<i8")])
        model = (vh.ModelTypes() | vh.register_agenttype_(A, "Immortal")
                 | vh.register_edgetype_(E, "Stateless", target=A) | vh.register_edgetype_(F, target=A)
                 | vh.create_model("rewire"))
        sim = vh.create_simulation(model)
        st = np.zeros(n, dtype=A.dtype)
        st["foo"] = rng.integers(0, 100, n)
        sim._add_agents_array(A, st)
        sim._add_edges_array(E, _ids(fr), _ids(to))
        vh.finish_init_(sim)
        return types.SimpleNamespace(case=case, sim=sim, A=A, E=E, F=F, out=_pinned(n, torch.int64))

    @staticmethod
    def run(s):
        send = vh.transitions.neighbor_foo_edges(s.E, s.F, -1)
        take = vh.transitions.sum_neighbors(s.F)
        for _ in range(s.case["steps"]):
            vh.apply_(s.sim, send, s.A, [s.A, s.E], s.F)
            vh.apply_(s.sim, take, s.A, [s.A, s.F], s.A)
        _read(s.sim, s.A, s.out)
        return [s.out, vh.mapreduce(s.sim, "foo", "+", s.F), vh.num_edges(s.sim, s.F)]

    @staticmethod
    def work(case):
        n, e = case["n"], case["n"] * case["deg"]
        # the links read, twice as many messages written (source, state) and
        # read (source), the states read and written
        return {"bytes": case["steps"] * (8 * n + 8 * n + 4 * e + 2 * e * (12 + 4) + 16 * n) + 8 * n,
                "flops": case["steps"] * 2 * e}


class _Stats:
    @staticmethod
    def inputs(case, seed):
        rng = np.random.default_rng(seed)
        n = case["n"]
        return rng.random(n) * 100.0, rng.random(n, dtype=np.float32), rng.integers(0, 8, n).astype(np.uint8)

    @staticmethod
    def prepare(case, seed):
        wealth, income, group = _Stats.inputs(case, seed)
        A = vh.struct("Household", [("wealth", "<f8"), ("income", "<f4"), ("group", "u1")])
        model = vh.ModelTypes() | vh.register_agenttype_(A, "Immortal") | vh.create_model("stats")
        sim = vh.create_simulation(model)
        st = np.zeros(case["n"], dtype=A.dtype)
        st["wealth"], st["income"], st["group"] = wealth, income, group
        sim._add_agents_array(A, st)
        vh.finish_init_(sim)
        return types.SimpleNamespace(case=case, sim=sim, A=A)

    @staticmethod
    def run(s):
        f, sim, A = vh.expr.field, s.sim, s.A
        return [vh.mapreduce(sim, "wealth", "+", A), vh.mapreduce(sim, "income", "max", A),
                vh.mapreduce(sim, "wealth", "min", A), vh.mapreduce(sim, vh.Field("group", 3), "+", A),
                vh.mapreduce(sim, f("wealth") * f("income"), "+", A), vh.mapreduce(sim, f("wealth") > 50.0, "+", A)]

    @staticmethod
    def work(case):
        return {"bytes": case["n"] * (8 + 4 + 8 + 1 + 12 + 8), "flops": 8 * case["n"]}

    @staticmethod
    def exact(case, seed):
        wealth, income, group = _Stats.inputs(case, seed)
        return [math.fsum(wealth), float(income.max()), float(wealth.min()), int((group == 3).sum()),
                math.fsum(wealth * income.astype(np.float64)), int((wealth > 50.0).sum())]


KINDS = {"opinion": _Opinion, "batch": _Batch, "sir": _Sir, "sweep": _Sweep, "contact": _Contact, "raster": _Raster,
         "neighbors": _Neighbors, "rewire": _Rewire, "stats": _Stats}


def prepare(case, seed):
    return KINDS[case["kind"]].prepare(case, seed)


def run(state):
    vh.enable_asserts(state.case.get("asserts", True))
    return KINDS[state.case["kind"]].run(state)


def work(case):
    return KINDS[case["kind"]].work(case)


def exact(case, seed):
    f = getattr(KINDS[case["kind"]], "exact", None)
    return f(case, seed) if f else None
