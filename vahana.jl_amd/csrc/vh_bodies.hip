// vh_bodies.hip — transition bodies as HIP device code.
//
// Generic bodies run thread-per-slot through k_generic (the agent loop of
// src/AgentMethods.jl:193-245 with the write policy of :159-181); the model
// bodies (SIR, weighted bounded confidence, dynamic contacts) have their own
// kernels over the CSR.
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <atomic>

#include "vh_engine.h"

using namespace vh;

namespace {

// ----------------------------------------------------------------- bodies
template <int TR>
struct Body;

template <>
struct Body<VH_TR_NOOP> {
    __device__ static bool run(const DCtx*, const uint8_t*, uint64_t, Emitter&, uint8_t*) { return true; }
};
// neighborids is not defined for :IgnoreFrom types: they keep no sources
__device__ __forceinline__ bool has_sources(const DCtx* c, const DEdge& E) {
    if (!VH_HAS(E.hints, VH_HINT_IGNOREFROM)) return true;
    vh_flag(c, VH_DERR_HINT);
    return false;
}
// create_sum_state_neighbors test/core.jl:71-83
template <>
struct Body<VH_TR_SUM_NEIGHBORS> {
    __device__ static bool run(const DCtx* c, const uint8_t*, uint64_t id, Emitter&, uint8_t* out) {
        int et = c->role_e[0];
        uint32_t b, e;
        int64_t sum = 0;
        if (d_row(c, et, id, b, e)) {
            const DEdge& E = c->e[et];
            if (!has_sources(c, E)) return true;
            const Neighbors nb(c, et);
            constexpr int SUM_N = 8;
            const uint8_t* n[SUM_N];
            uint32_t k = b;
            for (; k < e && nb.some(k, e, n); k = vh_row_next(k, e, SUM_N)) {
                int64_t v[SUM_N];
#pragma unroll
                for (int q = 0; q < SUM_N; q++) v[q] = ld_i64(n[q]);
#pragma unroll
                for (uint32_t q = 0; q < SUM_N; q++) sum += q < e - k ? v[q] : 0;
            }
            for (; k < e; k++) {
                const uint8_t* ns = nb.state(k);
                if (!ns) return true;
                sum += ld_i64(ns);
            }
        }
        st_i64(out, sum);
        return true;
    }
};
__device__ bool pred(const DCtx* c, const uint8_t* st, uint64_t id) {
    const vh_test_params* p = (const vh_test_params*)c->params;
    int64_t foo = c->a[vh_type_of(id)].bytes >= 8 ? ld_i64(st) : 0;
    switch (p->cmp) {
    case VH_CMP_ALWAYS: return true;
    case VH_CMP_NEVER: return false;
    case VH_CMP_LT: return foo < p->value;
    case VH_CMP_GE: return foo >= p->value;
    case VH_CMP_EQ: return foo == p->value;
    case VH_CMP_ODD: return (foo % 2) != 0;
    case VH_CMP_EVEN: return (foo % 2) == 0;
    case VH_CMP_NUM_EDGES_EQ: {
        uint32_t b, e;
        d_row(c, c->role_e[0], id, b, e);
        return (int64_t)(e - b) == p->value;
    }
    }
    return false;
}
template <>
struct Body<VH_TR_DIE_IF> {
    __device__ static bool run(const DCtx* c, const uint8_t* st, uint64_t id, Emitter&, uint8_t*) {
        return !pred(c, st, id);
    }
};
template <>
struct Body<VH_TR_ADD_SELF_EDGE> {
    __device__ static bool run(const DCtx* c, const uint8_t*, uint64_t id, Emitter& em, uint8_t*) {
        const vh_test_params* p = (const vh_test_params*)c->params;
        em.edge(id, id, p->edge_state);
        return true;
    }
};
// add_edges!(sim, id, edges(sim, id, ET)) test/edges.jl:357-359
template <>
struct Body<VH_TR_READD_EDGES> {
    __device__ static bool run(const DCtx* c, const uint8_t*, uint64_t id, Emitter& em, uint8_t*) {
        int et = c->role_e[0];
        uint32_t b, e;
        if (!d_row(c, et, id, b, e)) return true;
        const DEdge& E = c->e[et];
        for (uint32_t k = b; k < e; k++) {
            uint64_t from = VH_HAS(E.hints, VH_HINT_IGNOREFROM) ? 0 : vh_src_id(E, k);
            em.edge(from, id, E.st + (uint64_t)k * E.bytes);
        }
        return true;
    }
};
// test/independent.jl:55-68
template <>
struct Body<VH_TR_NEIGHBOR_FOO_EDGES> {
    __device__ static bool run(const DCtx* c, const uint8_t* st, uint64_t id, Emitter& em, uint8_t*) {
        const vh_test_params* p = (const vh_test_params*)c->params;
        int64_t foo = ld_i64(st);
        if (foo == p->value) return false;
        int et = c->role_e[0];
        uint32_t b, e;
        if (d_row(c, et, id, b, e)) {
            const DEdge& E = c->e[et];
            if (!has_sources(c, E)) return true;
            uint8_t es[8];
            st_i64(es, foo);
            const Sources src(E);
            for (uint32_t k = b; k < e; k = vh_row_next(k, e, 4)) {
                uint64_t nid[4];
                src.four(k, e, nid);
                uint64_t f[8], t[8];
#pragma unroll
                for (uint32_t q = 0; q < 4; q++) {
                    f[2 * q] = t[2 * q + 1] = nid[q];
                    t[2 * q] = f[2 * q + 1] = id;
                }
                em.edges(f, t, 2 * min(e - k, 4u), es);
            }
        }
        return true;
    }
};
// test/independent.jl:165-176 (value births of T(foo + 10j)); cmp selects
// the edges: 0 both directions with the newborn id as state (independent.jl),
// 1 newborn -> caller only (test/addexisting.jl:41-44)
template <>
struct Body<VH_TR_SPAWN> {
    __device__ static bool run(const DCtx* c, const uint8_t* st, uint64_t id, Emitter& em, uint8_t*) {
        const vh_test_params* p = (const vh_test_params*)c->params;
        int at = c->role_a[0];
        uint8_t ns[VH_MAX_STATE];
        uint32_t bytes = at > 0 ? c->a[at].bytes : 0u;
        uint32_t cbytes = c->a[vh_type_of(id)].bytes;
        for (int64_t j = 1; j <= p->value; j++) {
            for (uint32_t k = 0; k < bytes; k++) ns[k] = k < cbytes ? st[k] : 0;
            if (bytes >= 8 && cbytes >= 8) st_i64(ns, ld_i64(st) + 10 * j);
            uint64_t nid = em.agent(ns);
            if (c->role_e[0] >= 0) {
                uint8_t es[8];
                st_i64(es, (int64_t)nid);
                em.edge(nid, id, es);
                if (p->cmp == 0) em.edge(id, nid, es);
            }
        }
        return true;
    }
};
template <>
struct Body<VH_TR_COUNT_EDGES> {
    __device__ static bool run(const DCtx* c, const uint8_t*, uint64_t id, Emitter&, uint8_t* out) {
        uint32_t b, e;
        d_row(c, c->role_e[0], id, b, e);
        st_i64(out, (int64_t)(e - b));
        return true;
    }
};

// diffuse test/raster.jl:38-41 (diffuse3D :143-146): the Bool field at
// `field_offset` becomes true when it is, or when any in-neighbour's is
template <>
struct Body<VH_TR_DIFFUSE> {
    __device__ static bool run(const DCtx* c, const uint8_t* st, uint64_t id, Emitter&, uint8_t* out) {
        const vh_raster_params* p = (const vh_raster_params*)c->params;
        const uint32_t f = p->field_offset;
        uint8_t v = st[f] ? 1 : 0;
        int et = c->role_e[0];
        uint32_t b, e;
        if (!v && d_row(c, et, id, b, e)) {
            const DEdge& E = c->e[et];
            if (!has_sources(c, E)) return true;
            for (uint32_t k = b; k < e && !v; k++) {
                const uint8_t* ns = d_state(c, vh_src_id(E, k));
                if (!ns) return true;
                v = ns[f] ? 1 : 0;
            }
        }
        out[f] = v;
        return true;
    }
};
// value_on_pos test/raster.jl:279-285: v = the Int64 at offset 0 of the
// first in-neighbour over E; move_to!(sim, raster, id, (v, ..., v), E(), E())
// with distance 0 (src/Raster.jl:437-463): edge cell -> id, then id -> cell;
// the new state is v at offset 0
template <>
struct Body<VH_TR_MOVE_TO> {
    __device__ static bool run(const DCtx* c, const uint8_t*, uint64_t id, Emitter& em, uint8_t* out) {
        const vh_raster_params* p = (const vh_raster_params*)c->params;
        int et = c->role_e[0];
        uint32_t b, e;
        if (!d_row(c, et, id, b, e)) {   // first(nothing) fails in the reference
            vh_flag(c, VH_DERR_TARGET);
            return true;
        }
        if (!has_sources(c, c->e[et])) return true;
        const uint8_t* ns = d_state(c, vh_src_id(c->e[et], b));
        if (!ns) return true;
        const int64_t v = ld_i64(ns);
        uint64_t lin = 0, stride = 1;
        for (uint32_t d = 0; d < p->ndims && d < 4; d++) {
            if (v < 1 || v > p->dims[d]) {   // raster[pos] out of bounds
                vh_flag(c, VH_DERR_TARGET);
                return true;
            }
            lin += (uint64_t)(v - 1) * stride;
            stride *= (uint64_t)p->dims[d];
        }
        const uint64_t cell = vh_make_id(p->cell_type, p->first_nr + lin);
        if (p->flags & 1u) em.edge(cell, id, p->edge_state);
        if (p->flags & 2u) em.edge(id, cell, p->edge_state);
        st_i64(out, v);
        return true;
    }
};

// remove_edges! bodies of test/mpi/test_edgetypes.jl:295-445 (enum
// vh_remove_mode); `idx` is the Int64 at offset 0 of the caller's state
template <>
struct Body<VH_TR_REMOVE_EDGES> {
    // first (or second) in-neighbour of `id` over `et`; false when it has fewer
    __device__ static bool nth_neighbor(const DCtx* c, int et, uint64_t id, uint32_t n, uint64_t& out) {
        uint32_t b, e;
        if (!d_row(c, et, id, b, e) || e - b <= n) return false;
        const DEdge& E = c->e[et];
        if (!has_sources(c, E)) return false;
        out = vh_src_id(E, b + n);
        return true;
    }
    __device__ static bool run(const DCtx* c, const uint8_t* st, uint64_t id, Emitter& em, uint8_t*) {
        const vh_test_params* p = (const vh_test_params*)c->params;
        const int64_t idx = ld_i64(st);
        const int et = c->role_e[0], es = c->role_e[1];
        uint64_t nb = 0, nb2 = 0;
        switch ((int)p->value) {
        case VH_RM_OWN:
            if (idx % 2 == 0) em.remove(0, id, true);
            break;
        case VH_RM_NEIGHBOR:
            if (idx % 2 == 0) {
                if (!nth_neighbor(c, et, id, 0, nb)) vh_flag(c, VH_DERR_TARGET);
                else em.remove(0, nb, true);
            }
            break;
        case VH_RM_READD:
            if (!nth_neighbor(c, et, id, 0, nb)) {
                vh_flag(c, VH_DERR_TARGET);
                break;
            }
            em.remove(nb, id, false);
            em.edge(nb, id, p->edge_state);
            break;
        case VH_RM_FROM_TWO: {
            const bool single = VH_HAS(c->e[et].hints, VH_HINT_SINGLEEDGE);
            if (!nth_neighbor(c, et, id, 0, nb) || (!single && !nth_neighbor(c, et, id, 1, nb2))) {
                vh_flag(c, VH_DERR_TARGET);
                break;
            }
            em.remove(nb, id, false);
            if (!single) em.remove(nb2, id, false);
            break;
        }
        case VH_RM_TO_NEIGHBOR:
            if (idx % 2 == 0) {
                if (!nth_neighbor(c, et, id, 0, nb)) vh_flag(c, VH_DERR_TARGET);
                else em.remove(id, nb, false);
            }
            break;
        case VH_RM_SEND_ID:   // the log is bound to SendId (role_edge[1])
            if (!nth_neighbor(c, et, id, 0, nb)) vh_flag(c, VH_DERR_TARGET);
            else em.edge(id, nb, p->edge_state);
            break;
        case VH_RM_TO_SENDID:
            if (idx < 100) {
                if (!nth_neighbor(c, es, id, 0, nb)) vh_flag(c, VH_DERR_TARGET);
                else em.remove(id, nb, false);
            }
            break;
        case VH_RM_ZERO_FROM:
            em.remove(0, id, false);
            break;
        }
        return true;
    }
};

template <int TR>
__global__ __launch_bounds__(256) void k_generic(const DCtx* __restrict__ c, int ci, int t, int pass,
                                                 int with_edge) {
    vh_generic_call<Body<TR>>(c, ci, t, pass, with_edge);
}

// inclusive sum over the lanes of a wave up to each lane (DPP: shifts within
// rows of 16 lanes, then the row totals broadcast to the rows after them)
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, false);   // row_shr:1
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xF, 0xF, false);   // row_shr:2
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xF, 0xF, false);   // row_shr:4
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xF, 0xF, false);   // row_shr:8
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, false);   // row_bcast:15
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xC, 0xF, false);   // row_bcast:31
    return v;
}

// ----------------------------------------------------------------- SIR
// state word: health byte 0, pad byte 1, days bytes 2-3
// Exposure pass: every infected agent (read state) sets the bit of each of
// its out-neighbours in this launch's bitmap. A susceptible agent without the
// bit has no infected in-neighbour, so "some in-edge with an infected source
// and a draw below p" is false without drawing: k_sir skips its draws. (A bit
// too many only makes an agent draw.) The pass runs while the infected are few:
// k_sir counts the infected agents it writes into 64 counters (one atomic per
// block), whose sum decides in the next launch: every wave of the pass adds
// them up for itself, and its first block leaves the decision for k_sir.
// Counters and bitmaps are two of each, by launch parity: the pass clears the
// other counters, k_sir its agents' words of the other bitmap. With a launch each
// for the clearing and the decision, a step of 10^5 agents took 13 us of
// kernels and as many gaps more, so 7.5.
// Words of `ctl`: [0, 128) counters (parity * 64 + j), 128 + parity: the
// counters of that parity are complete, 130: the decision.
constexpr uint32_t SIR_CTL_WORDS = 131;

// four consecutive agents per lane; marks as vh_expose_wave does
__global__ __launch_bounds__(256) void k_sir_expose(const uint32_t* __restrict__ rs,
                                                    const uint32_t* __restrict__ out_off,
                                                    const uint32_t* __restrict__ out_dst, uint64_t n,
                                                    uint32_t parity, uint32_t* __restrict__ ctl,
                                                    uint32_t* __restrict__ expo) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)wave_incl_scan(ctl[parity * 64 + lane]), 63);
    const bool on = ctl[128 + parity] && (uint64_t)total * 32 <= n;
    if (blockIdx.x == 0 && threadIdx.x < 64) {
        ctl[(parity ^ 1u) * 64 + lane] = 0u;
        if (lane == 0) {
            ctl[130] = on ? 1u : 0u;
            ctl[128 + (parity ^ 1u)] = 1u;   // this launch's k_sir fills the other set
        }
    }
    if (!on) return;   // uniform
    const uint64_t i = ((uint64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    const uint32_t in = i >= n ? 0u : n - i < 4 ? (uint32_t)(n - i) : 4u;
    u32x4 v = {0u, 0u, 0u, 0u};
    if (in == 4) v = *(const u32x4*)(rs + i);
    else
        for (uint32_t q = 0; q < in; q++) v[q] = rs[i + q];
#pragma unroll
    for (uint32_t q = 0; q < 4; q++) vh_expose_wave(q < in && (v[q] & 0xFFu) == VH_I, i + q, out_off, out_dst, expo);
}

__global__ __launch_bounds__(256) void k_sir(const uint32_t* __restrict__ off,
                                             const uint32_t* __restrict__ src,
                                             const uint32_t* __restrict__ rs,
                                             uint32_t* __restrict__ ws, uint64_t n, uint64_t nrows,
                                             uint64_t rowbase, uint32_t t, double p, uint64_t seed,
                                             uint32_t rec, uint64_t step, const uint32_t* __restrict__ expo,
                                             uint32_t* __restrict__ expo_next, uint32_t parity,
                                             uint32_t* __restrict__ ctl) {
    __shared__ uint32_t s_inf[4];
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool in = i < n;
    uint32_t s = in ? rs[i] : 0u;
    uint32_t h = s & 0xFFu;
    const bool skip = in && h == VH_S && ctl && ctl[130] && !((expo[i >> 5] >> (i & 31u)) & 1u);
    if (ctl && in && (i & 31u) == 0) expo_next[i >> 5] = 0u;
    if (in && h == VH_S && !skip) {
        if (i < nrows) {
            const uint64_t pre = vh_hash_pre(seed, vh_make_id(t, i + 1), step);
            const uint64_t pt = vh_u01_below(p);
            uint32_t b = off[rowbase + i], e = off[rowbase + i + 1];
            // "some in-edge k has an infected source and u_k < p" is
            // order-free: the draw (ALU) first, the source's state (a random
            // gather) only for the few draws below p
            if (vh_any_infecting(pre, pt, b, e, [&](uint32_t k) { return (rs[src[k] - 1] & 0xFFu) == VH_I; }))
                s = (s & 0xFF00u) | VH_I;
        }
    } else if (in && h == VH_I) {
        uint32_t days = ((s >> 16) + 1u) & 0xFFFFu;
        s = (s & 0xFF00u) | (days << 16) | (days >= rec ? VH_R : VH_I);
    }
    if (in) ws[i] = s;
    if (ctl) {   // infected agents of the written state, for the next step
        const uint64_t m = __ballot(in && (s & 0xFFu) == VH_I);
        if ((threadIdx.x & 63u) == 0) s_inf[threadIdx.x >> 6] = (uint32_t)__popcll(m);
        __syncthreads();
        if (threadIdx.x == 0) {
            const uint32_t c = s_inf[0] + s_inf[1] + s_inf[2] + s_inf[3];
            if (c) atomicAdd(ctl + (parity ^ 1u) * 64 + (blockIdx.x & 63u), c);
        }
    }
}

// ----------------------------------------------------------------- opinion
// Weighted bounded confidence: x_i <- sum_{j: |x_j - x_i| <= eps} w x_j /
// sum w over the in-edges; x_i when none is accepted. Canonical order of both
// sums: degree <= 64 sequential in CSR (insertion) order; degree > 64 lane l
// of 64 adds k = l, l + 64, ... in order, then the xor butterfly
// p[l] + p[l ^ o], o = 32..1. A rejected neighbour adds +0.0, which is
// bit-identical to skipping it (the sums start at +0.0 and every term is
// >= +0.0). Agents of degree <= 64 are light (thread per agent in a 256-agent
// block), the others heavy (one wave each).
template <class T>
__device__ __forceinline__ void op_accum(T xj, float w, T xi, T eps, T& num, T& den) {
    const bool acc = fabs(xj - xi) <= eps;
    num = num + (acc ? (T)w * xj : (T)0);
    den = den + (acc ? (T)w : (T)0);
}

// the value of lane l ^ O (O = 1, 2: DPP quad permutations; 4, 8, 16:
// ds_swizzle in bitmask mode; 32: ds_bpermute)
template <int O>
__device__ __forceinline__ uint32_t lane_xor(uint32_t v) {
    if constexpr (O == 1) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, false);
    else if constexpr (O == 2) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, false);
    else if constexpr (O <= 16) return (uint32_t)__builtin_amdgcn_ds_swizzle((int)v, (O << 10) | 0x1F);
    else return (uint32_t)__shfl_xor((int)v, O, 64);
}
template <int O, class T>
__device__ __forceinline__ T lane_xor_t(T v) {
    if constexpr (sizeof(T) == 8) {
        const uint64_t u = __builtin_bit_cast(uint64_t, v);
        const uint64_t r = (uint64_t)lane_xor<O>((uint32_t)u) | (uint64_t)lane_xor<O>((uint32_t)(u >> 32)) << 32;
        return __builtin_bit_cast(T, r);
    } else {
        return __builtin_bit_cast(T, lane_xor<O>(__builtin_bit_cast(uint32_t, v)));
    }
}
// p[l] + p[l ^ o] for o = 32, 16, ..., 1: every lane ends with the sum in
// the canonical order of the wave-per-agent path
template <class T>
__device__ __forceinline__ T xor_butterfly(T v) {
    v = v + lane_xor_t<32>(v);
    v = v + lane_xor_t<16>(v);
    v = v + lane_xor_t<8>(v);
    v = v + lane_xor_t<4>(v);
    v = v + lane_xor_t<2>(v);
    v = v + lane_xor_t<1>(v);
    return v;
}

// block exclusive scan of the light degrees: the thread's first slot in the
// block's light edges and their total
__device__ __forceinline__ uint32_t op_light_scan(uint32_t ld, uint32_t* s_wsum, uint32_t& total) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const uint32_t incl = wave_incl_scan(ld);
    if (lane == 63) s_wsum[wv] = incl;
    __syncthreads();
    uint32_t pre = 0;
    total = 0;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const uint32_t v = s_wsum[q];
        pre += q < wv ? v : 0u;
        total += v;
    }
    return pre + incl - ld;
}

// -- one pass (state vectors below the plan threshold). The light edges of a
// block are processed in tiles of OP_TILE slots: all threads load sources and
// weights coalesced and gather OP_U neighbour states each, staging state and
// weight by slot in LDS; then every thread adds its own agent's slots.
//
// The rows of a block without heavy agents are one range of the CSR: slot q
// is in-edge b0 + q, and an agent's slots start at its own offset. Only a
// block with a heavy agent (its rows are skipped) has to number its slots by
// a scan and look up each slot's agent in LDS. us per step with the lookup in
// every block, without it, and tiles of 3072 slots (the mean block of 10 to 12
// in-edges an agent in one tile) in place of 2048: 1501 Float32 agents 8.9,
// 5.5, 4.5 (a chain of latencies); 2 10^5 Float64 agents 23.3, 19.4, 19.3; 24
// simulations of 5.8 10^6 agents in all 462, 408, 405, where the neighbours'
// lines from beyond the L2 bound it (about 9 TB/s).
constexpr int OP_TILE = 3072;
constexpr int OP_U = OP_TILE / 256;   // gathers in flight per thread

template <class T>
struct OpLDS {
    T x[OP_TILE];
    float w[OP_TILE];
    uint8_t own[OP_TILE];   // blocks with heavy agents: agent of each slot,
    uint32_t b[256], p[256], wsum[4];   // its first in-edge, its first slot
};

// the slots [lo, hi) of an agent, staged from t0 on, added in order
template <class T>
__device__ __forceinline__ void op_sum_slots(const OpLDS<T>& sm, uint32_t lo, uint32_t hi, uint32_t t0, T xi, T eps,
                                             T& num, T& den) {
    uint32_t p = lo;
    for (; p + 4 <= hi; p += 4) {   // (four slots' reads ahead of their sums)
        const uint32_t q = p - t0;
        const T x0 = sm.x[q], x1 = sm.x[q + 1], x2 = sm.x[q + 2], x3 = sm.x[q + 3];
        const float w0 = sm.w[q], w1 = sm.w[q + 1], w2 = sm.w[q + 2], w3 = sm.w[q + 3];
        op_accum(x0, w0, xi, eps, num, den);
        op_accum(x1, w1, xi, eps, num, den);
        op_accum(x2, w2, xi, eps, num, den);
        op_accum(x3, w3, xi, eps, num, den);
    }
    for (; p < hi; p++) op_accum(sm.x[p - t0], sm.w[p - t0], xi, eps, num, den);
}

//
// STREAM (op_stream): sources and weights are read non-temporally, which leaves
// more of the caches to the states (the 24 simulations, 468 MB of edges: 405 ->
// 377 us).
template <class V, bool STREAM>
__device__ __forceinline__ V op_edge(const V* p) {
    if constexpr (STREAM) return __builtin_nontemporal_load(p);
    else return *p;
}
template <class T, bool STREAM>
__device__ __forceinline__ void opinion_block(const uint32_t* __restrict__ off,
                                              const uint32_t* __restrict__ src,
                                              const T* __restrict__ x, const float* __restrict__ w,
                                              T* __restrict__ xo, uint64_t n, uint64_t nrows,
                                              uint64_t rowbase, T eps, uint32_t blk) {
    __shared__ OpLDS<T> sm;
    const int tid = threadIdx.x;
    const uint64_t i0 = (uint64_t)blk * 256, i = i0 + tid;
    const uint64_t r0 = i0 < nrows ? i0 : nrows, r1 = i0 + 256 < nrows ? i0 + 256 : nrows;
    const uint32_t b0 = nrows ? off[rowbase + r0] : 0u, e0 = nrows ? off[rowbase + r1] : 0u;   // the block's in-edges
    uint32_t b = 0, d = 0;
    T xi = (T)0;
    if (i < n) {
        xi = x[i];
        if (i < nrows) {
            b = off[rowbase + i];
            d = off[rowbase + i + 1] - b;
        }
    }
    const bool light = i < n && d <= 64u;
    T num = (T)0, den = (T)0;
    if (!__syncthreads_or(d > 64u)) {
        const uint32_t P = b - b0, total = e0 - b0;   // (P of an agent without a row: not used)
        for (uint32_t t0 = 0; t0 < total; t0 += OP_TILE) {
            uint32_t sj[OP_U];
            float wk[OP_U];
            T xj[OP_U];
#pragma unroll
            for (int u = 0; u < OP_U; u++) {
                const uint32_t q = t0 + (uint32_t)u * 256u + tid;
                const uint32_t k = b0 + (q < total ? q : 0u);   // (past the end: a valid dummy)
                sj[u] = op_edge<uint32_t, STREAM>(src + k);
                wk[u] = op_edge<float, STREAM>(w + k);
            }
#pragma unroll
            for (int u = 0; u < OP_U; u++) xj[u] = x[sj[u] - 1];
#pragma unroll
            for (int u = 0; u < OP_U; u++) {
                sm.x[u * 256 + tid] = xj[u];
                sm.w[u * 256 + tid] = wk[u];
            }
            __syncthreads();
            const uint32_t lo = P > t0 ? P : t0, hi = P + d < t0 + OP_TILE ? P + d : t0 + OP_TILE;
            if (d) op_sum_slots(sm, lo, hi, t0, xi, eps, num, den);
            if (t0 + OP_TILE < total) __syncthreads();
        }
    } else {
        const uint32_t ld = light ? d : 0u;
        uint32_t total;
        const uint32_t P = op_light_scan(ld, sm.wsum, total);
        sm.b[tid] = b;
        sm.p[tid] = P;
        for (uint32_t t0 = 0; t0 < total; t0 += OP_TILE) {
            const uint32_t lo = P > t0 ? P : t0;
            const uint32_t hi = (P + ld) < (t0 + OP_TILE) ? (P + ld) : (t0 + OP_TILE);
            for (uint32_t p = lo; p < hi; p++) sm.own[p - t0] = (uint8_t)tid;
            __syncthreads();
            const uint32_t cnt = (total - t0) < (uint32_t)OP_TILE ? (total - t0) : (uint32_t)OP_TILE;
            uint32_t kk[OP_U], sj[OP_U];
            float wk[OP_U];
            T xj[OP_U];
#pragma unroll
            for (int u = 0; u < OP_U; u++) {
                const uint32_t q = (uint32_t)u * 256u + tid;
                const uint32_t a = q < cnt ? sm.own[q] : 0u;
                kk[u] = q < cnt ? sm.b[a] + (t0 + q - sm.p[a]) : 0xFFFFFFFFu;
            }
#pragma unroll
            for (int u = 0; u < OP_U; u++) {
                sj[u] = kk[u] != 0xFFFFFFFFu ? src[kk[u]] : 1u;
                wk[u] = kk[u] != 0xFFFFFFFFu ? w[kk[u]] : 0.0f;
            }
#pragma unroll
            for (int u = 0; u < OP_U; u++) xj[u] = kk[u] != 0xFFFFFFFFu ? x[sj[u] - 1] : (T)0;
#pragma unroll
            for (int u = 0; u < OP_U; u++) {
                sm.x[u * 256 + tid] = xj[u];
                sm.w[u * 256 + tid] = wk[u];
            }
            __syncthreads();
            if (lo < hi) op_sum_slots(sm, lo, hi, t0, xi, eps, num, den);
            __syncthreads();
        }
    }
    if (light) xo[i] = den > (T)0 ? num / den : xi;
}

template <class T>
__device__ __forceinline__ void opinion_heavy(const uint32_t* __restrict__ off,
                                              const uint32_t* __restrict__ src,
                                              const T* __restrict__ x, const float* __restrict__ w,
                                              T* __restrict__ xo, uint64_t r, uint64_t rowbase, T eps) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t i = r - rowbase;
    const T xi = x[i];
    T num = (T)0, den = (T)0;
    // lane l adds k = l, l+64, ... in order; four strides in flight per lane
    auto four = [&](uint32_t k) {
        const uint32_t s0 = src[k], s1 = src[k + 64], s2 = src[k + 128], s3 = src[k + 192];
        const float w0 = w[k], w1 = w[k + 64], w2 = w[k + 128], w3 = w[k + 192];
        const T x0 = x[s0 - 1], x1 = x[s1 - 1], x2 = x[s2 - 1], x3 = x[s3 - 1];
        op_accum(x0, w0, xi, eps, num, den);
        op_accum(x1, w1, xi, eps, num, den);
        op_accum(x2, w2, xi, eps, num, den);
        op_accum(x3, w3, xi, eps, num, den);
    };
    vh_lane_edges(off[r], off[r + 1], lane, four,
                  [&](uint32_t k) { op_accum(x[src[k] - 1], w[k], xi, eps, num, den); });
    num = xor_butterfly(num);
    den = xor_butterfly(den);
    if (lane == 0) xo[i] = den > (T)0 ? num / den : xi;
}

// blocks [0, nh) run one wave per heavy agent (the longest work starts
// first), the others are light blocks
template <class T, bool STREAM>
__global__ __launch_bounds__(256) void k_opinion(const uint32_t* __restrict__ off,
                                                 const uint32_t* __restrict__ src,
                                                 const T* __restrict__ x, const float* __restrict__ w,
                                                 T* __restrict__ xo, uint64_t n, uint64_t nrows,
                                                 uint64_t rowbase, T eps, const uint32_t* __restrict__ heavy,
                                                 uint64_t nheavy, uint32_t nh) {
    if (blockIdx.x >= nh) {
        opinion_block<T, STREAM>(off, src, x, w, xo, n, nrows, rowbase, eps, blockIdx.x - nh);
    } else {
        const uint64_t wv = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
        if (wv < nheavy) opinion_heavy<T>(off, src, x, w, xo, heavy[wv], rowbase, eps);
    }
}

// Many simulations' one-pass opinion steps in one launch: block b belongs to
// the member with the largest blk0 <= b (its heavy-wave blocks first, then
// its light blocks), every member with its own CSR, states and eps.
// Blocks go to the 8 XCDs in turn, so XCD q takes the logical blocks
// [q per, (q + 1) per): its L2 then holds the states of one or two members at
// a time instead of a share of every member's (24 members of 10^4 to 10^6
// Float64 agents: 494 -> 462 us a step, with the kernel as it was then).
template <class T, bool STREAM>
__global__ __launch_bounds__(256) void k_opinion_multi(const OpMember* __restrict__ mem, uint32_t nm,
                                                       uint32_t nblocks) {
    const uint32_t per = gridDim.x / 8u, blk = (blockIdx.x % 8u) * per + blockIdx.x / 8u;
    if (blk >= nblocks) return;
    uint32_t lo = 0, hi = nm;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (mem[mid].blk0 <= blk) lo = mid;
        else hi = mid;
    }
    const OpMember& m = mem[lo];
    const uint32_t local = blk - m.blk0;
    if (local >= m.nh) {
        opinion_block<T, STREAM>(m.off, m.src, (const T*)m.x, m.w, (T*)m.xo, m.n, m.nrows, m.rowbase, (T)m.eps,
                         local - m.nh);
    } else {
        const uint64_t wv = ((uint64_t)local * blockDim.x + threadIdx.x) >> 6;
        if (wv < m.nheavy) opinion_heavy<T>(m.off, m.src, (const T*)m.x, m.w, (T*)m.xo, m.heavy[wv], m.rowbase,
                                           (T)m.eps);
    }
}

// ----------------------------------------------------------------- gather plan
// For a large state vector the neighbour states of a static edge store are
// gathered in two passes through a plan built once per edge store.
//
// Windows: the sources are cut into windows of `wsz` consecutive agents, at
// most 160 KB of states (one CU's LDS) and at most WIN_RUNS windows. Blocks:
// the agents are cut into blocks of consecutive agents with fewer than TB
// staged in-edges, TB being the slots a block stages in LDS; an agent's
// in-edges are staged when its in-degree is at most WIN_HMAX (rows above go
// through chunk lists). An agent costs its staged in-degree + 1; block b
// holds the agents whose exclusive cost prefix lies in [b S, (b + 1) S),
// S = TB - WIN_HMAX - 1. The plan orders the CSR slots by (window, block),
// the chunk-list rows' slots after the staged ones of their window, keeping
// CSR order within: the staged in-edges of a block from one window are one
// run of the plan.
//
// Pass 1 (k_win_gather) streams the plan: each block of the launch takes a
// contiguous share, stages each window it meets in LDS and writes
// y[j] = x[src(j)] for its share, so the random reads are LDS reads and HBM
// sees sequential streams (the plan's local source indices, y, the windows).
//
// Pass 2 (k_win_sum) takes the agent blocks from a queue. A block's staged
// entries are listed by (window, CSR slot): entry e holds its slot in LDS (bit
// 15 set on the first entry of a run) and its weight, and its value is
// y[prun[r] + e - pfirst[r]] for its run r, counted from the run starts
// before its 64-entry chunk (cbase) and a ballot of the start bits. Values and
// weights are staged in LDS by slot; then a lane adds the slots of each agent
// of in-degree <= 64 in order, and a wave those of each agent of in-degree
// 65..WIN_HMAX (lane l the l-th, l + 64th, ..., then the xor butterfly), with
// the agents ordered by in-degree (k_win_order). Agents above WIN_HMAX go
// first, one wave each, through their chunk lists. Most of the next block's
// values, and its list, runs and agents, load while a block is summed. The
// values are exactly x[src[k]] and the sums keep the canonical order, so the
// results are the one-pass kernel's.
template <class T>
struct WinCfg {
    static constexpr uint32_t WSZ = 163840 / sizeof(T);             // states per window at most
    static constexpr uint32_t TB = sizeof(T) == 8 ? 12288 : 16384;  // staged slots per block at most
    static constexpr uint32_t QU = TB / 1024;                       // list entries per thread
    static constexpr uint32_t QA = sizeof(T) == 8 ? 6 : 10;         // of them, loaded during the previous sums
    static constexpr uint32_t CPB = TB / 64;                        // 64-entry chunks per block
    static constexpr uint32_t CHUNK = sizeof(T) == 8 ? 256 : 384;   // heavy-row slots staged per wave
};
constexpr uint32_t WIN_RUNS = 1024;   // windows at most (runs of a block)
constexpr uint32_t WIN_HMAX = 512;    // in-degrees staged within blocks (larger: chunk lists)
constexpr uint32_t WIN_SLOT = 0x3FFFu, WIN_START = 0x8000u;

// A heavy agent (one wave) from its chunk lists: the in-edges of heavy agent
// h are numbered from hbase[h] in CSR order, in chunks of CHUNK slots, each
// chunk listed in plan order (hty: plan position, hslot: slot in the chunk).
// The wave copies a chunk's values into its LDS region `buf` by slot, then
// lane l adds slots l, l + 64, ... in order: the canonical lane-strided
// partials, then the xor butterfly.
template <class T>
__device__ __forceinline__ void opinion_heavy_plan(const T* __restrict__ x, const T* __restrict__ y,
                                                   const float* __restrict__ w, T* __restrict__ xo,
                                                   const uint4 hi, T eps, const uint32_t* __restrict__ hty,
                                                   const uint16_t* __restrict__ hslot, T* buf) {
    constexpr uint32_t CH = WinCfg<T>::CHUNK;
    constexpr int HU = CH / 64;
    const uint32_t lane = threadIdx.x & 63;
    // hi: row, CSR start, degree, first chunk-list entry
    const uint64_t r = hi.x;
    const uint32_t b = hi.y, d = hi.z, hb = hi.w;
    const T xi = x[r];
    T num = (T)0, den = (T)0;
    for (uint32_t c0 = 0; c0 < d; c0 = vh_row_next(c0, d, CH)) {
        const uint32_t cnt = d - c0 < CH ? d - c0 : CH;
        float wq[HU];
        uint32_t jj[HU], sl[HU];
        T v[HU];
#pragma unroll
        for (int u = 0; u < HU; u++) {
            const uint32_t q = lane + 64u * (uint32_t)u;
            wq[u] = 0.0f;
            jj[u] = 0u;
            sl[u] = 0xFFFFFFFFu;
            if (q < cnt) {
                wq[u] = w[b + c0 + q];
                jj[u] = hty[hb + c0 + q];
                sl[u] = hslot[hb + c0 + q];
            }
        }
#pragma unroll
        for (int u = 0; u < HU; u++) v[u] = sl[u] != 0xFFFFFFFFu ? y[jj[u]] : (T)0;
#pragma unroll
        for (int u = 0; u < HU; u++)
            if (sl[u] != 0xFFFFFFFFu) buf[sl[u]] = v[u];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int u = 0; u < HU; u++) {
            const uint32_t q = lane + 64u * (uint32_t)u;
            if (q < cnt) op_accum(buf[q], wq[u], xi, eps, num, den);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    num = xor_butterfly(num);
    den = xor_butterfly(den);
    if (lane == 0) xo[r] = den > (T)0 ? num / den : xi;
}


// Pass 1: block l of the grid (one per CU) takes plan entries
// [ne l / G, ne (l + 1) / G). For each window its share meets: the window's
// states go to LDS (16-byte loads), then wave v, step u writes the 256
// entries from c = g0 + 256 (v + 16 u) in two halves, lane l entries
// c + 2l, c + 2l + 1 and c + 128 + 2l, c + 129 + 2l (one 4-byte load of their
// two source indices, one 2-state store: each store instruction writes one
// contiguous range; measured 236 us against 308 us with 4 entries per lane
// at 10^8 entries), for U steps u at a time: the loads of all U issued
// before the stores (10^7 agents, 10^8 entries, ms per opinion step, FP64 /
// FP32: U = 2 0.689-0.692 / 0.515-0.520, U = 4 0.670-0.674 / 0.472-0.477,
// U = 6 0.660-0.672 / 0.455-0.461, U = 8 0.664-0.673 / 0.456-0.460).
typedef uint32_t pu32x4 __attribute__((ext_vector_type(4)));

template <class T>
struct Pair;
template <>
struct Pair<double> {
    typedef double type __attribute__((ext_vector_type(2)));
};
template <>
struct Pair<float> {
    typedef float type __attribute__((ext_vector_type(2)));
};

template <class T>
__global__ __launch_bounds__(1024) void k_win_gather(const uint16_t* __restrict__ psl, const T* __restrict__ x,
                                                     T* __restrict__ y, const uint32_t* __restrict__ wstart,
                                                     uint32_t W, uint32_t wsz, uint64_t nsrc, uint64_t ne) {
    typedef typename Pair<T>::type T2;
    constexpr uint32_t PER16 = 16 / sizeof(T);
    constexpr int U = 6;
    __shared__ __align__(16) T win[WinCfg<T>::WSZ];
    const uint32_t G = gridDim.x, l = blockIdx.x;
    const uint64_t j0 = ne * l / G, j1 = ne * (l + 1) / G;
    if (j0 >= j1) return;   // whole block
    uint32_t lo = 0, hi = W;   // the window of j0: wstart[lo] <= j0 < wstart[lo + 1]
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (wstart[mid] <= j0) lo = mid;
        else hi = mid;
    }
    const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    uint32_t w = lo;
    uint64_t j = j0;
    while (j < j1) {
        const uint64_t we = wstart[w + 1];
        if (we <= j) {   // empty window
            w++;
            continue;
        }
        const uint64_t s0 = (uint64_t)w * wsz;
        const uint32_t wn = (uint32_t)((nsrc - s0) < wsz ? nsrc - s0 : wsz);
        for (uint32_t q = threadIdx.x * PER16; q < wn; q += 1024 * PER16) {
            if (q + PER16 <= wn) {
                *(pu32x4*)(win + q) = __builtin_nontemporal_load((const pu32x4*)(x + s0 + q));
            } else {
                for (uint32_t t = q; t < wn; t++) win[t] = x[s0 + t];
            }
        }
        __syncthreads();
        const uint64_t je = we < j1 ? we : j1;
        for (uint64_t g0 = j & ~3ull; g0 < je; g0 += 4096ull * U) {
            uint32_t p0[U], p1[U];
            bool f0[U], f1[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const uint64_t ga = g0 + 256ull * (wv + 16 * u) + 2 * lane, gb = ga + 128;
                f0[u] = ga >= j && ga + 2 <= je;
                f1[u] = gb >= j && gb + 2 <= je;
                p0[u] = f0[u] ? __builtin_nontemporal_load((const uint32_t*)(psl + ga)) : 0u;
                p1[u] = f1[u] ? __builtin_nontemporal_load((const uint32_t*)(psl + gb)) : 0u;
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const uint64_t ga = g0 + 256ull * (wv + 16 * u) + 2 * lane, gb = ga + 128;
                if (f0[u]) {
                    const T2 v = {win[p0[u] & 0xFFFFu], win[p0[u] >> 16]};
                    *(T2*)(y + ga) = v;
                } else {
                    for (uint64_t t = ga; t < ga + 2; t++)
                        if (t >= j && t < je) y[t] = win[psl[t]];
                }
                if (f1[u]) {
                    const T2 v = {win[p1[u] & 0xFFFFu], win[p1[u] >> 16]};
                    *(T2*)(y + gb) = v;
                } else {
                    for (uint64_t t = gb; t < gb + 2; t++)
                        if (t >= j && t < je) y[t] = win[psl[t]];
                }
            }
        }
        __syncthreads();
        j = je;
        w++;
    }
}

template <class T>
struct WinLDS {
    T val[WinCfg<T>::TB];          // values by slot (heavy waves: CHUNK each)
    float wgt[WinCfg<T>::TB];      // weights by slot
    uint32_t rp[2][WIN_RUNS];      // runs of this block and the next: plan position - list index (mod 2^32)
    uint32_t nextq[2];             // queue items taken ahead
    uint32_t nmed[4];              // agents of in-degree 65..WIN_HMAX in each wave's first 64 (< TB / 64 in all)
    uint32_t mpk[WinCfg<T>::TB / 64], magent[WinCfg<T>::TB / 64];   // slot | in-degree << 16
    T mx[WinCfg<T>::TB / 64];
};

// A block's agents are ordered by in-degree: those of 65..WIN_HMAX ("medium"),
// then 64 down to 0 ("light"), then the ones with chunk lists. An entry of the
// order is the agent's index in the block | in-degree << 14 (ORD_HUGE: chunk
// lists), and 64 entries are a group, summed by a wave. The slots of a group
// follow those of the groups before it (gbase): its medium agents' one after
// the other, then the light ones' by position: position q of all light agents
// that have one, in order. So the lanes of a wave add the same number of
// slots, give or take one, and read neighbouring ones. With a lane per agent
// in agent order and its slots in a row, a wave took as many rounds as its
// largest in-degree (10^7 agents, BA m = 5, about 40 for a mean of 9) with
// bank conflicts, and the slots' starts were a block scan: 434 us a launch, so
// 403; Float32, 5 10^6 agents of mean in-degree 10: 126, so 109. (What is left
// is loads: without the sums 397 us, with the values read in list order 371,
// with all values from the caches 307.)
constexpr uint32_t ORD_LOCAL = 0x3FFFu, ORD_HUGE = 1023u;

// The agents of a block at tid and 1024 + tid of its order: the entries,
// loaded with the block's list, the waves' first slots, and the states, loaded
// once the entries are there
template <class T>
struct WinAgents {
    uint32_t e0, e1, g0, g1;
    T x0, x1;
};
__device__ __forceinline__ uint32_t win_group(uint32_t a0, uint32_t b) { return a0 / 64u + b; }   // block b's first

template <class T>
__device__ __forceinline__ void win_entries(WinAgents<T>& g, const uint32_t* __restrict__ aord,
                                            const uint32_t* __restrict__ gbase, uint32_t b, uint32_t a0,
                                            uint32_t a1, uint32_t tid, uint32_t wv) {
    const uint32_t i0 = a0 + tid, i1 = i0 + 1024, gi = win_group(a0, b) + wv, ng = (a1 - a0 + 63) / 64;
    g.e0 = aord[i0 < a1 ? i0 : a0];
    g.e1 = aord[i1 < a1 ? i1 : a0];
    g.g0 = gbase[wv < ng ? gi : 0u];
    g.g1 = gbase[wv + 16 < ng ? gi + 16 : 0u];
}
template <class T>
__device__ __forceinline__ void win_states(WinAgents<T>& g, const T* __restrict__ x, uint32_t a0) {
    g.x0 = x[a0 + (g.e0 & ORD_LOCAL)];
    g.x1 = x[a0 + (g.e1 & ORD_LOCAL)];
}

// The light agents of a group: lane l has entry e, state xi (act: there is
// one), the group's slots start at gb
template <class T>
__device__ __forceinline__ void win_sum_group(WinLDS<T>& sm, T* __restrict__ xo, T eps, uint32_t a0, uint32_t e,
                                              bool act, T xi, uint32_t gb) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t c = act ? e >> 14 : ORD_HUGE;
    const bool light = c <= 64u;
    const uint64_t med = __ballot(act && c > 64u && c <= WIN_HMAX);
    uint32_t base = gb, nm = 0;
    if (med) {   // uniform; the first lanes
        nm = (uint32_t)__popcll(med);
        base += (uint32_t)__builtin_amdgcn_readlane((int)wave_incl_scan((med >> lane) & 1ull ? c : 0u), 63);
    }
    const uint32_t d = light ? c : 0u;
    const uint32_t dmax = nm < 64u ? (uint32_t)__builtin_amdgcn_readlane((int)d, (int)nm) : 0u;
    T num = (T)0, den = (T)0;
    uint32_t p = base + lane - nm;   // (lanes without a slot q read another value, unused; past the slots: the LDS
    for (uint32_t q = 0; q < dmax; q += 4) {   // behind them)
        T y[4];
        float w[4];
        uint64_t m[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            m[u] = __ballot(d > q + u);
            y[u] = sm.val[p];
            w[u] = sm.wgt[p];
            p += (uint32_t)__popcll(m[u]);
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const bool acc = d > q + u && fabs(y[u] - xi) <= eps;   // (a rejected one adds +0.0, as in op_accum)
            num = num + (acc ? (T)w[u] * y[u] : (T)0);
            den = den + (acc ? (T)w[u] : (T)0);
        }
    }
    if (light) xo[a0 + (e & ORD_LOCAL)] = den > (T)0 ? num / den : xi;
}

// The agents of block b, in rounds of 1024 of its order; the staged values are
// published by the first barrier. Rounds 0 and 1 use the entries and states
// loaded early (g); later rounds load theirs when LD (without LD the block has
// at most two rounds, and no global load is issued). The medium agents, which
// are among the first TB / 64, are listed before the barrier and summed by a
// wave each (lane-strided partials, xor butterfly). after_barrier() runs right
// after the barrier.
template <class T, bool LD, class F>
__device__ __forceinline__ void win_sum_agents(WinLDS<T>& sm, const uint32_t* __restrict__ aord,
                                               const uint32_t* __restrict__ gbase, const T* __restrict__ x,
                                               T* __restrict__ xo, T eps, uint32_t b, uint32_t a0, uint32_t a1,
                                               const WinAgents<T>& g, F after_barrier) {
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wv = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    static_assert(WinCfg<T>::TB / 64 <= 256, "the medium agents are the first four waves'");
    if (wv < 4) {
        const uint32_t c = a0 + tid < a1 ? g.e0 >> 14 : 0u;
        const bool med = c > 64u && c <= WIN_HMAX;
        const uint64_t m = __ballot(med);
        if (lane == 0) sm.nmed[wv] = (uint32_t)__popcll(m);
        if (m) {   // uniform
            const uint32_t md = med ? c : 0u, P = g.g0 + wave_incl_scan(md) - md;
            if (med) {
                sm.mpk[tid] = P | c << 16;
                sm.magent[tid] = a0 + (g.e0 & ORD_LOCAL);
                sm.mx[tid] = g.x0;
            }
        }
    }
    __syncthreads();
    after_barrier();
    win_sum_group<T>(sm, xo, eps, a0, g.e0, a0 + tid < a1, g.x0, g.g0);
    if (a1 - a0 > 1024u) win_sum_group<T>(sm, xo, eps, a0, g.e1, a0 + 1024 + tid < a1, g.x1, g.g1);
    if (LD)
        for (uint32_t r = 2; r * 1024u < a1 - a0; r++) {
            const uint32_t i = a0 + r * 1024 + tid, gi = r * 16 + wv;
            const bool act = i < a1;
            const uint32_t e = aord[act ? i : a0];
            const uint32_t gb = gi < (a1 - a0 + 63) / 64 ? gbase[win_group(a0, b) + gi] : 0u;
            win_sum_group<T>(sm, xo, eps, a0, e, act, x[a0 + (e & ORD_LOCAL)], gb);
        }
    const uint32_t nmed = sm.nmed[0] + sm.nmed[1] + sm.nmed[2] + sm.nmed[3];
    for (uint32_t m = 15 - wv; m < nmed; m += 16) {   // (the last waves have the smallest light in-degrees)
        const uint32_t P = sm.mpk[m] & 0xFFFFu, d = sm.mpk[m] >> 16;
        const T xi = sm.mx[m];
        T num = (T)0, den = (T)0;
        for (uint32_t q = lane; q < d; q += 64) op_accum(sm.val[P + q], sm.wgt[P + q], xi, eps, num, den);
        num = xor_butterfly(num);
        den = xor_butterfly(den);
        if (lane == 0) xo[sm.magent[m]] = den > (T)0 ? num / den : xi;
    }
}

// Pass 2: one block of 1024 per CU. The waves first take the heavy agents
// (wave g of the grid agents g, g + 16 G, ...), then the blocks take light
// blocks from a queue (queue[0]: next light block, queue[1]: blocks done;
// the last block to finish sets both to 0 for the next launch). Each thread
// stages QU list entries of a block; the values of its first QA entries load
// while the previous block is summed (in registers: the block's LDS is in
// use), the other QU - QA after the sums. Measured slower or no faster at 10^7
// Float64 agents (403 us): QA = 4, 8 or 10 of 12 (405, 404, 407); two blocks
// of 512 threads and 5120 slots per CU (442: shorter runs); the entries in
// pairs per lane with the lists loaded two blocks ahead (414); the tables' words
// by a vector load an iteration ahead in place of scalar loads (403); a queue
// per XCD that hands out 8 or 32 blocks in a row, which takes the bytes read
// from 2.06 to 1.68 and 1.62 GB (405, 411).
template <class T>
__global__ __launch_bounds__(1024) void k_win_sum(const uint32_t* __restrict__ aord,
                                                  const uint32_t* __restrict__ gbase, const T* __restrict__ x,
                                                  const T* __restrict__ y, const float* __restrict__ w,
                                                  T* __restrict__ xo, T eps,
                                                  const uint4* __restrict__ hinfo, uint64_t nheavy,
                                                  const uint32_t* __restrict__ hty,
                                                  const uint16_t* __restrict__ hslot,
                                                  const uint32_t* __restrict__ ablk,
                                                  const uint32_t* __restrict__ lbase,
                                                  const uint16_t* __restrict__ tpk, const float* __restrict__ twt,
                                                  const uint32_t* __restrict__ rbase,
                                                  const uint32_t* __restrict__ prun,
                                                  const uint16_t* __restrict__ pfirst,
                                                  const uint16_t* __restrict__ cbase, uint32_t nb,
                                                  uint32_t* __restrict__ queue) {
    constexpr uint32_t QU = WinCfg<T>::QU, QA = WinCfg<T>::QA, QB = QU - QA;
    static_assert(QA % 2 == 0 && QB % 2 == 0 && QB > 0, "chunk run counts are read in 16-bit pairs");
    __shared__ __align__(16) unsigned char smraw[sizeof(WinLDS<T>)];
    WinLDS<T>& sm = *reinterpret_cast<WinLDS<T>*>(smraw);
    const uint32_t tid = threadIdx.x;
    const int lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint64_t lemask = lane == 63 ? ~0ull : ((1ull << (lane + 1)) - 1ull);
    for (uint64_t h = (uint64_t)blockIdx.x * 16 + (uint32_t)wv; h < nheavy; h += (uint64_t)gridDim.x * 16)
        opinion_heavy_plan<T>(x, y, w, xo, hinfo[h], eps, hty, hslot, sm.val + wv * WinCfg<T>::CHUNK);
    // every load is branch-free (lanes past a list read a valid dummy, an
    // inactive list reads as empty): a load under a branch makes the compiler
    // wait for all loads in flight where the branch joins; and loads complete
    // in issue order, so the sums issue no global load (blocks of at most two
    // rounds of agents, the others take a path that does)
    constexpr uint32_t NONE = 0xFFFFFFFFu;
    uint32_t ltid = tid;
    auto load_list = [&](uint32_t b, bool act, uint32_t* pk) __attribute__((always_inline)) {
        const uint32_t lb = lbase[b], L = act ? lbase[b + 1] - lb : 0u;
#pragma unroll
        for (uint32_t u = 0; u < QU; u++) {
            const uint32_t e = ltid + 1024 * u;
            pk[u] = tpk[lb + (e < L ? e : 0u)];   // (past the list: masked where used)
        }
    };
    auto load_runs = [&](uint32_t b) __attribute__((always_inline)) {
        const uint32_t rb = rbase[b], R = rbase[b + 1] - rb;
        const uint32_t r = rb + (ltid < R ? ltid : 0u);   // (R == 0: the slack after the runs)
        return make_uint2(prun[r], pfirst[r]);
    };
    // values and weights of entries u in [U0, U0 + QH) of block b (its runs in
    // sm.rp[c]; the wave's chunk run counts by scalar loads)
    auto load_vals = [&](auto NN, uint32_t b, bool act, uint32_t c, uint32_t U0, const uint32_t* pk, T* v,
                         float* wt) __attribute__((always_inline)) {
        constexpr uint32_t QH = decltype(NN)::value;
        const uint32_t lb = lbase[b], L = act ? lbase[b + 1] - lb : 0u;
        const uint32_t* cw = (const uint32_t*)(cbase + ((uint64_t)b * 256 + (uint32_t)wv * 16));
        uint32_t cwv[QH / 2];
#pragma unroll
        for (uint32_t q = 0; q < QH / 2; q++) cwv[q] = cw[U0 / 2 + q];
        // the run table reads of all QH entries first (unconditional: run 0
        // for lanes past the list), then the global loads
        uint32_t rpv[QH];
#pragma unroll
        for (uint32_t k = 0; k < QH; k++) {
            const uint32_t u = U0 + k;
            const uint32_t e = ltid + 1024 * u;
            const bool ok = e < L;
            const uint64_t m = __ballot(ok && (pk[u] & WIN_START));
            const uint32_t cb = (cwv[k >> 1] >> ((k & 1) * 16)) & 0xFFFFu;
            const uint32_t run = ok ? cb + __popcll(m & lemask) - 1u : 0u;
            rpv[k] = sm.rp[c][run];
        }
#pragma unroll
        for (uint32_t k = 0; k < QH; k++) {
            const uint32_t e = ltid + 1024 * (U0 + k);
            const bool ok = e < L;
            const uint32_t pos = ok ? rpv[k] + e : 0u;
            v[k] = y[pos];
            wt[k] = twt[lb + (ok ? e : 0u)];
        }
    };
    auto scatter = [&](auto NN, uint32_t L, uint32_t U0, const uint32_t* pk, const T* v, const float* wt)
                       __attribute__((always_inline)) {
        constexpr uint32_t QH = decltype(NN)::value;
#pragma unroll
        for (uint32_t k = 0; k < QH; k++)
            if (ltid + 1024 * (U0 + k) < L) {
                sm.val[pk[U0 + k] & WIN_SLOT] = v[k];
                sm.wgt[pk[U0 + k] & WIN_SLOT] = wt[k];
            }
    };
    if (tid == 0) {
        sm.nextq[0] = atomicAdd(queue, 1u);
        sm.nextq[1] = atomicAdd(queue, 1u);
    }
    __syncthreads();   // (also ends the heavy agents' use of sm.val)
    const uint32_t q0 = __builtin_amdgcn_readfirstlane(sm.nextq[0]), q1 = __builtin_amdgcn_readfirstlane(sm.nextq[1]);
    uint32_t b = q0 < nb ? q0 : NONE, bn = q1 < nb ? q1 : NONE;
    __syncthreads();
    if (b != NONE) {
        uint32_t pk[QU];
        T vA[QA];
        float wA[QA];
        WinAgents<T> ag;
        int cur = 0, par = 0;
        {
            const uint2 ra = load_runs(b);
            load_list(b, true, pk);
            win_entries<T>(ag, aord, gbase, b, ablk[b], ablk[b + 1], ltid, (uint32_t)wv);
            win_states<T>(ag, x, ablk[b]);
            sm.rp[0][tid] = ra.x - ra.y;
            __syncthreads();
            load_vals(std::integral_constant<uint32_t, QA>(), b, true, 0, 0, pk, vA, wA);
        }
        // per block: the rest of its values; the next block's list, runs and
        // agents; all its values staged; the next queue item; the sums, whose
        // first barrier publishes the staged values and the next runs, after
        // which the next block's states and first QA values are issued (in
        // flight during the sums); a barrier
        for (;;) {
            asm volatile("" : "+v"(ltid));
            const bool hasn = bn != NONE;
            const uint32_t bnc = hasn ? bn : b;
            const uint32_t L = lbase[b + 1] - lbase[b];
            T vB[QB];
            float wB[QB];
            load_vals(std::integral_constant<uint32_t, QB>(), b, true, cur, QA, pk, vB, wB);
            uint32_t pkn[QU];
            load_list(bnc, hasn, pkn);
            const uint2 ra = load_runs(bnc);
            WinAgents<T> agn;
            win_entries<T>(agn, aord, gbase, bnc, ablk[bnc], ablk[bnc + 1], ltid, (uint32_t)wv);
            scatter(std::integral_constant<uint32_t, QA>(), L, 0, pk, vA, wA);
            scatter(std::integral_constant<uint32_t, QB>(), L, QA, pk, vB, wB);
            sm.rp[cur ^ 1][tid] = ra.x - ra.y;
            if (tid == 0) sm.nextq[par] = atomicAdd(queue, 1u);
            auto after_barrier = [&]() __attribute__((always_inline)) {
                win_states<T>(agn, x, ablk[bnc]);
                load_vals(std::integral_constant<uint32_t, QA>(), bnc, hasn, cur ^ 1, 0, pkn, vA, wA);
            };
            {
                // a block of at most two rounds sums without a global load,
                // so the next block's values stay in flight
                const uint32_t a0 = ablk[b], a1 = ablk[b + 1];
                if (a1 - a0 <= 2048u)
                    win_sum_agents<T, false>(sm, aord, gbase, x, xo, eps, b, a0, a1, ag, after_barrier);
                else {
                    win_sum_agents<T, true>(sm, aord, gbase, x, xo, eps, b, a0, a1, ag, after_barrier);
                    __builtin_amdgcn_s_waitcnt(0);   // (its loads have drained the counter anyway)
                }
            }
            __syncthreads();
            if (!hasn) break;
            const uint32_t it = __builtin_amdgcn_readfirstlane(sm.nextq[par]);
            b = bn;
            bn = it < nb ? it : NONE;
#pragma unroll
            for (uint32_t u = 0; u < QU; u++) pk[u] = pkn[u];
            ag = agn;
            cur ^= 1;
            par ^= 1;
        }
    }
    if (tid == 0 && atomicAdd(queue + 1, 1u) == gridDim.x - 1) {
        queue[0] = 0;
        queue[1] = 0;
    }
}

// consistency of a built plan, one thread per block: its agents, order, list
// and runs in range, every run's first entry and only those marked, each run
// inside y, each chunk's run count; any failure sets *bad (the plan is then
// refused: pass 2 trusts these bounds)
__global__ void k_win_check(const uint32_t* __restrict__ ablk, const uint32_t* __restrict__ lbase,
                            const uint32_t* __restrict__ rbase, const uint32_t* __restrict__ prun,
                            const uint16_t* __restrict__ pfirst, const uint16_t* __restrict__ tpk,
                            const uint16_t* __restrict__ cbase, const uint32_t* __restrict__ aord,
                            const uint32_t* __restrict__ gbase, uint32_t nb, uint64_t n, uint64_t nl,
                            uint64_t nruns, uint64_t ne, uint32_t TB, uint32_t cpb, uint32_t* __restrict__ bad) {
    const uint64_t b = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nb) return;
    const uint32_t a0 = ablk[b], a1 = ablk[b + 1], lb = lbase[b], lb1 = lbase[b + 1];
    const uint32_t rb = rbase[b], rb1 = rbase[b + 1];
    bool ok = a0 < a1 && a1 <= n && lb <= lb1 && lb1 <= nl && lb1 - lb < TB && rb <= rb1 && rb1 <= nruns &&
              rb1 - rb <= WIN_RUNS && (lb1 > lb) == (rb1 > rb);
    if (ok) {
        const uint32_t L = lb1 - lb;
        uint32_t prev = 0;
        for (uint32_t r = rb; r < rb1 && ok; r++) {
            const uint32_t f = pfirst[r], f1 = r + 1 < rb1 ? pfirst[r + 1] : L;
            ok = (r == rb ? f == 0 : f > prev) && f1 > f && f1 <= L && (uint64_t)prun[r] + (f1 - f) <= ne;
            for (uint32_t e = f; e < f1 && ok; e++) {
                const uint32_t pk = tpk[lb + e];
                ok = ((pk & WIN_START) != 0) == (e == f) && (pk & WIN_SLOT) < L;
            }
            prev = f;
        }
        uint32_t r = rb;
        for (uint32_t c = 0; c < cpb && 64u * c < L && ok; c++) {
            while (r < rb1 && pfirst[r] < 64u * c) r++;
            ok = cbase[b * 256 + (c % 16) * 16 + c / 16] == r - rb;
        }
    }
    uint32_t slots = 0;   // (agents of the order in the block, slots of its groups in the list)
    for (uint32_t p = 0; p < a1 - a0 && ok; p++) {
        const uint32_t e = aord[a0 + p], d = e >> 14;
        ok = (e & ORD_LOCAL) < a1 - a0 && (d <= WIN_HMAX || d == ORD_HUGE) &&
             (p % 64 || gbase[win_group(a0, (uint32_t)b) + p / 64] == slots);
        slots += d != ORD_HUGE ? d : 0u;
    }
    if (!ok || slots != lb1 - lb) atomicOr(bad, 1u);
}

// plan build: staged in-degree + 1 of each agent (rows past nrows: 1)
__global__ void k_win_cost(const uint32_t* __restrict__ off, uint64_t n, uint64_t nrows,
                           uint32_t* __restrict__ cost) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t d = i < nrows ? off[i + 1] - off[i] : 0u;
    cost[i] = (d <= WIN_HMAX ? d : 0u) + 1u;
}

// first agent and first list entry of each block (C: exclusive cost prefix,
// n + 1 entries; the thread of agent n writes the ends)
__global__ void k_win_blocks(const uint32_t* __restrict__ C, uint64_t n, uint32_t S, uint32_t nb,
                             uint32_t* __restrict__ ablk, uint32_t* __restrict__ lbase) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i > n) return;
    if (i == n) {
        ablk[nb] = (uint32_t)n;
        lbase[nb] = C[n] - (uint32_t)n;
        return;
    }
    const uint32_t b = C[i] / S;
    if (i == 0 || C[i - 1] / S != b) {
        ablk[b] = (uint32_t)i;
        lbase[b] = C[i] - (uint32_t)i;
    }
}

// order of each block's agents (entries by position), first slot of each of
// its groups, and the slot of each staged in-edge (sl, numbered by the staged
// prefix C[r] - r + position): a block of the launch per block
__global__ __launch_bounds__(1024) void k_win_order(const uint32_t* __restrict__ off, uint64_t nrows,
                                                    const uint32_t* __restrict__ C,
                                                    const uint32_t* __restrict__ ablk, uint32_t* __restrict__ aord,
                                                    uint32_t* __restrict__ gbase, uint16_t* __restrict__ sl) {
    __shared__ uint32_t s_first[67], s_gb[256];   // keys: medium, 64 .. 0, chunk lists
    __shared__ uint16_t s_code[16384], s_loc[16384];
    const uint32_t b = blockIdx.x, tid = threadIdx.x, lane = tid & 63u, wv = tid >> 6;
    const uint32_t a0 = ablk[b], na = ablk[b + 1] - a0;   // (< TB: every agent costs one)
    auto code = [&](uint32_t i) {
        const uint64_t r = (uint64_t)a0 + i;
        const uint32_t d = r < nrows ? off[r + 1] - off[r] : 0u;
        return d <= WIN_HMAX ? d : ORD_HUGE;
    };
    auto key = [](uint32_t c) { return c <= 64u ? 65u - c : c == ORD_HUGE ? 66u : 0u; };
    if (tid < 67) s_first[tid] = 0;
    __syncthreads();
    for (uint32_t i = tid; i < na; i += 1024) atomicAdd(&s_first[key(code(i))], 1u);
    __syncthreads();
    if (tid == 0) {
        uint32_t f = 0;
        for (int k = 0; k < 67; k++) {
            const uint32_t c = s_first[k];
            s_first[k] = f;
            f += c;
        }
    }
    __syncthreads();
    for (uint32_t i = tid; i < na; i += 1024) {
        const uint32_t c = code(i), p = atomicAdd(&s_first[key(c)], 1u);
        s_code[p] = (uint16_t)c;
        s_loc[p] = (uint16_t)i;
        aord[a0 + p] = i | c << 14;
    }
    __syncthreads();
    const uint32_t ng = (na + 63) / 64;
    for (uint32_t g = wv; g < ng; g += 16) {
        const uint32_t p = g * 64 + lane, c = p < na ? s_code[p] : ORD_HUGE;
        const uint32_t t = wave_incl_scan(c != ORD_HUGE ? c : 0u);
        if (lane == 63) s_gb[g] = t;
    }
    __syncthreads();
    if (tid == 0) {
        uint32_t f = 0;
        for (uint32_t g = 0; g < ng; g++) {
            const uint32_t t = s_gb[g];
            s_gb[g] = f;
            f += t;
        }
    }
    __syncthreads();
    for (uint32_t g = tid; g < ng; g += 1024) gbase[win_group(a0, b) + g] = s_gb[g];
    for (uint32_t g = wv; g < ng; g += 16) {
        const uint32_t p = g * 64 + lane, c = p < na ? s_code[p] : ORD_HUGE;
        const uint32_t r = a0 + (p < na ? s_loc[p] : 0u), l0 = C[r] - r;
        const bool light = c <= 64u, med = !light && c != ORD_HUGE;
        const uint32_t md = med ? c : 0u, mi = wave_incl_scan(md);
        for (uint32_t q = 0; q < md; q++) sl[l0 + q] = (uint16_t)(s_gb[g] + mi - md + q);
        const uint32_t nm = (uint32_t)__popcll(__ballot(med)), d = light ? c : 0u;
        uint32_t s0 = s_gb[g] + (uint32_t)__builtin_amdgcn_readlane((int)mi, 63) + lane - nm;
        for (uint32_t q = 0; q < 64; q++) {
            const uint64_t m = __ballot(d > q);
            if (!m) break;
            if (d > q) sl[l0 + q] = (uint16_t)s0;
            s0 += (uint32_t)__popcll(m);
        }
    }
}

// plan sort key of each CSR slot: window * (nb + 1) + (chunk-list row ? nb : block)
__global__ void k_win_keys(const uint32_t* __restrict__ off, const uint32_t* __restrict__ src, uint64_t nrows,
                           const uint32_t* __restrict__ C, uint32_t S, uint32_t nb, uint32_t wsz,
                           uint32_t* __restrict__ keys) {
    const uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= nrows) return;
    const uint32_t b = off[r], e = off[r + 1];
    const uint32_t col = e - b > WIN_HMAX ? nb : C[r] / S;
    for (uint32_t k = b; k < e; k++) keys[k] = ((src[k] - 1u) / wsz) * (nb + 1u) + col;
}

// per plan entry j: local source index, inverse permutation; the first plan
// entry of every window (wstart, W + 1 entries)
__global__ void k_win_fill(const uint32_t* __restrict__ src, const uint32_t* __restrict__ keys,
                           const uint32_t* __restrict__ perm, uint64_t ne, uint32_t nb, uint32_t wsz, uint32_t W,
                           uint16_t* __restrict__ psl, uint32_t* __restrict__ pinv, uint32_t* __restrict__ wstart) {
    const uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= ne) return;
    const uint32_t k = perm[j], w = keys[j] / (nb + 1u);
    psl[j] = (uint16_t)((src[k] - 1u) - w * wsz);
    pinv[k] = (uint32_t)j;
    const int64_t wp = j ? (int64_t)(keys[j - 1] / (nb + 1u)) : -1;
    for (int64_t q = wp + 1; q <= (int64_t)w; q++) wstart[q] = (uint32_t)j;
    if (j == ne - 1)
        for (uint32_t q = w + 1; q <= W; q++) wstart[q] = (uint32_t)ne;
}

// list sort key of each staged in-edge (numbered by the staged prefix
// C[r] - r + position): block * W + window; its CSR slot
__global__ void k_win_lkeys(const uint32_t* __restrict__ off, const uint32_t* __restrict__ src, uint64_t nrows,
                            const uint32_t* __restrict__ C, uint32_t S, uint32_t W, uint32_t wsz,
                            uint32_t* __restrict__ keys, uint32_t* __restrict__ kidx) {
    const uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= nrows) return;
    const uint32_t b = off[r], d = off[r + 1] - b;
    if (d > WIN_HMAX) return;
    const uint32_t blk = C[r] / S, l0 = C[r] - (uint32_t)r;
    for (uint32_t q = 0; q < d; q++) {
        keys[l0 + q] = blk * W + (src[b + q] - 1u) / wsz;
        kidx[l0 + q] = b + q;
    }
}

// 1 at the first list entry of each run (sorted keys)
__global__ void k_win_starts(const uint32_t* __restrict__ keys, uint64_t nl, uint32_t* __restrict__ flag) {
    const uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= nl) return;
    flag[e] = (e == 0 || keys[e] != keys[e - 1]) ? 1u : 0u;
}

// packed lists: slot | run start, weight in list order; per run its plan
// position and list index in the block (ridx: exclusive run count)
__global__ void k_win_pack(const uint32_t* __restrict__ keys, const uint32_t* __restrict__ order,
                           const uint32_t* __restrict__ kidx, const uint32_t* __restrict__ flag,
                           const uint32_t* __restrict__ ridx, const uint32_t* __restrict__ pinv,
                           const uint32_t* __restrict__ lbase, const uint16_t* __restrict__ sl, uint32_t W,
                           uint64_t nl, const float* __restrict__ w, uint16_t* __restrict__ tpk,
                           float* __restrict__ twt, uint32_t* __restrict__ prun, uint16_t* __restrict__ pfirst) {
    const uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= nl) return;
    const uint32_t idx = order[e], blk = keys[e] / W, k = kidx[idx];
    const uint32_t st = flag[e];
    tpk[e] = (uint16_t)(sl[idx] | (st ? WIN_START : 0u));
    twt[e] = w ? w[k] : 0.0f;
    if (st) {
        prun[ridx[e]] = pinv[k];
        pfirst[ridx[e]] = (uint16_t)(e - lbase[blk]);
    }
}

// first run of each block (nb + 1 entries) and each chunk's run count, at
// cbase[b 256 + (c % 16) 16 + c / 16]: the run counts of wave w's chunks
// (c = w, w + 16, ...) are 32 contiguous bytes
__global__ void k_win_rbase(const uint32_t* __restrict__ lbase, const uint32_t* __restrict__ ridx, uint32_t nb,
                            uint32_t cpb, uint32_t* __restrict__ rbase, uint16_t* __restrict__ cbase) {
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t b = (uint32_t)(t / cpb), c = (uint32_t)(t % cpb);
    if (b > nb) return;
    if (b == nb) {
        if (c == 0) rbase[nb] = ridx[lbase[nb]];
        return;
    }
    const uint32_t lb = lbase[b], L = lbase[b + 1] - lb;
    if (c == 0) rbase[b] = ridx[lb];
    cbase[(uint64_t)b * 256 + (c % 16) * 16 + c / 16] = (uint16_t)(64u * c < L ? ridx[lb + 64u * c] - ridx[lb] : 0u);
}

// heavy chunk lists: plan position and chunk slot per entry
__global__ void k_heavy_fill(const uint32_t* __restrict__ order, const uint32_t* __restrict__ kidx,
                             const uint16_t* __restrict__ tsl, const uint32_t* __restrict__ pinv, uint64_t nl,
                             uint32_t* __restrict__ hty, uint16_t* __restrict__ hslot) {
    const uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= nl) return;
    const uint32_t idx = order[e];
    hty[e] = pinv[kidx[idx]];
    hslot[e] = tsl[idx];
}

// in-edge count and chunk count of each heavy row
__global__ void k_heavy_sizes(const uint32_t* __restrict__ off, const uint32_t* __restrict__ heavy, uint64_t nheavy,
                              uint32_t chunk, uint32_t* __restrict__ deg, uint32_t* __restrict__ chunks) {
    const uint64_t h = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (h >= nheavy) return;
    const uint32_t r = heavy[h], d = off[r + 1] - off[r];
    deg[h] = d;
    chunks[h] = (d + chunk - 1) / chunk;
}

// one wave per heavy row: sort key (chunk, source window), CSR slot and
// slot within the chunk of each of its in-edges (numbered from hbase[h])
__global__ __launch_bounds__(256) void k_heavy_keys(const uint32_t* __restrict__ off,
                                                    const uint32_t* __restrict__ src,
                                                    const uint32_t* __restrict__ heavy, uint64_t nheavy,
                                                    const uint32_t* __restrict__ hbase,
                                                    const uint32_t* __restrict__ cbase, uint32_t psize,
                                                    uint32_t pbits, uint32_t chunk, uint32_t* __restrict__ keys,
                                                    uint32_t* __restrict__ kidx, uint16_t* __restrict__ tsl) {
    const uint64_t h = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    if (h >= nheavy) return;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t r = heavy[h], b = off[r], d = off[r + 1] - b, hb = hbase[h], cb = cbase[h];
    for (uint32_t t = lane; t < d; t = vh_row_next(t, d, 64)) {
        keys[hb + t] = ((cb + t / chunk) << pbits) | ((src[b + t] - 1u) / psize);
        kidx[hb + t] = b + t;
        tsl[hb + t] = (uint16_t)(t % chunk);
    }
}

// row, CSR start, degree and first chunk-list entry of each heavy row
__global__ void k_heavy_info(const uint32_t* __restrict__ off, const uint32_t* __restrict__ heavy, uint64_t nheavy,
                             const uint32_t* __restrict__ hbase, uint4* __restrict__ hinfo) {
    const uint64_t h = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (h >= nheavy) return;
    const uint32_t r = heavy[h], b = off[r];
    hinfo[h] = make_uint4(r, b, off[r + 1] - b, hbase[h]);
}

__global__ void k_heavy_rows(const uint32_t* __restrict__ off, uint64_t rows, uint64_t rowbase,
                             uint64_t nrows, uint32_t* __restrict__ list, uint32_t* __restrict__ cnt) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nrows) return;
    const uint64_t r = rowbase + i;
    if (off[r + 1] - off[r] > 64u) list[atomicAdd(cnt, 1u)] = (uint32_t)r;
}

// ----------------------------------------------------------------- contact
// state: health byte 0, susceptibility float at bytes 4-7.
// The step runs on per-slot flag bitmaps (64 slots per word): `sp` marks
// slots that are dead in the read state or die in this step, `dead` the
// former, `inf` slots infected in the read state. At 10^7 slots each is 1.25
// MB, in reach of every XCD's L2, but the 2 10^8 partner draws of a step are
// more than the L2s' random reads deliver (0.78 ms of them): so a draw first
// asks a filter in LDS, one bit per group of 2^fshift slots, the smallest
// groups that fit (8 slots at 10^7: 28% of the draws go on to `sp` with 4% of
// the slots marked).
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bool cbit(const uint64_t* __restrict__ b, uint64_t i) {
    return (b[i >> 6] >> (i & 63)) & 1ull;
}

// one thread per slot, whole blocks of 4 words (the last block's words past
// nwords are not stored)
__global__ __launch_bounds__(256) void k_contact_flags(const uint64_t* __restrict__ rs,
                                                       const uint8_t* __restrict__ died, uint64_t n,
                                                       uint32_t t, vh_contact_params p, uint64_t step,
                                                       ContactBits B) {
    __shared__ uint32_t s_f[4];
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t w = i >> 6;
    const uint32_t lane = threadIdx.x & 63u;
    const bool in = i < n;
    const bool dead = !in || died[i] != 0;
    const uint32_t h = in ? (uint32_t)(__builtin_nontemporal_load(rs + i) & 0xFFu) : 0u;
    const bool inf = in && h == VH_I;
    const bool dn = !dead && vh_u01(vh_hash(p.seed, vh_make_id(t, i + 1), step, VH_KEY_DEATH)) < p.p_death;
    const uint64_t md = __ballot(dead), mi = __ballot(inf), mn = __ballot(dn), m = md | mn;
    const uint64_t ms = __ballot(h == VH_S) & ~m;
    if (lane == 0 && w < B.nwords) {
        B.sp[w] = m;
        B.dead[w] = md;
        B.inf[w] = mi;
        B.sus[w] = ms;
        B.cnt[w] = (uint32_t)__popcll(mn);
    }
    if (B.filt) {   // 256 >> fshift bits per block
        const uint32_t g = B.fshift, nb = 64u >> g;
        const uint64_t f = __ballot(lane < nb && ((m >> ((lane << g) & 63u)) & ((1ull << (1u << g)) - 1ull)));
        uint8_t* out = B.filt + (uint64_t)blockIdx.x * (32u >> g);
        if (g <= 2) {
            if (lane == 0) {
                uint8_t* o = out + (threadIdx.x >> 6) * (8u >> g);
                if (g == 0) *(uint64_t*)o = f;
                else if (g == 1) *(uint32_t*)o = (uint32_t)f;
                else *(uint16_t*)o = (uint16_t)f;
            }
        } else {
            if (lane == 0) s_f[threadIdx.x >> 6] = (uint32_t)f;
            __syncthreads();
            if (threadIdx.x == 0) {
                const uint32_t v = s_f[0] | s_f[1] << nb | s_f[2] << 2 * nb | s_f[3] << 3 * nb;
                if (g == 3) *(uint32_t*)out = v;
                else if (g == 4) *(uint16_t*)out = (uint16_t)v;
                else *out = (uint8_t)v;
            }
        }
    }
}

// the partner of draw r of contact cc (0-based slot; n < 2^32)
__device__ __forceinline__ uint32_t contact_draw(uint64_t pre, uint32_t n, const vh_contact_params& p, uint32_t cc,
                                                 uint32_t r) {
    const uint64_t hh = vh_hash_fin(pre, VH_KEY_PARTNER + (uint64_t)cc * p.max_redraw + r);
    return __umulhi((uint32_t)(hh >> 32), n);
}
// contact cc of slot i: draws, from draw r on, until a partner that lives in
// the read state and is not i (at most max_redraw in all); false when there is
// none or it dies in this step
__device__ __forceinline__ bool contact_partner(uint64_t pre, uint32_t n, const vh_contact_params& p, uint64_t i,
                                                uint32_t cc, uint32_t r, const ContactBits& B, uint32_t& j) {
    for (; r < p.max_redraw; r++) {
        j = contact_draw(pre, n, p, cc, r);
        if (j == i) continue;
        if (!cbit(B.sp, j)) return true;
        if (!cbit(B.dead, j)) return false;   // dies in this step: not kept
    }
    return false;
}
// A wave's contacts that draw again (todo: a bit each), 64 at a time, one per
// lane: every lane calls f(act, lane of the slot, contact). With 2% deaths a
// slot has 0.8 of them and the worst of 64 slots four: on the slots' own lanes,
// a wave goes four times through the draws and their lookups for 51 of them
// (k_contact_edges at 10^7 slots: 238 us so, 220 in pairs, 211 with the draws
// after the first only; k_contact_main, whose ALU is busy anyway and whose
// filter leaves no LDS for the lists without larger groups elsewhere, 441 and
// 460: not there).
template <class F>
__device__ __forceinline__ void contact_pairs(uint32_t todo, uint16_t* pair, F f) {
    const uint32_t lane = threadIdx.x & 63u;
    while (__ballot(todo != 0u)) {
        const uint32_t c = (uint32_t)__popc(todo), incl = wave_incl_scan(c);
        const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
        for (uint32_t k = incl - c; todo && k < 64u; k++) {
            pair[k] = (uint16_t)(lane | (uint32_t)__builtin_ctz(todo) << 6);
            todo &= todo - 1u;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const uint32_t e = lane < total ? pair[lane] : lane;
        f(lane < total, e & 63u, e >> 6);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}
__device__ __forceinline__ uint64_t contact_shfl(uint64_t v, uint32_t lane) {
    return (uint64_t)(uint32_t)__shfl((int)(uint32_t)v, (int)lane, 64) |
           (uint64_t)(uint32_t)__shfl((int)(uint32_t)(v >> 32), (int)lane, 64) << 32;
}
// Infections: a susceptible slot gets infected when some in-edge (a contact of
// the last step) has an infected source and a draw below beta * susceptibility.
// "Some" has no order: the draw (ALU) first, the source's flag only for the
// few draws below. A block lists the susceptible slots of INF_W words and its
// threads take them off the list, so that all lanes draw: at the endemic state
// 15% of the slots are susceptible, and with each slot on its own lane every
// wave went through all draws for those (390 us of the 10^7-slot step; listed,
// with the draws before the lookups, 68 us). The word of `sus` is replaced by
// the slots that get infected.
constexpr uint32_t INF_W = 32;
__global__ __launch_bounds__(256) void k_contact_infect(const uint32_t* __restrict__ off,
                                                        const uint32_t* __restrict__ src,
                                                        const uint64_t* __restrict__ rs, uint64_t nrows,
                                                        uint64_t rowbase, uint32_t t, vh_contact_params p,
                                                        uint64_t step, ContactBits B) {
    __shared__ uint32_t s_n, s_bits[2 * INF_W];
    __shared__ uint16_t s_list[64 * INF_W];
    const uint32_t tid = threadIdx.x;
    const uint64_t w0 = (uint64_t)blockIdx.x * INF_W;
    if (tid == 0) s_n = 0;
    if (tid < 2 * INF_W) s_bits[tid] = 0;
    __syncthreads();
    for (uint32_t q = tid; q < 64 * INF_W; q += 256) {   // a wave: the slots of a word
        const uint64_t w = w0 + (q >> 6);
        const uint64_t m = w < B.nwords ? B.sus[w] : 0ull;
        if (!m) continue;   // uniform per wave
        uint32_t base = 0;
        if ((q & 63u) == 0) base = atomicAdd(&s_n, (uint32_t)__popcll(m));
        base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
        const uint32_t l = q & 63u;
        if ((m >> l) & 1ull) s_list[base + (uint32_t)__popcll(m & ((1ull << l) - 1ull))] = (uint16_t)q;
    }
    __syncthreads();
    for (uint32_t k = tid; k < s_n; k += 256) {
        const uint32_t q = s_list[k];
        const uint64_t i = w0 * 64 + q;
        if (i >= nrows) continue;
        const uint32_t b = off[rowbase + i], e = off[rowbase + i + 1];
        if (b == e) continue;
        const double pinf = p.beta * (double)__uint_as_float((uint32_t)(rs[i] >> 32));
        const uint64_t pre = vh_hash_pre(p.seed, vh_make_id(t, i + 1), step);
        if (vh_any_infecting(pre, vh_u01_below(pinf), b, e, [&](uint32_t x) { return cbit(B.inf, src[x] - 1); }))
            atomicOr(&s_bits[q >> 5], 1u << (q & 31u));
    }
    __syncthreads();
    if (tid < INF_W && w0 + tid < B.nwords)
        B.sus[w0 + tid] = (uint64_t)s_bits[2 * tid] | (uint64_t)s_bits[2 * tid + 1] << 32;
}
// health update of live slot i; true when it survives the step
__device__ __forceinline__ bool contact_health(const uint64_t* __restrict__ rs, uint64_t* __restrict__ ws,
                                               const vh_contact_params& p, const ContactBits& B, uint64_t i,
                                               uint64_t pre) {
    const uint64_t s = __builtin_nontemporal_load(rs + i);
    uint32_t h = (uint32_t)(s & 0xFFu);
    if (cbit(B.sp, i)) return false;   // live and marked: dies in this step
    if (h == VH_S) {
        if (cbit(B.sus, i)) h = VH_I;
    } else if (h == VH_I) {
        if (vh_u01(vh_hash_fin(pre, VH_KEY_RECOVER)) < p.gamma) h = VH_R;
    }
    __builtin_nontemporal_store((s & ~(uint64_t)0xFFu) | h, ws + i);
    return true;
}

// Health update, death flag, and which of up to 32 contacts of every slot are
// kept: `masks` gets a bit per kept contact and a bit per kept contact that
// was not its first draw, from which k_contact_edges draws the partners again
// (8 bytes a slot in place of 4 per contact written and read back). Blocks
// stay with the filter in LDS and take tiles of BS slots in turn. Four first
// draws at a time: their hashes, filter bits, the reads of `sp` that are left
// and of `dead` for those that `sp` marks are in flight together. What has to
// be drawn again (the slot itself, or dead in the read state) is noted and
// drawn after the loop, a draw of some contact of its own per lane and round:
// a wave goes round as often as its busiest lane has draws, not as the busiest
// of each contact. Bound: instruction issue, 50 vector instructions a draw with
// seven quarter-rate products among them (0.3 ms for 2 10^8 draws). 10^7 slots,
// 20 contacts, 2% deaths (and, in brackets, 50%): with infections in the same
// loop, each draw in the L2 and the partners to a log 1055 us (1908); rejected
// first draws begun anew contact by contact after the loop 441 (2185), so 425
// (1177). Filter groups of 16 slots and two blocks per CU 500 in place of 441;
// 2, 5, 8 or 10 draws at a time 465, 437, 476, 436.
template <int BS, bool FILTER>
__global__ __launch_bounds__(BS) void k_contact_main(const uint64_t* __restrict__ rs, uint64_t* __restrict__ ws,
                                                     uint8_t* __restrict__ died_now, uint32_t n, uint32_t t,
                                                     vh_contact_params p, uint64_t step, ContactBits B,
                                                     uint32_t fwords, uint2* __restrict__ masks) {
    extern __shared__ u32x4 lds_v[];   // the filter: fwords words, a multiple of 4
    const uint32_t* F = (const uint32_t*)lds_v;
    const uint32_t tid = threadIdx.x, C = p.n_contacts;
    for (uint32_t q = tid; q < fwords / 4; q += BS) lds_v[q] = ((const u32x4*)B.filt)[q];
    __syncthreads();
    for (uint64_t i0 = (uint64_t)blockIdx.x * BS; i0 < n; i0 += (uint64_t)gridDim.x * BS) {
        const uint64_t i = i0 + tid;
        uint32_t km = 0, rm = 0;
        if (i < n && !cbit(B.dead, i)) {
            const uint64_t pre = vh_hash_pre(p.seed, vh_make_id(t, i + 1), step);
            if (contact_health(rs, ws, p, B, i, pre) && p.max_redraw) {
                uint32_t again = 0;   // contacts to draw again: the slot itself, or dead in the read state
                for (uint32_t c0 = 0; c0 < C; c0 += 4) {
                    uint32_t j[4];
                    bool ask[4];
                    uint32_t word[4];
#pragma unroll
                    for (uint32_t u = 0; u < 4; u++) j[u] = contact_draw(pre, n, p, c0 + u, 0);
#pragma unroll
                    for (uint32_t u = 0; u < 4; u++) {
                        const uint32_t g = j[u] >> B.fshift;
                        ask[u] = !FILTER || ((F[g >> 5] >> (g & 31u)) & 1u);
                    }
#pragma unroll
                    for (uint32_t u = 0; u < 4; u++) {
                        word[u] = 0;
                        if (ask[u]) word[u] = ((const uint32_t*)B.sp)[j[u] >> 5];
                    }
#pragma unroll
                    for (uint32_t u = 0; u < 4; u++) {
                        ask[u] = (word[u] >> (j[u] & 31u)) & 1u;   // dead or dying
                        word[u] = 0;
                        if (ask[u]) word[u] = ((const uint32_t*)B.dead)[j[u] >> 5];
                    }
#pragma unroll
                    for (uint32_t u = 0; u < 4; u++) {
                        const bool self = j[u] == (uint32_t)i, dead = (word[u] >> (j[u] & 31u)) & 1u;
                        km |= !self && !ask[u] ? 1u << (c0 + u) : 0u;
                        again |= self || dead ? 1u << (c0 + u) : 0u;
                    }
                }
                const uint32_t all = C == 32 ? 0xFFFFFFFFu : (1u << C) - 1u;   // (the last group may pass C)
                km &= all;
                again &= p.max_redraw > 1 ? all : 0u;
                for (uint32_t r = 1; again;) {   // a draw each time round, of whichever contact the lane is at
                    const uint32_t cc = (uint32_t)__builtin_ctz(again), jj = contact_draw(pre, n, p, cc, r);
                    bool redo = jj == (uint32_t)i;
                    if (!redo) {
                        redo = cbit(B.sp, jj);
                        if (!redo) {
                            km |= 1u << cc;
                            rm |= 1u << cc;
                        } else {
                            redo = cbit(B.dead, jj);
                        }
                    }
                    r++;
                    if (!redo || r == p.max_redraw) {
                        again &= again - 1u;
                        r = 1;
                    }
                }
            }
        }
        if (i < n) {
            masks[i] = make_uint2(km, rm);
            died_now[i] = cbit(B.sp, i) && !cbit(B.dead, i);
        }
        const uint32_t sum = wave_incl_scan((uint32_t)__popc(km));
        if ((tid & 63u) == 63u && i >> 6 < B.nwords) B.cnt[B.nwords + (i >> 6)] = sum;
    }
}

// The rebuilt contact CSR (row i = caller slot i, kept partners in draw
// order) from the masks: cpos is the scan of B.cnt (its entry nwords: the
// deaths, then contacts before each word of slots). A wave's rows are one
// range of the CSR: the partners are drawn into LDS at their place and
// written out as one range per block. Dynamic LDS: 256 * n_contacts words.
// Bound: the 800 MB of a 2 10^8 contact CSR (0.16 ms) and the hashes
// (0.22 ms); from the log it was 337 us, so 211 us (the contacts drawn again
// on their slots' lanes 238).
__global__ __launch_bounds__(256) void k_contact_edges(uint32_t n, uint32_t t, vh_contact_params p, uint64_t step,
                                                       ContactBits B, const uint2* __restrict__ masks,
                                                       const uint32_t* __restrict__ cpos, uint32_t* __restrict__ off,
                                                       uint32_t* __restrict__ src) {
    extern __shared__ u32x4 lds_v[];
    uint32_t* lds = (uint32_t*)lds_v;
    const uint32_t tid = threadIdx.x, C = p.n_contacts;
    const uint64_t i0 = (uint64_t)blockIdx.x * 256, i = i0 + tid, w0 = i0 >> 6;
    const uint64_t w1 = w0 + 4 < B.nwords ? w0 + 4 : B.nwords;
    const uint32_t deaths = cpos[B.nwords];
    const uint32_t base = cpos[B.nwords + w0] - deaths, end = cpos[B.nwords + w1] - deaths;
    uint2 m = make_uint2(0u, 0u);
    if (i < n) m = masks[i];
    const uint32_t cnt = (uint32_t)__popc(m.x), incl = wave_incl_scan(cnt);
    __shared__ uint16_t s_pair[256];
    uint32_t r0 = 0;   // first of the slot's contacts in lds
    const uint64_t pre = vh_hash_pre(p.seed, vh_make_id(t, i + 1), step);
    if (i < n) {
        const uint32_t o = cpos[B.nwords + (i >> 6)] - deaths + incl - cnt;
        off[i] = o;
        if (i == n - 1) off[n] = o + cnt;
        r0 = o - base;
        uint32_t* row = lds + r0;
        const uint32_t first = m.x & ~m.y;
        for (uint32_t cc = 0; cc < C; cc++)
            if ((first >> cc) & 1u)
                row[__popc(m.x & ((1u << cc) - 1u))] = contact_draw(pre, n, p, cc, 0) + 1u;
    }
    contact_pairs(m.y, s_pair + (tid & ~63u), [&](bool act, uint32_t who, uint32_t cc) {
        const uint64_t pw = contact_shfl(pre, who);
        const uint32_t mw = (uint32_t)__shfl((int)m.x, (int)who, 64), rw = (uint32_t)__shfl((int)r0, (int)who, 64);
        uint32_t j = 0;
        if (act) {
            (void)contact_partner(pw, n, p, (i & ~(uint64_t)63) + who, cc, 1, B, j);   // (kept, and not its first draw)
            lds[rw + (uint32_t)__popc(mw & ((1u << cc) - 1u))] = j + 1u;
        }
    });
    __syncthreads();
    for (uint32_t q = tid; q < end - base; q += 256) __builtin_nontemporal_store(lds[q], src + base + q);
}

// More than 32 contacts per slot: the kept partners of a slot go to a
// fixed-stride log (row i at log[i * n_contacts]), their counts to `kept`.
__global__ __launch_bounds__(256) void k_contact_main_log(const uint64_t* __restrict__ rs, uint64_t* __restrict__ ws,
                                                          uint8_t* __restrict__ died_now, uint32_t n, uint32_t t,
                                                          vh_contact_params p, uint64_t step, ContactBits B,
                                                          uint32_t* __restrict__ kept, uint32_t* __restrict__ log) {
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    uint32_t nk = 0;
    if (!cbit(B.dead, i)) {
        const uint64_t pre = vh_hash_pre(p.seed, vh_make_id(t, i + 1), step);
        if (contact_health(rs, ws, p, B, i, pre)) {
            uint32_t* row = log + i * p.n_contacts;
            for (uint32_t cc = 0; cc < p.n_contacts; cc++) {
                uint32_t j;
                if (contact_partner(pre, n, p, i, cc, 0, B, j)) row[nk++] = j + 1u;
            }
        }
    }
    kept[i] = nk;
    died_now[i] = cbit(B.sp, i) && !cbit(B.dead, i);
}
// the CSR from the log (pos: the scan of `kept`)
__global__ __launch_bounds__(256) void k_contact_edges_log(uint64_t n, uint32_t C, const uint32_t* __restrict__ kept,
                                                           const uint32_t* __restrict__ log,
                                                           const uint32_t* __restrict__ pos,
                                                           uint32_t* __restrict__ off, uint32_t* __restrict__ src) {
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const uint32_t k = kept[i], o = pos[i];
    off[i] = o;
    if (i == n - 1) off[n] = o + k;
    for (uint32_t r = 0; r < k; r++) src[o + r] = log[i * C + r];
}

// Newborns and deaths go by bytes of the bitmaps, a thread each. At 10^7 slots
// with 2% and with 50% deaths, newborns take 14 and 68 us and deaths 6 and 17;
// by words, whose 64 slots are a thread's chain of reads and writes, 12 and 147
// and 5 and 50; by slots, whose waves mostly hold one death or none, 36 and 71
// and 19 and 34.
// The slots i0 .. i0 + 7 of this thread that die in this step, and the number
// of the first of them
__device__ __forceinline__ uint32_t dying_byte(const ContactBits& B, const uint32_t* __restrict__ dpos, uint64_t& i0,
                                               uint64_t& g) {
    const uint64_t q = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x, w = q >> 3;
    const uint32_t s = 8u * (uint32_t)(q & 7u);
    if (w >= B.nwords) return 0u;
    const uint64_t m = B.sp[w] & ~B.dead[w];
    i0 = 8 * q;
    g = dpos[w] + (uint64_t)__popcll(m & ((1ull << s) - 1ull));
    return (uint32_t)(m >> s) & 0xFFu;
}
// Newborns of this step's deaths, in slot order of the dying callers: the top
// of the reuse stack first, then fresh slots (src/AgentMethods.jl:37-89).
__global__ void k_contact_births(uint32_t t, vh_contact_params p, uint64_t step, ContactBits B,
                                 const uint32_t* __restrict__ dpos, const uint32_t* __restrict__ reuse,
                                 uint64_t nreuse, uint64_t nextid, uint64_t* __restrict__ ws,
                                 uint8_t* __restrict__ died) {
    uint64_t g, i0;
    for (uint32_t m = dying_byte(B, dpos, i0, g); m; m &= m - 1u, g++) {
        const uint64_t i = i0 + (uint32_t)__builtin_ctz(m);
        const uint64_t slot = g < nreuse ? reuse[nreuse - 1 - g] : nextid + (g - nreuse);
        const float ns = 0.5f + 0.5f * vh_u01f(vh_hash(p.seed, vh_make_id(t, i + 1), step, VH_KEY_BIRTH));
        ws[slot - 1] = (uint64_t)VH_S | ((uint64_t)__float_as_uint(ns) << 32);
        died[slot - 1] = 0;
    }
}

// this step's deaths onto the reuse stack in slot order (src/AgentMethods.jl:314-345)
__global__ void k_contact_deaths(ContactBits B, const uint32_t* __restrict__ dpos, uint32_t* __restrict__ reuse,
                                 uint64_t base, uint8_t* __restrict__ died) {
    uint64_t g, i0;
    for (uint32_t m = dying_byte(B, dpos, i0, g); m; m &= m - 1u, g++) {
        const uint64_t i = i0 + (uint32_t)__builtin_ctz(m);
        reuse[base + g] = (uint32_t)(i + 1);
        died[i] = 1;
    }
}

// rows past the last caller (fresh newborn slots) are empty
__global__ void k_contact_extend(uint32_t* __restrict__ off, uint64_t from_row, uint64_t rows) {
    uint64_t r = from_row + 1 + (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r <= rows) off[r] = off[from_row];
}

// ----------------------------------------------------------------- raster stencils
// Cell i of a raster (column-major) has coordinates c; its in-edges over a
// stencil come from org = c - off[k] (wrapped per dimension when periodic,
// else only when inside the raster), one per stencil offset k, ordered as
// connect_raster_neighbors! inserts them: by org's index, then by k.
__device__ inline void cell_coords(const StencilSpec& sp, uint64_t i, int64_t* c) {
    for (uint32_t d = 0; d < sp.ndims; d++) {
        c[d] = (int64_t)(i % (uint64_t)sp.dims[d]);
        i /= (uint64_t)sp.dims[d];
    }
}
__device__ inline bool stencil_org(const StencilSpec& sp, const int64_t* c, uint32_t k, uint64_t& org) {
    uint64_t lin = 0, stride = 1;
    for (uint32_t d = 0; d < sp.ndims; d++) {
        int64_t o = c[d] - (int64_t)sp.off[k][d];
        if (o < 0 || o >= sp.dims[d]) {
            if (!sp.periodic) return false;
            o %= sp.dims[d];
            if (o < 0) o += sp.dims[d];
        }
        lin += (uint64_t)o * stride;
        stride *= (uint64_t)sp.dims[d];
    }
    org = lin;
    return true;
}
__global__ void k_stencil_degree(StencilSpec sp, uint64_t ncells, uint64_t rowbase, uint32_t* __restrict__ deg) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ncells) return;
    int64_t c[4];
    cell_coords(sp, i, c);
    uint32_t n = 0;
    uint64_t org;
    for (uint32_t k = 0; k < sp.nst; k++) n += stencil_org(sp, c, k, org) ? 1u : 0u;
    deg[rowbase + i] = n;
}
__global__ void k_stencil_fill(StencilSpec sp, uint64_t ncells, uint64_t rowbase,
                               const uint32_t* __restrict__ off, void* __restrict__ src, uint32_t src64,
                               uint8_t* __restrict__ st, uint32_t bytes) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ncells) return;
    int64_t c[4];
    cell_coords(sp, i, c);
    // keys (org << 8 | k), insertion-sorted; offsets are visited last to
    // first, so inside the raster (org falling with k) each key appends
    uint64_t key[VH_STENCIL_MAX];
    uint32_t n = 0;
    for (int k = (int)sp.nst - 1; k >= 0; k--) {
        uint64_t org;
        if (!stencil_org(sp, c, (uint32_t)k, org)) continue;
        const uint64_t kk = (org << 8) | (uint64_t)k;
        uint32_t j = n++;
        while (j > 0 && key[j - 1] > kk) {
            key[j] = key[j - 1];
            j--;
        }
        key[j] = kk;
    }
    const uint64_t o = off[rowbase + i];
    for (uint32_t j = 0; j < n; j++) {
        const uint64_t nr = sp.first_nr + (key[j] >> 8);
        if (src64) ((uint64_t*)src)[o + j] = vh_make_id(sp.cell_type, nr);
        else ((uint32_t*)src)[o + j] = (uint32_t)nr;
        for (uint32_t b = 0; b < bytes; b++) st[(o + j) * bytes + b] = sp.state[b];
    }
}

// diffuse (test/raster.jl diffuse) of every slot of the cell type: a slot is
// active when it is or some in-neighbour is; the in-neighbours of cell c are
// the cells c - offset of the stencil (wrapped when periodic), the sources
// k_stencil_fill gives its CSR row. Other slots of the type have no in-edges.
__global__ __launch_bounds__(256) void k_diffuse_stencil(StencilSpec sp, const uint8_t* __restrict__ rs,
                                                         uint8_t* __restrict__ ws, uint64_t nslots, uint64_t ncells,
                                                         uint32_t bytes, uint32_t f) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nslots) return;
    const uint8_t* r = rs + i * bytes;
    uint8_t* w = ws + i * bytes;
    for (uint32_t k = 0; k < bytes; k++) w[k] = r[k];
    uint8_t v = r[f] ? 1 : 0;
    const uint64_t nr = i + 1;
    if (!v && nr >= sp.first_nr && nr - sp.first_nr < ncells) {
        if (ncells <= 0x7FFFFFFFull) {
            // 32-bit coordinates; a wrap needs one add or subtract while the
            // offset is at most the extent (else the general path below)
            int32_t c[4], dim[4];
            uint32_t rest = (uint32_t)(nr - sp.first_nr);
            for (uint32_t d = 0; d < sp.ndims; d++) {
                dim[d] = (int32_t)sp.dims[d];
                c[d] = (int32_t)(rest % (uint32_t)dim[d]);
                rest /= (uint32_t)dim[d];
            }
            for (uint32_t k = 0; k < sp.nst && !v; k++) {
                uint32_t lin = 0, stride = 1;
                bool in = true;
                for (uint32_t d = 0; d < sp.ndims; d++) {
                    int32_t o = c[d] - (int32_t)sp.off[k][d];
                    if (o < 0 || o >= dim[d]) {
                        if (!sp.periodic) {
                            in = false;
                            break;
                        }
                        o = o < 0 ? o + dim[d] : o - dim[d];
                        if (o < 0 || o >= dim[d]) {
                            o %= dim[d];
                            if (o < 0) o += dim[d];
                        }
                    }
                    lin += (uint32_t)o * stride;
                    stride *= (uint32_t)dim[d];
                }
                if (in && rs[(sp.first_nr - 1 + lin) * bytes + f]) v = 1;
            }
        } else {
            int64_t c[4];
            cell_coords(sp, nr - sp.first_nr, c);
            for (uint32_t k = 0; k < sp.nst && !v; k++) {
                uint64_t org;
                if (stencil_org(sp, c, k, org) && rs[(sp.first_nr - 1 + org) * bytes + f]) v = 1;
            }
        }
    }
    w[f] = v;
}

// The same step for a type of one-byte records (a lone Bool) that is the
// raster and nothing else, as add_raster! makes it. A raster row is the cells
// of one line along dimension 0 (consecutive bytes), worked on in groups of 8
// cells, each from one 8-byte window per stencil offset. Only the first and
// the last two groups of a row meet its ends. The others are computed by
// waves of 64 groups of ROW_R rows: lane q works out the row of offset k + q (an
// offset outside the raster becomes the cells themselves, which changes
// nothing) and the wave takes it from there into a scalar address. The end
// groups of all rows go to lanes of their own waves (the last blocks in y):
// there a window is clamped into the row and shifted back, which leaves 0 for
// cells outside, and a periodic row ors in the wrapped end. Bound: 20 MB of
// cells read and written at 3162^2 are 4 us at the copy rate; instruction
// issue comes first. 3162^2 cells, Moore neighbourhood, nearly all inactive:
// k_diffuse_stencil 266 us (divisions and byte loads per cell); this with the
// rows in scalar instructions 24 us, with the rows by lanes but the end groups
// within the other waves 18 us, apart 16 us, two rows a wave 15 us (four: the
// same). A wave stops before the next ROW_U offsets once all its cells are
// active, a lane of the end groups before the next offset: diffusion fills the
// raster, and k_diffuse_stencil, which stops at a cell's first active
// neighbour, takes 11 us for 10^6 active cells of any stencil. 100^3 cells,
// 124 offsets, all active: 92 us without the stop, 11 with it; all inactive:
// 91 and 95 (602 by cells), 3000 x 2000 and Moore 14.6 and 14.7.
constexpr uint32_t ROW_U = 8;   // offsets at a time
constexpr uint32_t ROW_R = 2;   // rows of a wave
struct RowSpec {
    int32_t dims[4];
    uint32_t periodic, nst;                            // nst: a multiple of ROW_U (padded with zero offsets)
    uint32_t off[VH_STENCIL_MAX];                      // four signed bytes in a word
};
// 8 bytes at any address: three words from the word they start in and a byte
// shift. Reads up to 4 bytes past them (at an address that is a multiple of 4;
// the last group of the last row reads them behind the cells).
typedef uint32_t u32x3 __attribute__((ext_vector_type(3), aligned(4)));
__device__ __forceinline__ uint64_t ld8(const uint8_t* p) {
    const uint32_t m = (uint32_t)(uintptr_t)p & 3u;
    const u32x3 t = *(const u32x3*)(p - m);
    return (uint64_t)__builtin_amdgcn_alignbyte(t.y, t.x, m) | (uint64_t)__builtin_amdgcn_alignbyte(t.z, t.y, m) << 32;
}
constexpr uint64_t ALL_ACTIVE = 0x0101010101010101ull;   // (cells with other nonzero values go on, to the same result)
__device__ __forceinline__ uint64_t nonzero_bytes(uint64_t v) {   // each to 1
    return ((((v & 0x7F7F7F7F7F7F7F7Full) + 0x7F7F7F7F7F7F7F7Full) | v) >> 7) & 0x0101010101010101ull;
}
// the row at offset word `off` from the one at coordinates c (its first cell)
// and the offset along dimension 0; outside the raster the row itself and 0
__device__ __forceinline__ void stencil_row(const RowSpec& sp, const int32_t* c, uint32_t row, uint32_t off,
                                            int32_t& first, int32_t& dx) {
    uint32_t lin = 0, stride = 1;
    bool in = true;
    for (uint32_t d = 1; d < 4; d++) {
        const int32_t dim = sp.dims[d];
        const int32_t o = c[d] - (int32_t)(int8_t)(off >> (8 * d));   // |offset| <= extent
        const int32_t ow = o < 0 ? o + dim : o >= dim ? o - dim : o;
        in = in && (sp.periodic || ow == o);
        lin += (uint32_t)ow * stride;
        stride *= (uint32_t)dim;
    }
    dx = in ? (int32_t)(int8_t)off : 0;
    first = (int32_t)((in ? lin : row) * (uint32_t)sp.dims[0]);   // (< 2^31 cells)
}
__device__ __forceinline__ void row_coords(const RowSpec& sp, uint32_t row, int32_t* c) {
    for (uint32_t d = 1; d < 4; d++) {   // (unused dimensions have extent 1)
        const uint32_t dim = (uint32_t)sp.dims[d];
        c[d] = (int32_t)(dim == 1u ? 0u : row % dim);
        row = dim == 1u ? row : row / dim;
    }
}
__global__ __launch_bounds__(256) void k_diffuse_rows(RowSpec sp, const uint8_t* __restrict__ rs,
                                                      uint8_t* __restrict__ ws, uint32_t nrows, uint32_t yblocks) {
    const int32_t nx = sp.dims[0], groups = (nx + 7) / 8;
    if (blockIdx.y < yblocks) {   // groups 1 .. groups - 3
        const int32_t lane = (int32_t)(threadIdx.x & 63u);
        const uint32_t row = (blockIdx.y * 4u + (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6))) * ROW_R;
        if (row >= nrows) return;   // uniform
        const int32_t g = 1 + (int32_t)(blockIdx.x * 64u) + lane;
        if (g - lane > groups - 3) return;                  // uniform
        const int32_t x = 8 * (g <= groups - 3 ? g : 1);    // (every lane works out offsets)
        uint32_t rw[ROW_R];
        int32_t c[ROW_R][4];
        uint64_t v[ROW_R];
#pragma unroll
        for (uint32_t j = 0; j < ROW_R; j++) {
            rw[j] = row + j < nrows ? row + j : row;
            row_coords(sp, rw[j], c[j]);
            v[j] = ld8(rs + (uint64_t)rw[j] * (uint32_t)nx + x);
        }
        for (uint32_t k = 0; k < sp.nst; k += ROW_U) {
            uint64_t on = v[0];
#pragma unroll
            for (uint32_t j = 1; j < ROW_R; j++) on &= v[j];
            if (!__ballot(on != ALL_ACTIVE)) break;
            uint32_t off = sp.off[k];   // lane q: offset k + q, from scalar loads (the launch
#pragma unroll                          // arguments are slow to reach by vector loads)
            for (uint32_t q = 1; q < ROW_U; q++) off = lane == (int32_t)q ? sp.off[k + q] : off;
            uint64_t u[ROW_R][ROW_U];
#pragma unroll
            for (uint32_t j = 0; j < ROW_R; j++) {
                int32_t first, dx;
                stencil_row(sp, c[j], rw[j], off, first, dx);
                const int32_t from = first - dx;
#pragma unroll
                for (uint32_t q = 0; q < ROW_U; q++)
                    u[j][q] = ld8(rs + (int64_t)__builtin_amdgcn_readlane(from, (int)q) + x);
            }
#pragma unroll
            for (uint32_t j = 0; j < ROW_R; j++)
#pragma unroll
                for (uint32_t q = 0; q < ROW_U; q++) v[j] |= u[j][q];
        }
#pragma unroll
        for (uint32_t j = 0; j < ROW_R; j++) {
            const uint64_t w = nonzero_bytes(v[j]);
            if (g <= groups - 3 && row + j < nrows) __builtin_memcpy(ws + (uint64_t)(row + j) * (uint32_t)nx + x, &w, 8);
        }
        return;
    }
    int32_t c[4];
    // the end groups: 0, groups - 2 and groups - 1 of every row
    const uint32_t t = ((blockIdx.y - yblocks) * gridDim.x + blockIdx.x) * 256u + threadIdx.x;
    const uint32_t row = t / 3u, which = t % 3u;
    if (row >= nrows) return;
    const int32_t x = which == 0 ? 0 : 8 * (groups - 3 + (int32_t)which);   // (groups >= 2; twice the same for 2)
    row_coords(sp, row, c);
    const uint8_t* r0 = rs + (uint64_t)row * (uint32_t)nx;
    const int32_t xc = x + 8 > nx ? nx - 8 : x;   // clamped; the shift drops the cells before x
    uint64_t v = ld8(r0 + xc) >> (8 * (x - xc));
    for (uint32_t k = 0; k < sp.nst && v != ALL_ACTIVE; k++) {
        int32_t first, dx;
        stencil_row(sp, c, row, sp.off[k], first, dx);
        const uint8_t* r = rs + first;
        const int32_t a = x - dx, past = a + 8 - nx;   // cells a .. a + 7; a >= -7, past <= 14
        // the cells in the row, then (periodic) the wrapped ones
        uint64_t u = ld8(r + (a < 0 ? 0 : past > 0 ? nx - 8 : a));
        u = a < 0 ? u << (-8 * a) : past >= 8 ? 0ull : past > 0 ? u >> (8 * past) : u;
        if (sp.periodic && (a < 0 || past > 0)) {
            const uint64_t w = ld8(r + (a < 0 ? nx - 8 : past > 8 ? past - 8 : 0));
            u |= a < 0 ? w >> (8 * (8 + a)) : past < 8 ? w << (8 * (8 - past)) : w;
        }
        v |= u;
    }
    v = nonzero_bytes(v);
    uint8_t* w = ws + (uint64_t)row * (uint32_t)nx + x;
    for (int32_t q = 0; q < 8 && x + q < nx; q++) w[q] = (uint8_t)(v >> (8 * q));
}

}  // namespace

// ====================================================================== launchers
namespace vh {

int launch_generic(int tr, const DCtx* d_ctx, int ci, int call_t, uint64_t nslots, int pass,
                   int with_edge, hipStream_t st) {
    if (!nslots) return VH_OK;
    if (tr >= (int)VH_TR_USER) return launch_user_body((uint32_t)tr, d_ctx, ci, call_t, nslots, pass, with_edge, st);
    dim3 g(grid_for(nslots, 256)), b(256);
    switch (tr) {
#define CASE(X)                                                                            \
    case X:                                                                                \
        hipLaunchKernelGGL(k_generic<X>, g, b, 0, st, d_ctx, ci, call_t, pass, with_edge); \
        break;
        CASE(VH_TR_NOOP)
        CASE(VH_TR_SUM_NEIGHBORS)
        CASE(VH_TR_DIE_IF)
        CASE(VH_TR_ADD_SELF_EDGE)
        CASE(VH_TR_READD_EDGES)
        CASE(VH_TR_NEIGHBOR_FOO_EDGES)
        CASE(VH_TR_SPAWN)
        CASE(VH_TR_COUNT_EDGES)
        CASE(VH_TR_DIFFUSE)
        CASE(VH_TR_REMOVE_EDGES)
        CASE(VH_TR_MOVE_TO)
#undef CASE
    default:
        return set_error(VH_ERR_UNREGISTERED, "transition %d has no generic kernel", tr);
    }
    HIPCHECK(hipGetLastError());
    return VH_OK;
}

static int check_model_layout(Sim& s, int t, int et, uint32_t abytes, uint32_t ebytes, const char* who) {
    AgentStore& A = s.a[t];
    EdgeStore& E = s.e[et];
    if (A.bytes != abytes) return set_error(VH_ERR_ARG, "%s: agent state must be %u bytes", who, abytes);
    if (E.bytes != ebytes) return set_error(VH_ERR_ARG, "%s: edge state must be %u bytes", who, ebytes);
    if (VH_HAS(E.hints, VH_HINT_IGNOREFROM))
        return set_error(VH_ERR_ARG, "%s: the edge type must keep source ids", who);
    if (E.rows && E.nedges && (E.src64 || (int)E.src_type != t))
        return set_error(VH_ERR_ARG, "%s: edges must come from the called agent type only "
                                     "(one-agent-type model)", who);
    return VH_OK;
}


// Out-edges of E's rows (one agent type, rows from 0, 1-based sources up to
// nsrc): the transpose of its in-edges; the exposure bitmaps and the counters
static int build_out_csr(Sim& s, EdgeStore& E, uint64_t nsrc) {
    const uint64_t words = (nsrc + 31) / 32;
    if (E.out_version == E.version && E.out_n == nsrc && E.expo.p) return VH_OK;
    hipStream_t st = s.stream;
    RC(E.out_off.ensure((nsrc + 1) * 4 + 8, st));
    RC(E.out_dst.ensure(E.nedges * 4 + 8, st));
    OutSeg seg = {E.off.as<uint32_t>(), E.src.as<uint32_t>(), E.out_off.as<uint32_t>(), E.out_dst.as<uint32_t>(),
                  nullptr, 2 * words, E.rows, nsrc, E.nedges};
    E.out_version = ~0ull;
    RC(E.expo.ensure(2 * words * 4 + 16, st));
    seg.bits = E.expo.as<uint32_t>();
    out_edges_plan(&seg, 1);
    RC(build_out_edges(&seg, nullptr, 1, s.scratch, st));
    RC(E.expo_cnt.ensure(SIR_CTL_WORDS * 4 + 8, st));
    fill_u32(E.expo_cnt.as<uint32_t>(), 0u, SIR_CTL_WORDS, st);   // no complete counts yet
    HIPCHECK(hipGetLastError());
    E.out_version = E.version;
    E.out_n = nsrc;
    E.expo_parity = 0;
    return VH_OK;
}

int launch_sir(Sim& s, int t, int et, const vh_sir_params& p, uint64_t step) {
    RC(check_model_layout(s, t, et, 4, 0, "SIR"));
    AgentStore& A = s.a[t];
    EdgeStore& E = s.e[et];
    if (!A.writeable) return set_error(VH_ERR_ASSERT, "SIR: the agent type must be in `write`");
    if (!A.nslots) return VH_OK;
    // the exposure pass needs the in-edges of `t` only (rows from 0, sources
    // of `t`); it runs for at least sir_expose_min agents (default 65536:
    // below, its extra launch per step costs more than the draws it saves)
    // unless the options turn it off
    uint32_t* expo = nullptr;
    uint32_t* next = nullptr;
    uint32_t* cnt = nullptr;
    uint32_t parity = 0;
    const uint64_t nrows = E.rows ? E.nrows[t] : 0ull;
    if (nrows && E.nedges && !E.src64 && E.src_type == (uint32_t)t && E.rowbase[t] == 0 && nrows == E.rows &&
        A.nslots < 0xFFFFFFFFull && g_opts.sir_expose != 0 && (int64_t)A.nslots >= g_opts.sir_expose_min) {
        RC(build_out_csr(s, E, A.nslots));
        parity = E.expo_parity;
        E.expo_parity ^= 1u;
        const uint64_t words = (E.out_n + 31) / 32;
        expo = E.expo.as<uint32_t>() + parity * words;
        next = E.expo.as<uint32_t>() + (parity ^ 1u) * words;
        cnt = E.expo_cnt.as<uint32_t>();
        hipLaunchKernelGGL(k_sir_expose, dim3(grid_for(A.nslots, 1024)), dim3(256), 0, s.stream,
                           (const uint32_t*)A.rstate(), E.out_off.as<uint32_t>(), E.out_dst.as<uint32_t>(),
                           A.nslots, parity, cnt, expo);
    }
    hipLaunchKernelGGL(k_sir, dim3(grid_for(A.nslots, 256)), dim3(256), 0, s.stream,
                       E.off.as<uint32_t>(), E.src.as<uint32_t>(), (const uint32_t*)A.rstate(),
                       (uint32_t*)A.wstate(), A.nslots, nrows, E.rowbase[t],
                       (uint32_t)t, p.p_inf, p.seed, p.recovery, step, (const uint32_t*)expo, next, parity, cnt);
    HIPCHECK(hipGetLastError());
    return VH_OK;
}

// Rows of degree > 64 (heavy), ascending; built once per CSR version
int build_heavy_bins(Sim& s, EdgeStore& E, int t) {
    if (E.bins_version == E.version) return VH_OK;
    const uint64_t nrows = E.nrows[t];
    RC(E.heavy.ensure(nrows * 4 + 8, s.stream));
    uint32_t* cnt = (uint32_t*)s.d_stats.p;
    fill_u32(cnt, 0, 1, s.stream);
    if (nrows)
        hipLaunchKernelGGL(k_heavy_rows, dim3(grid_for(nrows, 256)), dim3(256), 0, s.stream,
                           E.off.as<uint32_t>(), E.rows, E.rowbase[t], nrows, E.heavy.as<uint32_t>(), cnt);
    uint32_t h = 0;
    HIPCHECK(hipMemcpyAsync(&h, cnt, 4, hipMemcpyDeviceToHost, s.stream));
    HIPCHECK(hipStreamSynchronize(s.stream));
    if (h > 1) {   // the atomic compaction's order varies between runs: sort it
        std::vector<uint32_t> rows(h);
        HIPCHECK(hipMemcpy(rows.data(), E.heavy.p, (size_t)h * 4, hipMemcpyDeviceToHost));
        std::sort(rows.begin(), rows.end());
        HIPCHECK(hipMemcpy(E.heavy.p, rows.data(), (size_t)h * 4, hipMemcpyHostToDevice));
    }
    E.nheavy = h;
    E.bins_version = E.version;
    return VH_OK;
}

// The gather plan of the in-edges of E (one target type at row 0, n agents,
// sources 1-based numbers <= n < 2^32) for states of `tb` bytes and windows
// of `wsz` sources: the plan's local source indices (psrc) and windows
// (wstart); the blocks (ablk, lbase), their light lists (tpk, twt), runs
// (rbase, prun, pfirst) and chunk run counts (cbase); the heavy rows' chunk
// lists (hbase, hty, hslot, hinfo). E.plan_ok stays false when a sort key
// would need more than 32 bits (the one-pass kernel runs).
int build_gather_plan(Sim& s, EdgeStore& E, uint32_t wsz, uint64_t n, uint32_t tb) {
    if (E.plan_version == E.version && E.plan_wsz == wsz && E.plan_n == n && E.plan_tb == tb) return VH_OK;
    hipStream_t st = s.stream;
    E.plan_ok = false;
    E.plan_version = E.version;
    E.plan_wsz = wsz;
    E.plan_n = n;
    E.plan_tb = tb;
    const uint64_t ne = E.nedges, nrows = E.rows;
    const uint32_t TB = tb == 8 ? WinCfg<double>::TB : WinCfg<float>::TB;
    const uint32_t CPB = TB / 64, S = TB - WIN_HMAX - 1;
    const uint32_t chunk = tb == 8 ? WinCfg<double>::CHUNK : WinCfg<float>::CHUNK;
    const uint64_t W = (n + wsz - 1) / wsz;
    if (!ne || ne + n >= 0xFFFFFFFFull || W > WIN_RUNS || nrows > n) return VH_OK;
    const uint32_t* off = E.off.as<uint32_t>();
    const uint32_t* src = E.src.as<uint32_t>();
    // blocks
    uint32_t* C = (uint32_t*)s.scratch.take((n + 1) * 4);
    uint32_t* cost = (uint32_t*)s.scratch.take(n * 4 + 4);
    if (!C || !cost) return set_error(VH_ERR_OOM, "scratch");
    hipLaunchKernelGGL(k_win_cost, dim3(grid_for(n, 256)), dim3(256), 0, st, off, n, nrows, cost);
    if (scan_excl_u32(cost, C, n, s.scratch, st)) return set_error(VH_ERR_DEVICE, "scan");
    uint32_t cl[2] = {0, 0};
    HIPCHECK(hipMemcpyAsync(cl, C + n - 1, 8, hipMemcpyDeviceToHost, st));
    HIPCHECK(hipStreamSynchronize(st));
    const uint32_t nb = cl[0] / S + 1;
    const uint64_t nl = (uint64_t)cl[1] - n;
    if (W * (nb + 1ull) > 0xFFFFFFFFull) return VH_OK;
    // the build's pieces in one block (the sorts take many), released at the
    // next reset when large
    const uint64_t nh_e = ne - nl;
    if (s.scratch.room(24 * ne + 30 * nl + 22 * nh_e + 32 * (uint64_t)nb + ne / 4 + ((uint64_t)256 << 20)))
        return set_error(VH_ERR_OOM, "scratch for the gather plan");
    s.scratch.shrink = true;
    uint32_t kbits = 1, lbits = 1;
    while ((1ull << kbits) < W * (nb + 1ull)) kbits++;
    while ((1ull << lbits) < W * (uint64_t)nb) lbits++;
    RC(E.ablk.ensure(((uint64_t)nb + 1) * 4 + 8, st));
    RC(E.lbase.ensure(((uint64_t)nb + 1) * 4 + 8, st));
    hipLaunchKernelGGL(k_win_blocks, dim3(grid_for(n + 1, 256)), dim3(256), 0, st, C, n, S, nb,
                       E.ablk.as<uint32_t>(), E.lbase.as<uint32_t>());
    RC(E.aord.ensure(n * 4 + 8, st));
    RC(E.gbase.ensure((n / 64 + nb + 1) * 4 + 8, st));
    uint16_t* sl = (uint16_t*)s.scratch.take(nl * 2 + 8);
    if (!sl) return set_error(VH_ERR_OOM, "scratch");
    hipLaunchKernelGGL(k_win_order, dim3(nb), dim3(1024), 0, st, off, nrows, C, E.ablk.as<uint32_t>(),
                       E.aord.as<uint32_t>(), E.gbase.as<uint32_t>(), sl);
    // plan order: stable sort of the CSR slots by (window, block or heavy)
    RC(E.psrc.ensure(ne * 2 + 16, st));
    RC(E.wstart.ensure((W + 1) * 4 + 8, st));
    uint32_t* pinv = (uint32_t*)s.scratch.take(ne * 4 + 4);
    {
        uint32_t* keys = (uint32_t*)s.scratch.take(ne * 4);
        uint32_t* vals = (uint32_t*)s.scratch.take(ne * 4);
        uint32_t* ka = (uint32_t*)s.scratch.take(ne * 4);
        uint32_t* va = (uint32_t*)s.scratch.take(ne * 4);
        if (!pinv || !keys || !vals || !ka || !va) return set_error(VH_ERR_OOM, "scratch");
        hipLaunchKernelGGL(k_win_keys, dim3(grid_for(nrows, 256)), dim3(256), 0, st, off, src, nrows, C, S, nb, wsz,
                           keys);
        if (radix_sort_pairs(&keys, &vals, ka, va, ne, kbits, true, s.scratch, st))
            return set_error(VH_ERR_DEVICE, "plan sort");
        hipLaunchKernelGGL(k_win_fill, dim3(grid_for(ne, 256)), dim3(256), 0, st, src, keys, vals, ne, nb, wsz,
                           (uint32_t)W, E.psrc.as<uint16_t>(), pinv, E.wstart.as<uint32_t>());
        HIPCHECK(hipGetLastError());
    }
    // light lists: each block's light in-edges by (window, slot)
    RC(E.tpk.ensure(nl * 2 + 8, st));
    RC(E.twt.ensure(nl * 4 + 8, st));
    RC(E.rbase.ensure(((uint64_t)nb + 1) * 4 + 8, st));
    RC(E.cbase.ensure((uint64_t)nb * 256 * 2 + 64, st));
    const float* w4 = E.bytes == 4 ? E.st.as<float>() : nullptr;
    {
        uint32_t* ridx = (uint32_t*)s.scratch.take((nl + 1) * 4);
        if (!ridx) return set_error(VH_ERR_OOM, "scratch");
        uint32_t nruns = 0;
        if (nl) {
            uint32_t* keys = (uint32_t*)s.scratch.take(nl * 4 + 4);
            uint32_t* vals = (uint32_t*)s.scratch.take(nl * 4 + 4);
            uint32_t* ka = (uint32_t*)s.scratch.take(nl * 4 + 4);
            uint32_t* va = (uint32_t*)s.scratch.take(nl * 4 + 4);
            uint32_t* kidx = (uint32_t*)s.scratch.take(nl * 4 + 4);
            uint32_t* flag = (uint32_t*)s.scratch.take(nl * 4 + 4);
            if (!keys || !vals || !ka || !va || !kidx || !flag) return set_error(VH_ERR_OOM, "scratch");
            hipLaunchKernelGGL(k_win_lkeys, dim3(grid_for(nrows, 256)), dim3(256), 0, st, off, src, nrows, C, S,
                               (uint32_t)W, wsz, keys, kidx);
            if (radix_sort_pairs(&keys, &vals, ka, va, nl, lbits, true, s.scratch, st))
                return set_error(VH_ERR_DEVICE, "list sort");
            hipLaunchKernelGGL(k_win_starts, dim3(grid_for(nl, 256)), dim3(256), 0, st, keys, nl, flag);
            if (scan_excl_u32(flag, ridx, nl, s.scratch, st)) return set_error(VH_ERR_DEVICE, "scan");
            HIPCHECK(hipMemcpyAsync(&nruns, ridx + nl, 4, hipMemcpyDeviceToHost, st));
            HIPCHECK(hipStreamSynchronize(st));
            RC(E.prun.ensure((uint64_t)nruns * 4 + 8, st));
            RC(E.pfirst.ensure((uint64_t)nruns * 2 + 8, st));
            hipLaunchKernelGGL(k_win_pack, dim3(grid_for(nl, 256)), dim3(256), 0, st, keys, vals, kidx, flag, ridx,
                               pinv, E.lbase.as<uint32_t>(), sl, (uint32_t)W, nl, w4, E.tpk.as<uint16_t>(),
                               E.twt.as<float>(), E.prun.as<uint32_t>(), E.pfirst.as<uint16_t>());
        } else {
            fill_u32(ridx, 0, 1, st);
            RC(E.prun.ensure(8, st));
            RC(E.pfirst.ensure(8, st));
        }
        hipLaunchKernelGGL(k_win_rbase, dim3(grid_for(((uint64_t)nb + 1) * CPB, 256)), dim3(256), 0, st,
                           E.lbase.as<uint32_t>(), ridx, nb, CPB, E.rbase.as<uint32_t>(), E.cbase.as<uint16_t>());
        HIPCHECK(hipGetLastError());
    }
    RC(E.wq.ensure(16, st));
    fill_u32(E.wq.as<uint32_t>(), 0, 3, st);   // queue (2) and the check flag
    {
        uint32_t nruns = 0, bad = 0;
        HIPCHECK(hipMemcpyAsync(&nruns, E.rbase.as<uint32_t>() + nb, 4, hipMemcpyDeviceToHost, st));
        HIPCHECK(hipStreamSynchronize(st));
        hipLaunchKernelGGL(k_win_check, dim3(grid_for(nb, 64)), dim3(64), 0, st, E.ablk.as<uint32_t>(),
                           E.lbase.as<uint32_t>(), E.rbase.as<uint32_t>(), E.prun.as<uint32_t>(),
                           E.pfirst.as<uint16_t>(), E.tpk.as<uint16_t>(), E.cbase.as<uint16_t>(),
                           E.aord.as<uint32_t>(), E.gbase.as<uint32_t>(), nb, n, nl,
                           (uint64_t)nruns, ne, TB, CPB, E.wq.as<uint32_t>() + 2);
        HIPCHECK(hipGetLastError());
        HIPCHECK(hipMemcpyAsync(&bad, E.wq.as<uint32_t>() + 2, 4, hipMemcpyDeviceToHost, st));
        HIPCHECK(hipStreamSynchronize(st));
        if (bad) return set_error(VH_ERR_DEVICE, "gather plan inconsistent");
    }
    // rows of in-degree above WIN_HMAX (from E.heavy, ascending): chunk lists
    // sorted by (chunk, window)
    uint64_t nheavy = 0;
    if (E.nheavy) {
        uint32_t* hd = (uint32_t*)s.scratch.take(E.nheavy * 4 + 4);
        uint32_t* hc = (uint32_t*)s.scratch.take(E.nheavy * 4 + 4);
        if (!hd || !hc) return set_error(VH_ERR_OOM, "scratch");
        hipLaunchKernelGGL(k_heavy_sizes, dim3(grid_for(E.nheavy, 256)), dim3(256), 0, st, off,
                           E.heavy.as<uint32_t>(), E.nheavy, chunk, hd, hc);
        std::vector<uint32_t> rows(E.nheavy), deg(E.nheavy);
        HIPCHECK(hipMemcpyAsync(rows.data(), E.heavy.p, E.nheavy * 4, hipMemcpyDeviceToHost, st));
        HIPCHECK(hipMemcpyAsync(deg.data(), hd, E.nheavy * 4, hipMemcpyDeviceToHost, st));
        HIPCHECK(hipStreamSynchronize(st));
        std::vector<uint32_t> huge;
        for (uint64_t h = 0; h < E.nheavy; h++)
            if (deg[h] > WIN_HMAX) huge.push_back(rows[h]);
        nheavy = huge.size();
        if (nheavy) {
            RC(E.huge.ensure(nheavy * 4 + 8, st));
            HIPCHECK(hipMemcpyAsync(E.huge.p, huge.data(), nheavy * 4, hipMemcpyHostToDevice, st));
            HIPCHECK(hipStreamSynchronize(st));
        }
    }
    E.plan_nhuge = nheavy;
    if (nheavy) {
        uint32_t* hd = (uint32_t*)s.scratch.take(nheavy * 4 + 4);
        uint32_t* hc = (uint32_t*)s.scratch.take(nheavy * 4 + 4);
        uint32_t* hcb = (uint32_t*)s.scratch.take(nheavy * 4 + 8);
        if (!hd || !hc || !hcb) return set_error(VH_ERR_OOM, "scratch");
        RC(E.hbase.ensure(nheavy * 4 + 8, st));
        hipLaunchKernelGGL(k_heavy_sizes, dim3(grid_for(nheavy, 256)), dim3(256), 0, st, off,
                           E.huge.as<uint32_t>(), nheavy, chunk, hd, hc);
        if (scan_excl_u32(hd, E.hbase.as<uint32_t>(), nheavy, s.scratch, st) ||
            scan_excl_u32(hc, hcb, nheavy, s.scratch, st))
            return set_error(VH_ERR_DEVICE, "scan");
        uint32_t htot[2] = {0, 0};
        HIPCHECK(hipMemcpyAsync(&htot[0], E.hbase.as<uint32_t>() + nheavy, 4, hipMemcpyDeviceToHost, st));
        HIPCHECK(hipMemcpyAsync(&htot[1], hcb + nheavy, 4, hipMemcpyDeviceToHost, st));
        HIPCHECK(hipStreamSynchronize(st));
        const uint32_t nhe = htot[0], nch = htot[1];
        uint32_t cbits = 1, wbits = 1;
        while ((1ull << cbits) < nch) cbits++;
        while ((1ull << wbits) < W) wbits++;
        if (cbits + wbits > 32 || nl + nhe != ne) return VH_OK;
        RC(E.hty.ensure((uint64_t)nhe * 4 + 8, st));
        RC(E.hslot.ensure((uint64_t)nhe * 2 + 8, st));
        uint32_t* keys = (uint32_t*)s.scratch.take((uint64_t)nhe * 4);
        uint32_t* vals = (uint32_t*)s.scratch.take((uint64_t)nhe * 4);
        uint32_t* ka = (uint32_t*)s.scratch.take((uint64_t)nhe * 4);
        uint32_t* va = (uint32_t*)s.scratch.take((uint64_t)nhe * 4);
        uint32_t* kidx = (uint32_t*)s.scratch.take((uint64_t)nhe * 4);
        uint16_t* tsl = (uint16_t*)s.scratch.take((uint64_t)nhe * 2);
        if (!keys || !vals || !ka || !va || !kidx || !tsl) return set_error(VH_ERR_OOM, "scratch");
        hipLaunchKernelGGL(k_heavy_keys, dim3(grid_for(nheavy * 64, 256)), dim3(256), 0, st, off, src,
                           E.huge.as<uint32_t>(), nheavy, E.hbase.as<uint32_t>(), hcb, wsz, wbits, chunk, keys,
                           kidx, tsl);
        if (radix_sort_pairs(&keys, &vals, ka, va, nhe, cbits + wbits, true, s.scratch, st))
            return set_error(VH_ERR_DEVICE, "chunk sort");
        hipLaunchKernelGGL(k_heavy_fill, dim3(grid_for(nhe, 256)), dim3(256), 0, st, vals, kidx, tsl, pinv,
                           (uint64_t)nhe, E.hty.as<uint32_t>(), E.hslot.as<uint16_t>());
        RC(E.hinfo.ensure(nheavy * 16 + 16, st));
        hipLaunchKernelGGL(k_heavy_info, dim3(grid_for(nheavy, 256)), dim3(256), 0, st, off,
                           E.huge.as<uint32_t>(), nheavy, E.hbase.as<uint32_t>(), E.hinfo.as<uint4>());
        HIPCHECK(hipGetLastError());
        // longest rows first: pass 2's waves take them round-robin, so every
        // wave's first row is among the longest
        std::vector<uint4> hi(nheavy);
        HIPCHECK(hipMemcpyAsync(hi.data(), E.hinfo.p, nheavy * 16, hipMemcpyDeviceToHost, st));
        HIPCHECK(hipStreamSynchronize(st));
        std::stable_sort(hi.begin(), hi.end(), [](const uint4& a, const uint4& b) { return a.z > b.z; });
        HIPCHECK(hipMemcpyAsync(E.hinfo.p, hi.data(), nheavy * 16, hipMemcpyHostToDevice, st));
        HIPCHECK(hipStreamSynchronize(st));
    } else if (nl != ne) {
        return VH_OK;
    }
    E.plan_nb = nb;
    E.plan_w = (uint32_t)W;
    E.plan_ok = true;
    return VH_OK;
}

// compute units of the current device (the persistent plan kernels run one
// block per CU)
static uint32_t device_cus() {
    static uint32_t cus[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (!cus[dev]) {
        int v = 0;
        if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0) {
            (void)hipGetLastError();
            v = 256;
        }
        cus[dev] = (uint32_t)v;
    }
    return cus[dev];
}

// the degree bins and, when the step takes the two-pass gather, its plan and
// gathered-value buffer for an opinion step of agent type t over edge type et
// (kept while the edges and the state type stay the same); `plan` tells which
static int opinion_plan(Sim& s, int t, int et, bool f32, bool& plan) {
    AgentStore& A = s.a[t];
    EdgeStore& E = s.e[et];
    const uint32_t tb = f32 ? 4 : 8;
    const uint64_t nrows = E.rows ? E.nrows[t] : 0;
    if (E.rows) RC(build_heavy_bins(s, E, t));
    // two-pass gather through a plan from a state vector of at least
    // opinion_plan_bytes (< 0: never), with source windows of
    // opinion_part_bytes (0 or more than 160 KB: 160 KB; widened to make at
    // most WIN_RUNS windows, a multiple of 4 sources)
    const int64_t plan_min = g_opts.opinion_plan_bytes;
    plan = plan_min >= 0 && E.rows && E.nedges && !E.src64 && E.src_type == (uint32_t)t &&
           E.rowbase[t] == 0 && nrows == E.rows && A.nslots < 0xFFFFFFFFull &&
           (uint64_t)A.nslots * tb >= (uint64_t)plan_min;
    if (plan) {
        const uint64_t cap = f32 ? WinCfg<float>::WSZ : WinCfg<double>::WSZ;
        uint64_t wsz = g_opts.opinion_part_bytes <= 0 ? cap : (uint64_t)g_opts.opinion_part_bytes / tb;
        if (wsz > cap) wsz = cap;
        const uint64_t wmin = (A.nslots + WIN_RUNS - 1) / WIN_RUNS;
        if (wsz < wmin) wsz = wmin;
        wsz = (wsz + 3) / 4 * 4;
        if (wsz > cap) plan = false;   // more sources than WIN_RUNS windows hold
        if (plan) {
            RC(build_gather_plan(s, E, (uint32_t)wsz, A.nslots, tb));
            plan = E.plan_ok;
        }
    }
    if (plan) RC(E.pval.ensure(E.nedges * tb + 16, s.stream));
    return VH_OK;
}

// Whether a launch's edges (source and weight) are more than the 256 MB of the
// cache behind the L2s, where they would stay from step to step: 24 simulations,
// us for 20 steps and reading the states, without and with: Float64 187 MB 5637
// and 5672, 280 MB 7114 and 6960, 374 MB 8172 and 7798; Float32 234 MB 4274 and
// 4378, 280 MB 4886 and 4905, 374 MB 5862 and 5796
static bool op_stream(uint64_t nedges) { return nedges * 8 > (256u << 20); }

int launch_opinion(Sim& s, int t, int et, const vh_opinion_params& p, bool f32, uint64_t step) {
    (void)step;
    RC(check_model_layout(s, t, et, f32 ? 4 : 8, 4, "opinion"));
    AgentStore& A = s.a[t];
    EdgeStore& E = s.e[et];
    if (!A.writeable) return set_error(VH_ERR_ASSERT, "opinion: the agent type must be in `write`");
    if (!A.nslots) return VH_OK;
    const uint64_t nrows = E.rows ? E.nrows[t] : 0;
    bool plan = false;
    RC(opinion_plan(s, t, et, f32, plan));
    const uint64_t nheavy = E.rows ? E.nheavy : 0;
    const uint32_t nlight = grid_for(A.nslots, 256);
    const uint32_t nh = (uint32_t)((nheavy + 3) / 4);
    if (!plan && g_opinion_defer && g_opinion_defer->stream == s.stream) {
        OpMember om;
        om.off = E.off.as<uint32_t>();
        om.src = E.src.as<uint32_t>();
        om.x = A.rstate();
        om.w = E.st.as<float>();
        om.xo = A.wstate();
        om.heavy = E.heavy.as<uint32_t>();
        om.n = A.nslots;
        om.nrows = nrows;
        om.rowbase = E.rowbase[t];
        om.nheavy = nheavy;
        om.nedges = E.nedges;
        om.eps = f32 ? (double)(float)p.eps : p.eps;
        om.nh = nh;
        om.blk0 = nlight + nh;   // (the block count until the launch assigns offsets)
        g_opinion_defer->m[f32 ? 1 : 0].push_back(om);
        return VH_OK;
    }
    if (!plan) {
        const dim3 g(nlight + nh), b(256);
        const bool stream = op_stream(E.nedges);
#define VH_OPINION(T, S) \
    hipLaunchKernelGGL((k_opinion<T, S>), g, b, 0, s.stream, E.off.as<uint32_t>(), E.src.as<uint32_t>(), \
                       (const T*)A.rstate(), E.st.as<float>(), (T*)A.wstate(), A.nslots, nrows, E.rowbase[t], \
                       (T)p.eps, E.heavy.as<uint32_t>(), nheavy, nh)
        if (f32 && stream) VH_OPINION(float, true);
        else if (f32) VH_OPINION(float, false);
        else if (stream) VH_OPINION(double, true);
        else VH_OPINION(double, false);
#undef VH_OPINION
        HIPCHECK(hipGetLastError());
        return VH_OK;
    }
    const dim3 g(device_cus()), bb(1024);
    if (f32) {
        hipLaunchKernelGGL(k_win_gather<float>, g, bb, 0, s.stream, E.psrc.as<uint16_t>(), (const float*)A.rstate(),
                           E.pval.as<float>(), E.wstart.as<uint32_t>(), E.plan_w, E.plan_wsz, A.nslots, E.nedges);
        hipLaunchKernelGGL(k_win_sum<float>, g, bb, 0, s.stream, E.aord.as<uint32_t>(), E.gbase.as<uint32_t>(),
                           (const float*)A.rstate(),
                           E.pval.as<float>(), E.st.as<float>(), (float*)A.wstate(), (float)p.eps,
                           E.hinfo.as<uint4>(), E.plan_nhuge, E.hty.as<uint32_t>(), E.hslot.as<uint16_t>(),
                           E.ablk.as<uint32_t>(), E.lbase.as<uint32_t>(), E.tpk.as<uint16_t>(), E.twt.as<float>(),
                           E.rbase.as<uint32_t>(), E.prun.as<uint32_t>(), E.pfirst.as<uint16_t>(),
                           E.cbase.as<uint16_t>(), E.plan_nb, E.wq.as<uint32_t>());
    } else {
        hipLaunchKernelGGL(k_win_gather<double>, g, bb, 0, s.stream, E.psrc.as<uint16_t>(),
                           (const double*)A.rstate(), E.pval.as<double>(), E.wstart.as<uint32_t>(), E.plan_w,
                           E.plan_wsz, A.nslots, E.nedges);
        hipLaunchKernelGGL(k_win_sum<double>, g, bb, 0, s.stream, E.aord.as<uint32_t>(), E.gbase.as<uint32_t>(),
                           (const double*)A.rstate(),
                           E.pval.as<double>(), E.st.as<float>(), (double*)A.wstate(), p.eps,
                           E.hinfo.as<uint4>(), E.plan_nhuge, E.hty.as<uint32_t>(), E.hslot.as<uint16_t>(),
                           E.ablk.as<uint32_t>(), E.lbase.as<uint32_t>(), E.tpk.as<uint16_t>(), E.twt.as<float>(),
                           E.rbase.as<uint32_t>(), E.prun.as<uint32_t>(), E.pfirst.as<uint16_t>(),
                           E.cbase.as<uint16_t>(), E.plan_nb, E.wq.as<uint32_t>());
    }
    HIPCHECK(hipGetLastError());
    return VH_OK;
}

// the plan of an opinion step built ahead of its first apply!, on the
// simulation's stream, which the call waits for; the build's scratch is
// released when large
extern "C" int vh_opinion_prepare(vh_sim_t h, uint8_t t, uint8_t et, int f32) {
    if (!h) return set_error(VH_ERR_ARG, "null simulation");
    Sim& s = h->s;
    if (!s.initialized) return set_error(VH_ERR_ASSERT, "opinion_prepare after finish_init! only");
    if (t < 1 || t > s.m->na) return set_error(VH_ERR_UNREGISTERED, "unregistered agent type");
    if (et >= s.m->ne) return set_error(VH_ERR_UNREGISTERED, "unregistered edge type");
    RC(check_model_layout(s, t, et, f32 ? 4 : 8, 4, "opinion"));
    if (!s.a[t].nslots) return VH_OK;
    s.scratch.reset(s.stream);
    bool plan = false;
    RC(opinion_plan(s, t, et, f32 != 0, plan));
    s.scratch.reset(s.stream);
    HIPCHECK(hipStreamSynchronize(s.stream));
    return VH_OK;
}

thread_local OpinionDefer* g_opinion_defer = nullptr;

int opinion_defer_launch(OpinionDefer& c, hipStream_t st, DevBuf& dev, void** host, size_t* host_cap,
                         size_t* host_off) {
    for (int k = 0; k < 2; k++) {
        std::vector<OpMember>& v = c.m[k];
        if (v.empty()) continue;
        uint64_t blocks = 0, edges = 0;
        for (OpMember& om : v) {
            edges += om.nedges;
            const uint32_t nb = om.blk0;   // the member's block count
            om.blk0 = (uint32_t)blocks;
            blocks += nb;
        }
        if (blocks > 0x7FFFFFF0ull) return set_error(VH_ERR_CAPACITY, "batched opinion launch too large");
        const size_t bytes = v.size() * sizeof(OpMember);
        if (*host_off + bytes > *host_cap) return set_error(VH_ERR_CAPACITY, "batch staging");
        memcpy((uint8_t*)*host + *host_off, v.data(), bytes);
        HIPCHECK(hipMemcpyAsync((uint8_t*)dev.p + *host_off, (uint8_t*)*host + *host_off, bytes,
                                hipMemcpyHostToDevice, st));
        const uint32_t grid = (uint32_t)((blocks + 7) / 8 * 8);
        const OpMember* d = (const OpMember*)((uint8_t*)dev.p + *host_off);
        *host_off += (bytes + 255) & ~(size_t)255;
        const bool stream = op_stream(edges);
#define VH_OPINION(T, S) \
    hipLaunchKernelGGL((k_opinion_multi<T, S>), dim3(grid), dim3(256), 0, st, d, (uint32_t)v.size(), (uint32_t)blocks)
        if (k == 0 && stream) VH_OPINION(double, true);
        else if (k == 0) VH_OPINION(double, false);
        else if (stream) VH_OPINION(float, true);
        else VH_OPINION(float, false);
#undef VH_OPINION
        HIPCHECK(hipGetLastError());
        v.clear();
    }
    return VH_OK;
}

int launch_diffuse_stencil(Sim& s, int t, int et, uint32_t field) {
    AgentStore& A = s.a[t];
    const StencilSpec& sp = s.e[et].sspec;
    uint64_t ncells = 1;
    for (uint32_t d = 0; d < sp.ndims; d++) ncells *= (uint64_t)sp.dims[d];
    if (!A.nslots) return VH_OK;
    // rows of 8-cell groups: one-byte records, every slot a cell, a buffer with
    // the 4 bytes behind the cells that ld8 may read (ensure_slots leaves 8),
    // rows of at least 16 cells (every 8-cell window lies in its row), offsets
    // of at most 7 cells along dimension 0 (one wrap, one partial group) and of
    // at most the extent along the others (one wrap), and at most 128000 rows:
    // 17 500 blocks in y, of the grid's 65 535, which more than 479 000 rows
    // would pass (between the two, both kernels are possible and only the one
    // that works cell by cell is used); the rest takes that kernel
    const uint64_t nx = (uint64_t)sp.dims[0], nrows = ncells / nx;
    bool rows = A.bytes == 1 && field == 0 && sp.first_nr == 1 && ncells == A.nslots && ncells <= 0x7FFFFFFFull &&
                A.state[A.rd].cap >= ncells + 4 && nx >= 16 && nrows <= 128000;
    RowSpec rsp;
    rsp.periodic = sp.periodic;
    for (uint32_t d = 0; d < 4; d++) rsp.dims[d] = d < sp.ndims ? (int32_t)sp.dims[d] : 1;
    memset(rsp.off, 0, sizeof rsp.off);
    for (uint32_t k = 0; k < sp.nst && rows; k++) {
        rows = std::abs((int)sp.off[k][0]) <= 7;
        for (uint32_t d = 1; d < 4; d++) rows = rows && std::abs((int)sp.off[k][d]) <= rsp.dims[d];
        memcpy(&rsp.off[k], sp.off[k], 4);
    }
    rsp.nst = (sp.nst + ROW_U - 1) / ROW_U * ROW_U;
    if (rows) {
        // the blocks of 64 groups by 8 rows, then those of the end groups
        const unsigned gx = grid_for((nx + 7) / 8, 64), gy = grid_for(nrows, 4 * ROW_R);
        const unsigned ey = grid_for(3 * nrows, 256 * gx);
        hipLaunchKernelGGL(k_diffuse_rows, dim3(gx, gy + ey), dim3(256), 0, s.stream, rsp,
                           (const uint8_t*)A.rstate(), (uint8_t*)A.wstate(), (uint32_t)nrows, gy);
        HIPCHECK(hipGetLastError());
        return VH_OK;
    }
    hipLaunchKernelGGL(k_diffuse_stencil, dim3(grid_for(A.nslots, 256)), dim3(256), 0, s.stream, sp,
                       (const uint8_t*)A.rstate(), (uint8_t*)A.wstate(), A.nslots, ncells, A.bytes, field);
    HIPCHECK(hipGetLastError());
    return VH_OK;
}

int stencil_csr(Sim& s, EdgeStore& E, uint64_t rowbase, uint64_t rows) {
    const StencilSpec& sp = E.sspec;
    hipStream_t st = s.stream;
    uint64_t ncells = 1;
    for (uint32_t d = 0; d < sp.ndims; d++) ncells *= (uint64_t)sp.dims[d];
    uint32_t* deg = (uint32_t*)s.scratch.take(rows * 4 + 8);
    if (!deg) return set_error(VH_ERR_OOM, "scratch");
    fill_u32(deg, 0, rows, st);
    hipLaunchKernelGGL(k_stencil_degree, dim3(grid_for(ncells, 256)), dim3(256), 0, st, sp, ncells, rowbase, deg);
    RC(E.off.ensure((rows + 1) * 4 + 8, st));
    if (scan_excl_u32(deg, E.off.as<uint32_t>(), rows, s.scratch, st)) return set_error(VH_ERR_DEVICE, "scan");
    HIPCHECK(hipMemcpyAsync(s.d_stats.p, E.off.as<uint32_t>() + rows, 4, hipMemcpyDeviceToDevice, st));
    RC(readback(s, 1));
    uint64_t ne = (uint32_t)s.h_stats[0];
    RC(E.src.ensure(ne * (E.src64 ? 8 : 4) + 8, st));
    if (E.bytes) RC(E.st.ensure(ne * E.bytes + 8, st));
    hipLaunchKernelGGL(k_stencil_fill, dim3(grid_for(ncells, 256)), dim3(256), 0, st, sp, ncells, rowbase,
                       E.off.as<uint32_t>(), E.src.p, (uint32_t)E.src64, E.st.as<uint8_t>(), E.bytes);
    HIPCHECK(hipGetLastError());
    E.nedges = ne;
    return VH_OK;
}

constexpr uint32_t CONTACT_FILTER = 163840;
static std::atomic<uint32_t> g_contact_filter{CONTACT_FILTER};   // (less in tests)
void set_contact_filter(uint32_t bytes) { g_contact_filter = bytes && bytes < CONTACT_FILTER ? bytes : CONTACT_FILTER; }

// One apply! of the contact model: flags, infections, health update with the
// kept partners as masks (or logged), one readback (deaths, contacts), newborns
// and deaths on the reuse stack, then the contact CSR rebuilt in place (its
// previous entries were last read by k_contact_infect). Deaths of this step
// are returned for the edge filtering of other edge types.
int contact_apply(Sim& s, int t, int et, const vh_contact_params& p, uint64_t step, uint64_t* ndeaths) {
    RC(check_model_layout(s, t, et, 8, 0, "contact"));
    AgentStore& A = s.a[t];
    EdgeStore& E = s.e[et];
    hipStream_t st = s.stream;
    const uint64_t n = A.nslots;
    const uint32_t C = p.n_contacts;
    *ndeaths = 0;
    if (n >= 0xFFFFFFFFull) return set_error(VH_ERR_CAPACITY, "contact: too many slots");
    if ((uint64_t)n * C >= 0xFFFFFFFFull) return set_error(VH_ERR_CAPACITY, "contact: too many contacts");
    const uint64_t nw = (n + 63) / 64, nblk = (n + 255) / 256;
    // up to 32 contacts: a mask per slot and the partners drawn again; more:
    // a log. The filter takes the smallest groups whose bits fit a CU's LDS;
    // groups of more than 32 slots would nearly all be marked
    const bool masked = C <= 32;
    ContactBits B;
    B.nwords = nw;
    B.fshift = 0;
    B.filt = nullptr;
    while ((nblk * 32) >> B.fshift > g_contact_filter) B.fshift++;
    const uint32_t fwords = masked && n && B.fshift <= 5 ? (uint32_t)((((nblk * 32) >> B.fshift) + 15) / 16 * 4) : 0u;
    B.sp = (uint64_t*)s.scratch.take(nw * 8 + 8);
    B.dead = (uint64_t*)s.scratch.take(nw * 8 + 8);
    B.inf = (uint64_t*)s.scratch.take(nw * 8 + 8);
    B.sus = (uint64_t*)s.scratch.take(nw * 8 + 8);
    B.cnt = (uint32_t*)s.scratch.take(2 * nw * 4 + 8);
    if (fwords) B.filt = (uint8_t*)s.scratch.take((uint64_t)fwords * 4 + 64);
    uint32_t* dpos = (uint32_t*)s.scratch.take((2 * nw + 1) * 4 + 8);
    uint2* masks = masked ? (uint2*)s.scratch.take(n * 8 + 8) : nullptr;
    uint32_t* kept = masked ? nullptr : (uint32_t*)s.scratch.take(n * 4 + 8);
    uint32_t* kpos = masked ? nullptr : (uint32_t*)s.scratch.take((n + 1) * 4 + 8);
    uint32_t* log = masked ? nullptr : (uint32_t*)s.scratch.take(n * C * 4 + 8);
    if (!B.sp || !B.dead || !B.inf || !B.sus || !B.cnt || (fwords && !B.filt) || !dpos ||
        (masked ? !masks : !kept || !kpos || !log))
        return set_error(VH_ERR_OOM, "scratch");
    uint64_t nd = 0, ne = 0;
    if (n) {
        hipLaunchKernelGGL(k_contact_flags, dim3((unsigned)nblk), dim3(256), 0, st, (const uint64_t*)A.rstate(),
                           A.died.as<uint8_t>(), n, (uint32_t)t, p, step, B);
        hipLaunchKernelGGL(k_contact_infect, dim3(grid_for(nw, INF_W)), dim3(256), 0, st, E.off.as<uint32_t>(),
                           E.src.as<uint32_t>(), (const uint64_t*)A.rstate(), E.rows ? E.nrows[t] : 0ull, E.rowbase[t],
                           (uint32_t)t, p, step, B);
        const uint32_t* total;   // the contacts kept (less the deaths when masked)
        if (masked) {
            // blocks of 1024 when that leaves every CU one, as many per CU as
            // their filters fit
            const uint32_t cus = device_cus(), fb = fwords * 4;
            const bool big = n >= 1024ull * cus || !fwords;
            const uint32_t bs = big ? 1024u : 256u, fit = std::max(1u, std::min(2048u / bs, fb ? CONTACT_FILTER / fb : 32u));
            const dim3 g((unsigned)std::min<uint64_t>((n + bs - 1) / bs, (uint64_t)cus * fit));
            auto launch = [&](auto kernel) {
                hipLaunchKernelGGL(kernel, g, dim3(bs), fb, st, (const uint64_t*)A.rstate(), (uint64_t*)A.wstate(),
                                   A.died_now.as<uint8_t>(), (uint32_t)n, (uint32_t)t, p, step, B, fwords, masks);
            };
            if (!fwords) launch(k_contact_main<1024, false>);   // (too many slots for a filter)
            else if (big) launch(k_contact_main<1024, true>);
            else launch(k_contact_main<256, true>);
            HIPCHECK(hipGetLastError());
            // deaths and contacts numbered in one scan (its differences hold
            // modulo 2^32)
            if (scan_excl_u32(B.cnt, dpos, 2 * nw, s.scratch, st)) return set_error(VH_ERR_DEVICE, "scan");
            total = dpos + 2 * nw;
        } else {
            if (scan_excl_u32(B.cnt, dpos, nw, s.scratch, st)) return set_error(VH_ERR_DEVICE, "scan");
            hipLaunchKernelGGL(k_contact_main_log, dim3((unsigned)nblk), dim3(256), 0, st, (const uint64_t*)A.rstate(),
                               (uint64_t*)A.wstate(), A.died_now.as<uint8_t>(), (uint32_t)n, (uint32_t)t, p, step, B, kept,
                               log);
            HIPCHECK(hipGetLastError());
            if (scan_excl_u32(kept, kpos, n, s.scratch, st)) return set_error(VH_ERR_DEVICE, "scan");
            total = kpos + n;
        }
        HIPCHECK(hipMemcpyAsync((uint32_t*)s.d_stats.p, dpos + nw, 4, hipMemcpyDeviceToDevice, st));
        HIPCHECK(hipMemcpyAsync((uint32_t*)s.d_stats.p + 1, total, 4, hipMemcpyDeviceToDevice, st));
        RC(readback(s, 1));
        nd = ((const uint32_t*)s.h_stats)[0];
        ne = ((const uint32_t*)s.h_stats)[1];
        if (masked) ne = (uint32_t)(ne - nd);
    }
    if (nd) {
        uint64_t consumed = std::min<uint64_t>(nd, A.nreuse);
        uint64_t fresh = nd - consumed;
        if (fresh) {
            RC(ensure_slots(s, t, A.nextid - 1 + fresh));
            if (A.nextid - 1 + fresh > n)
                fill_u8(A.died_now.as<uint8_t>() + n, 0, A.nextid - 1 + fresh - n, st);
        }
        hipLaunchKernelGGL(k_contact_births, dim3(grid_for(8 * nw, 256)), dim3(256), 0, st, (uint32_t)t, p, step, B, dpos,
                           A.reuse.as<uint32_t>(), A.nreuse, A.nextid, (uint64_t*)A.wstate(), A.died.as<uint8_t>());
        A.nreuse -= consumed;
        A.nextid += fresh;
        RC(A.reuse.ensure((A.nreuse + nd) * 4 + 8, st, A.nreuse * 4));
        hipLaunchKernelGGL(k_contact_deaths, dim3(grid_for(8 * nw, 256)), dim3(256), 0, st, B, dpos,
                           A.reuse.as<uint32_t>(), A.nreuse, A.died.as<uint8_t>());
        A.nreuse += nd;
        HIPCHECK(hipGetLastError());
    }
    // rows = caller slots; rows of dead callers and of newborns are empty
    uint64_t rows = std::max(n, A.nextid - 1);
    RC(edge_room(E, (rows + 1) * 4 + 8, ne * 4 + 8, 0, st));
    if (!n) fill_u32(E.off.as<uint32_t>(), 0, 1, st);
    else if (masked)
        hipLaunchKernelGGL(k_contact_edges, dim3((unsigned)nblk), dim3(256), 256 * C * 4, st, (uint32_t)n, (uint32_t)t,
                           p, step, B, masks, dpos, E.off.as<uint32_t>(), E.src.as<uint32_t>());
    else
        hipLaunchKernelGGL(k_contact_edges_log, dim3((unsigned)nblk), dim3(256), 0, st, n, C, kept, log, kpos,
                           E.off.as<uint32_t>(), E.src.as<uint32_t>());
    if (rows > n)
        hipLaunchKernelGGL(k_contact_extend, dim3(grid_for(rows - n, 256)), dim3(256), 0, st,
                           E.off.as<uint32_t>(), n, rows);
    HIPCHECK(hipGetLastError());
    for (int u = 0; u <= VH_MAXA; u++) {
        E.rowbase[u] = 0;
        E.nrows[u] = 0;
    }
    E.nrows[t] = rows;
    E.rows = rows;
    E.nedges = ne;
    E.src64 = false;
    E.src_type = (uint32_t)t;
    E.version++;
    *ndeaths = nd;
    return VH_OK;
}

}  // namespace vh
