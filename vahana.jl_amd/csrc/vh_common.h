// vh_common.h — shared device/host definitions of the MI355X transition backend.
//
// The public device API (include/vahana_device.h: device views, accessors,
// codec, RNG) and what only the library's model bodies use.
#pragma once

#include "../../include/vahana_device.h"

// Whether some in-edge k in [b, e) has u01(vh_hash_fin(pre, k - b + 1)) < p
// (pt = vh_u01_below(p)) and an infected source (infected(k)). The answer
// does not depend on the order of the in-edges: the draws of up to 32
// in-edges come first, ALU work only, then the sources of those below p, two
// at a time. Asked draw by draw, every group of four draws waited for the
// lookups of some lane of the wave, one after the other: the infections of
// the 10^7-agent contact step took 162 us so, 68 us now.
template <class F>
__host__ __device__ __forceinline__ bool vh_any_infecting(uint64_t pre, uint64_t pt, uint32_t b, uint32_t e,
                                                          F infected) {
    for (uint32_t k = b; k < e; k = vh_row_next(k, e, 32)) {
        const uint32_t cnt = e - k < 32u ? e - k : 32u;
        uint32_t m = 0;   // bit q: the draw of in-edge k + q is below p
        for (uint32_t q = 0; q < cnt; q += 4) {
            const uint64_t c = k - b + q + 1;
            const bool d0 = (vh_hash_fin(pre, c) >> 11) < pt, d1 = (vh_hash_fin(pre, c + 1) >> 11) < pt;
            const bool d2 = (vh_hash_fin(pre, c + 2) >> 11) < pt, d3 = (vh_hash_fin(pre, c + 3) >> 11) < pt;
            m |= ((d0 ? 1u : 0u) | (d1 ? 2u : 0u) | (d2 ? 4u : 0u) | (d3 ? 8u : 0u)) << q;
        }
        m &= cnt == 32u ? ~0u : (1u << cnt) - 1u;   // (draws past the row)
        while (m) {
            const uint32_t q0 = (uint32_t)__builtin_ctz(m);
            m &= m - 1u;
            const uint32_t q1 = m ? (uint32_t)__builtin_ctz(m) : q0;
            m &= m ? m - 1u : 0u;
            const bool i0 = infected(k + q0), i1 = infected(k + q1);
            if (i0 | i1) return true;
        }
    }
    return false;
}
// The in-edges k = b + l, b + l + 64, ... of row [b, e) that lane l of a wave
// takes, in order: four(k) for k, k + 64, k + 128 and k + 192, then one(k).
template <class F4, class F1>
__host__ __device__ __forceinline__ void vh_lane_edges(uint32_t b, uint32_t e, uint32_t lane, F4 four, F1 one) {
    const uint32_t d = e - b;
    uint32_t t = lane;
    for (; t < d && d - t > 192u; t = vh_row_next(t, d, 256)) four(b + t);
    for (; t < d; t = vh_row_next(t, d, 64)) one(b + t);
}
// The exposure of a wave's infected agents (every lane of the wave calls; inf:
// the lane's agent i is to be marked from): the bit of each of their
// out-neighbours is set in `bits`. Four agents at a time, 16 lanes each: the
// few infected of a wave have their out-edges in flight together, where a lane
// of its own walks them one load and one atomic after the other.
__device__ __forceinline__ void vh_expose_wave(bool inf, uint64_t i, const uint32_t* __restrict__ out_off,
                                               const uint32_t* __restrict__ out_dst, uint32_t* __restrict__ bits) {
    uint64_t m = __ballot(inf);
    if (!m) return;
    const uint32_t lane = threadIdx.x & 63u, g = lane >> 4, l = lane & 15u;
    uint32_t b = 0, n = 0;
    if (inf) {
        b = out_off[i];
        const uint32_t e = out_off[i + 1];
        n = e > b ? e - b : 0u;   // (sources past the agents leave the offsets in no order: no walk then)
    }
    while (m) {
        uint64_t t = m;   // its lowest bit: the agent of lane group g
        for (uint32_t q = 0; q < g; q++) t &= t ? t - 1ull : 0ull;
        const int who = t ? (int)__builtin_ctzll(t) : 0;
        const uint32_t bb = (uint32_t)__shfl((int)b, who, 64), d = (uint32_t)__shfl((int)n, who, 64);
        if (t)
            for (uint32_t k = l; k < d; k = vh_row_next(k, d, 16)) {
                const uint32_t v = out_dst[bb + k];
                atomicOr(bits + (v >> 5), 1u << (v & 31u));
            }
        for (uint32_t q = 0; q < 4; q++) m &= m ? m - 1ull : 0ull;
    }
}
// stream keys of the model bodies (the `c` word of vh_hash)
#define VH_KEY_RECOVER (1ull << 40)
#define VH_KEY_DEATH   (2ull << 40)
#define VH_KEY_BIRTH   (3ull << 40)
#define VH_KEY_PARTNER (4ull << 40)
#define VH_KEY_INIT    (5ull << 40)
#define VH_KEY_WEIGHT  (6ull << 40)
#define VH_KEY_OPINION (7ull << 40)
#define VH_KEY_SUSC    (8ull << 40)

