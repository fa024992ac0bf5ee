// vh_prims.hip — device-wide scan, stable LSD radix sort, fills and gathers
// for gfx950 (wave64).
#include <atomic>

#include "vh_prims.h"

#include <algorithm>

namespace vh {

// ------------------------------------------------------------------ arena
// every device allocation of the library; a test hook makes some fail: `after`
// (high word) go through, then n (low word) fail
static std::atomic<uint64_t> g_fail_allocs{0};
hipError_t device_alloc(void** p, size_t bytes) {
    uint64_t k = g_fail_allocs.load();
    while (k & 0xFFFFFFFFull) {
        const bool ok = k >> 32 != 0;
        if (!g_fail_allocs.compare_exchange_weak(k, ok ? k - (1ull << 32) : k - 1)) continue;
        if (ok) break;
        return hipErrorOutOfMemory;
    }
    return hipMalloc(p, bytes);
}
void fail_next_allocs(uint32_t n, uint32_t after) { g_fail_allocs.store((uint64_t)after << 32 | n); }

void* Scratch::take(size_t bytes) {
    bytes = (bytes + 255) & ~(size_t)255;
    if (bytes == 0) bytes = 256;
    if (used + bytes <= cap) {
        void* r = (char*)main + used;
        used += bytes;
        return r;
    }
    if (xb && xused + bytes <= xcap) {
        void* r = xb + xused;
        xused += bytes;
        return r;
    }
    if (nextra >= 64) return nullptr;
    void* p = nullptr;
    if (device_alloc(&p, bytes) != hipSuccess) return nullptr;
    extra[nextra++] = p;
    spilled += bytes;
    return p;
}
int Scratch::room(size_t bytes) {
    bytes = (bytes + 255) & ~(size_t)255;
    if (used + bytes <= cap || (xb && xused + bytes <= xcap)) return 0;
    if (nextra >= 64) return -3;
    void* p = nullptr;
    if (device_alloc(&p, bytes) != hipSuccess) return -3;
    extra[nextra++] = p;
    spilled += bytes;
    xb = (char*)p;
    xcap = bytes;
    xused = 0;
    return 0;
}
void Scratch::reset(hipStream_t st) {
    xb = nullptr;
    xcap = xused = 0;
    if (shrink) {
        shrink = false;
        if (bytes_held() > ((size_t)1 << 30)) {
            hipStreamSynchronize(st);
            release();
            return;
        }
    }
    if (nextra) {
        // fold the spill into one main block sized for the whole round
        size_t need = used + spilled;
        hipStreamSynchronize(st);
        for (int i = 0; i < nextra; i++) hipFree(extra[i]);
        nextra = 0;
        spilled = 0;
        if (main) hipFree(main);
        main = nullptr;
        cap = 0;
        size_t ncap = need + need / 4 + (1 << 20);
        if (device_alloc(&main, ncap) == hipSuccess) cap = ncap;
    }
    used = 0;
}
int Scratch::reserve(size_t bytes, hipStream_t st) {
    if (used || nextra || cap >= bytes) return 0;
    hipStreamSynchronize(st);
    if (main) hipFree(main);
    main = nullptr;
    cap = 0;
    if (device_alloc(&main, bytes) != hipSuccess) return -3;
    cap = bytes;
    return 0;
}
void Scratch::release() {
    xb = nullptr;
    xcap = xused = 0;
    for (int i = 0; i < nextra; i++) hipFree(extra[i]);
    nextra = 0;
    spilled = 0;
    if (main) hipFree(main);
    main = nullptr;
    cap = used = 0;
}

// ------------------------------------------------------------------ scan
constexpr int SB = 256;           // threads per block
constexpr int SI = 8;             // items per thread
constexpr int STILE = SB * SI;    // 2048 items per block

template <class T>
__device__ __forceinline__ T wave_incl_scan(T x) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        T y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    return x;
}

// exclusive block scan of one value per thread; *total gets the block sum
template <class T>
__device__ __forceinline__ T block_excl_scan(T v, T* lds, T* total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    T x = wave_incl_scan(v);
    if (lane == 63) lds[w] = x;
    __syncthreads();
    T pre = 0, tot = 0;
    for (int i = 0; i < nw; i++) {
        T s = lds[i];
        if (i < w) pre += s;
        tot += s;
    }
    __syncthreads();
    *total = tot;
    return pre + x - v;
}

template <class IT, class OT>
__global__ __launch_bounds__(SB) void k_scan_reduce(const IT* __restrict__ in, uint64_t n,
                                                    OT* __restrict__ bsum) {
    __shared__ OT lds[SB / 64];
    uint64_t base = (uint64_t)blockIdx.x * STILE + (uint64_t)threadIdx.x * SI;
    OT s = 0;
#pragma unroll
    for (int i = 0; i < SI; i++)
        if (base + i < n) s += (OT)in[base + i];
    OT tot;
    block_excl_scan<OT>(s, lds, &tot);
    if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}

// exclusive scan of `in` into out[0..n]; boff[b] is the offset of block b
// (nullptr: single block), out[n] receives the total from the last block
template <class IT, class OT>
__global__ __launch_bounds__(SB) void k_scan_down(const IT* __restrict__ in, OT* __restrict__ out,
                                                  uint64_t n, const OT* __restrict__ boff) {
    __shared__ OT lds[SB / 64];
    uint64_t base = (uint64_t)blockIdx.x * STILE + (uint64_t)threadIdx.x * SI;
    OT v[SI];
    OT s = 0;
#pragma unroll
    for (int i = 0; i < SI; i++) {
        v[i] = (base + i < n) ? (OT)in[base + i] : (OT)0;
        s += v[i];
    }
    OT tot;
    OT pre = block_excl_scan<OT>(s, lds, &tot);
    OT off = boff ? boff[blockIdx.x] : (OT)0;
    OT run = off + pre;
#pragma unroll
    for (int i = 0; i < SI; i++) {
        if (base + i < n) out[base + i] = run;
        run += v[i];
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) out[n] = off + tot;
}

template <class IT, class OT>
static int scan_impl(const IT* in, OT* out, uint64_t n, Scratch& s, hipStream_t st) {
    uint64_t nb = (n + STILE - 1) / STILE;
    if (nb == 0) nb = 1;
    if (nb == 1) {
        hipLaunchKernelGGL((k_scan_down<IT, OT>), dim3(1), dim3(SB), 0, st, in, out, n,
                           (const OT*)nullptr);
        return hipGetLastError() == hipSuccess ? 0 : -1;
    }
    OT* bsum = (OT*)s.take(nb * sizeof(OT));
    OT* boff = (OT*)s.take((nb + 1) * sizeof(OT));
    if (!bsum || !boff) return -3;
    hipLaunchKernelGGL((k_scan_reduce<IT, OT>), dim3((unsigned)nb), dim3(SB), 0, st, in, n, bsum);
    int r = scan_impl<OT, OT>(bsum, boff, nb, s, st);
    if (r) return r;
    hipLaunchKernelGGL((k_scan_down<IT, OT>), dim3((unsigned)nb), dim3(SB), 0, st, in, out, n,
                       (const OT*)boff);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int scan_excl_u32(const uint32_t* in, uint32_t* out, uint64_t n, Scratch& s, hipStream_t st) {
    return scan_impl<uint32_t, uint32_t>(in, out, n, s, st);
}
int scan_excl_u64(const uint32_t* in, uint64_t* out, uint64_t n, Scratch& s, hipStream_t st) {
    return scan_impl<uint32_t, uint64_t>(in, out, n, s, st);
}

// ------------------------------------------------------------------ radix sort
// Digits of DB bits, tiles of 512 threads x RI items.  Tile element e of wave
// w is tile_base + w * 64 RI + i * 64 + lane (i < RI), so each wave walks its
// contiguous eighth in index order; ranks inside an item row come from a
// ballot match over the digit's bits and the wave's count of the digit so
// far, which keeps the sort stable.
//
// The scatter puts the tile in digit order in LDS first and writes it from
// there, so that the elements of a digit leave as one run: written straight
// from the ranks, a wave's 64 elements went to as many lines, and the lines of
// all tiles at work (2 x 256 each) were evicted half written (a pass over 10^8
// pairs: 1416 us, so 558; over 10^6: 31, so 21).
constexpr int RB = 512;
constexpr int RW = RB / 64;
constexpr uint64_t RADIX_LARGE = 4u << 20;

template <int DB, int RI>
__global__ __launch_bounds__(RB) void k_radix_hist(const uint32_t* __restrict__ keys, uint64_t n,
                                                   uint32_t shift, uint32_t ntiles,
                                                   uint32_t* __restrict__ hist) {
    constexpr uint32_t NB = 1u << DB;
    __shared__ uint32_t h[NB];
    for (uint32_t d = threadIdx.x; d < NB; d += RB) h[d] = 0;
    __syncthreads();
    const uint64_t base = (uint64_t)blockIdx.x * (RB * RI);
    if (n - base >= RB * RI) {
        const uint4* k4 = (const uint4*)(keys + base);   // (the buffers start at multiples of 256 bytes)
#pragma unroll
        for (int i = 0; i < RI / 4; i++) {
            const uint4 k = k4[i * RB + threadIdx.x];
            atomicAdd(&h[(k.x >> shift) & (NB - 1)], 1u);
            atomicAdd(&h[(k.y >> shift) & (NB - 1)], 1u);
            atomicAdd(&h[(k.z >> shift) & (NB - 1)], 1u);
            atomicAdd(&h[(k.w >> shift) & (NB - 1)], 1u);
        }
    } else {
        for (uint64_t e = base + threadIdx.x; e < n; e += RB) atomicAdd(&h[(keys[e] >> shift) & (NB - 1)], 1u);
    }
    __syncthreads();
    for (uint32_t d = threadIdx.x; d < NB; d += RB) hist[(uint64_t)d * ntiles + blockIdx.x] = h[d];
}

template <int DB, int RI>
__global__ __launch_bounds__(RB) void k_radix_scatter(const uint32_t* __restrict__ kin,
                                                      const uint32_t* __restrict__ vin,
                                                      uint32_t* __restrict__ kout,
                                                      uint32_t* __restrict__ vout, uint64_t n,
                                                      uint32_t shift, uint32_t ntiles,
                                                      const uint32_t* __restrict__ goff) {
    constexpr uint32_t TILE = RB * RI, NB = 1u << DB;
    constexpr uint32_t PT = NB > RB ? NB / RB : 1;   // digits per thread of the tile's scan
    __shared__ uint32_t whist[RW][NB];   // the waves' digit counts, then their first places in the tile
    __shared__ uint32_t gbase[NB], wsum[RW];
    __shared__ uint32_t sk[TILE], sv[TILE];
    const uint32_t tid = threadIdx.x;
    const int lane = tid & 63, w = tid >> 6;
    for (uint32_t d = tid; d < RW * NB; d += RB) (&whist[0][0])[d] = 0;
    __syncthreads();
    const uint64_t tbase = (uint64_t)blockIdx.x * TILE, wbase = tbase + (uint64_t)w * (64 * RI);
    const uint32_t cnt = n - tbase < TILE ? (uint32_t)(n - tbase) : TILE;
    const uint64_t lt = (1ull << lane) - 1ull;
    uint32_t k[RI], v[RI], rank[RI];
#pragma unroll
    for (int i = 0; i < RI; i++) {
        const uint64_t e = wbase + (uint64_t)i * 64 + lane;
        k[i] = e < n ? kin[e] : 0u;
        v[i] = vin ? (e < n ? vin[e] : 0u) : (uint32_t)e;
    }
#pragma unroll
    for (int i = 0; i < RI; i++) {
        const bool valid = wbase + (uint64_t)i * 64 + lane < n;
        const uint32_t d = (k[i] >> shift) & (NB - 1);
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < DB; b++) {
            const uint64_t bal = __ballot((d >> b) & 1u);
            peers &= ((d >> b) & 1u) ? bal : ~bal;
        }
        const uint32_t r = (uint32_t)__popcll(peers & lt);
        rank[i] = valid ? whist[w][d] + r : 0u;
        __builtin_amdgcn_wave_barrier();
        if (valid && r == 0) whist[w][d] += (uint32_t)__popcll(peers);
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    // digit d: its place in the tile and the waves' places behind it
    uint32_t c[PT], sum = 0;
#pragma unroll
    for (uint32_t q = 0; q < PT; q++) {
        const uint32_t d = tid * PT + q;
        c[q] = 0;
        if (d < NB)
#pragma unroll
            for (int x = 0; x < RW; x++) {
                const uint32_t t = whist[x][d];
                whist[x][d] = c[q];
                c[q] += t;
            }
        sum += c[q];
    }
    uint32_t start = wave_incl_scan(sum);
    if (lane == 63) wsum[w] = start;
    __syncthreads();
    start -= sum;
    for (int q = 0; q < w; q++) start += wsum[q];
#pragma unroll
    for (uint32_t q = 0; q < PT; q++) {
        const uint32_t d = tid * PT + q;
        if (d < NB) {
#pragma unroll
            for (int x = 0; x < RW; x++) whist[x][d] += start;
            gbase[d] = goff[(uint64_t)d * ntiles + blockIdx.x] - start;
        }
        start += c[q];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < RI; i++)
        if (wbase + (uint64_t)i * 64 + lane < n) {
            const uint32_t p = whist[w][(k[i] >> shift) & (NB - 1)] + rank[i];
            sk[p] = k[i];
            sv[p] = v[i];
        }
    __syncthreads();
    for (uint32_t p = tid; p < cnt; p += RB) {
        const uint32_t key = sk[p], o = gbase[(key >> shift) & (NB - 1)] + p;
        kout[o] = key;
        vout[o] = sv[p];
    }
}

template <int DB, int RI>
static int radix_sort_impl(uint32_t** keys, uint32_t** vals, uint32_t* kalt, uint32_t* valt, uint64_t n,
                           uint32_t bits, bool iota_vals, Scratch& s, hipStream_t st) {
    const uint32_t ntiles = (uint32_t)((n + RB * RI - 1) / (RB * RI));
    const uint64_t nh = (uint64_t)ntiles << DB;
    uint32_t* hist = (uint32_t*)s.take(nh * sizeof(uint32_t));
    uint32_t* goff = (uint32_t*)s.take((nh + 1) * sizeof(uint32_t));
    if (!hist || !goff) return -3;
    uint32_t *kin = *keys, *vin = *vals, *kout = kalt, *vout = valt;
    bool first = true;
    for (uint32_t shift = 0; shift < bits; shift += DB) {
        hipLaunchKernelGGL((k_radix_hist<DB, RI>), dim3(ntiles), dim3(RB), 0, st, kin, n, shift, ntiles, hist);
        int r = scan_excl_u32(hist, goff, nh, s, st);
        if (r) return r;
        hipLaunchKernelGGL((k_radix_scatter<DB, RI>), dim3(ntiles), dim3(RB), 0, st, kin,
                           (first && iota_vals) ? (const uint32_t*)nullptr : vin, kout, vout, n,
                           shift, ntiles, goff);
        first = false;
        std::swap(kin, kout);
        std::swap(vin, vout);
    }
    *keys = kin;
    *vals = vin;
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
// Below RADIX_LARGE pairs a pass is launches and latency: digits of 9 or 10
// bits where they save one (17..20 bits of rows: two passes for three; 3.2 10^6
// pairs, 18 bits: 88 us, three passes of 8 bits 122), with tiles of 4096, as
// their counts per tile are two or four times as many; else tiles of 2048.
// From there on 8-bit digits and tiles of 8192 (10^7 pairs, 20 bits: scatters
// of 3 x 49 us, with 10-bit digits 2 x 76).
int radix_sort_pairs(uint32_t** keys, uint32_t** vals, uint32_t* kalt, uint32_t* valt, uint64_t n,
                     uint32_t bits, bool iota_vals, Scratch& s, hipStream_t st) {
    if (n == 0) return 0;
    if (bits == 0) bits = 1;
    const uint32_t passes = (bits + 9) / 10;
#define VH_RADIX(DB, RI) radix_sort_impl<DB, RI>(keys, vals, kalt, valt, n, bits, iota_vals, s, st)
    if (n >= RADIX_LARGE) return VH_RADIX(8, 16);
    if ((bits + 7) / 8 == passes) return VH_RADIX(8, 4);
    return bits <= 9 * passes ? VH_RADIX(9, 8) : VH_RADIX(10, 8);
#undef VH_RADIX
}

// ------------------------------------------------------------------ helpers
__global__ void k_fill_u8(uint8_t* p, uint8_t v, uint64_t n) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}
__global__ void k_fill_u32(uint32_t* p, uint32_t v, uint64_t n) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}
__global__ void k_iota_u32(uint32_t* p, uint64_t n) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = (uint32_t)i;
}
void fill_u8(uint8_t* p, uint8_t v, uint64_t n, hipStream_t st) {
    if (n) hipLaunchKernelGGL(k_fill_u8, dim3(grid_for(n, 256)), dim3(256), 0, st, p, v, n);
}
void fill_u32(uint32_t* p, uint32_t v, uint64_t n, hipStream_t st) {
    if (n) hipLaunchKernelGGL(k_fill_u32, dim3(grid_for(n, 256)), dim3(256), 0, st, p, v, n);
}
void iota_u32(uint32_t* p, uint64_t n, hipStream_t st) {
    if (n) hipLaunchKernelGGL(k_iota_u32, dim3(grid_for(n, 256)), dim3(256), 0, st, p, n);
}

__global__ void k_gather_u32(uint32_t* __restrict__ dst, const uint32_t* __restrict__ src,
                             const uint32_t* __restrict__ idx, uint64_t n) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[idx[i]];
}
void gather_u32(uint32_t* dst, const uint32_t* src, const uint32_t* idx, uint64_t n, hipStream_t st) {
    if (n) hipLaunchKernelGGL(k_gather_u32, dim3(grid_for(n, 256)), dim3(256), 0, st, dst, src, idx, n);
}

__global__ void k_check_sorted(const uint32_t* __restrict__ k, uint64_t n, uint32_t* unsorted) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x + 1;
    if (i < n && k[i] < k[i - 1]) *unsorted = 1;
}
void check_sorted(const uint32_t* keys, uint64_t n, uint32_t* unsorted, hipStream_t st) {
    if (n > 1)
        hipLaunchKernelGGL(k_check_sorted, dim3(grid_for(n, 256)), dim3(256), 0, st, keys, n, unsorted);
}

}  // namespace vh
