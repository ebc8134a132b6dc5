// sph_radix.hip -- stable LSD radix sort of (voxel key, slot) pairs for gfx950 (the VOXEL
// formulation, whose keys follow the reference's wrapping semantics and may lie outside the
// grid; the NAIVE formulation's clamped keys use the counting sort of sph_cellsort.hip).
//
// Replaces the host-side sort of the voxel map (voxel_sph_strategy.py:81-89), whose
// result is the lexicographic order on (voxel_id, particle_id).  The input pairs are
// laid out in particle-id order, so a stable sort on the key alone reproduces that order.
//
// Each pass sorts on up to 8 key bits with three launches:
//   upsweep   one workgroup per tile of 512, 1024 or 2048 keys counts digits in LDS (one
//             histogram per wavefront to spread LDS atomics) and writes counts digit-major;
//   scan      one workgroup per digit turns the counts of that digit into exclusive
//             tile offsets and a digit total (few tiles: the upsweep writes tile-major and
//             each workgroup of the downsweep adds the counts up itself, without this launch);
//   downsweep each tile ranks its keys stably with wave64 ballots (the lanes holding the
//             same digit are found with one ballot per digit bit), places them in LDS in
//             digit order and writes each digit run contiguously.  On the last pass it can
//             also gather the particle state into cell order (posB/velB/pidB -> A), so
//             the separate reorder pass disappears.
#include "sph_device.h"

namespace sph {
namespace {

constexpr int RB = 8;
constexpr int RADIX = 1 << RB;   // 256 digits
constexpr int ST = 256;          // threads per workgroup, 4 wavefronts
constexpr int WAVES = ST / 64;

// Keys per thread (a tile is 256 times as many): a pass over few keys is a chain of waits, which more
// and smaller tiles shorten, until their counts and short runs of equal digits cost more than
// that.  Up to kFewTiles tiles the downsweep adds all counts up.  us per sort with the gather
// (dam break, 2 / 4 / 8 keys with the scan): 55,296 particles 45 / 52 / 66, 131,072 51 / 55 / 70,
// 262,144 60 / 59 / 71, 524,288 - / 70 / 75, 1,048,576 - / 105 / 102; 2 keys without / 8 with the
// scan: 4,096 33 / 64, 24,576 42 / 65, 49,152 51 / 66.
constexpr int kFewTiles = 96;
int keys_per_thread(int64_t n) { return n <= 196608 ? 2 : n <= 786432 ? 4 : 8; }

// Exclusive scan of one value per thread across the 256-thread workgroup.
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t* lds_wave, uint32_t* total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        uint32_t y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    if (lane == 63) lds_wave[w] = x;
    __syncthreads();
    uint32_t woff = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < WAVES; ++i) {
        uint32_t t = lds_wave[i];
        woff += i < w ? t : 0u;
        tot += t;
    }
    *total = tot;
    __syncthreads();
    return woff + x - v;
}

template <int SI, bool FEW>
__global__ __launch_bounds__(ST) void radix_upsweep(const uint32_t* __restrict__ keys, int n, int shift,
                                                     uint32_t mask, uint32_t* __restrict__ hist, int ntiles,
                                                     uint32_t* __restrict__ clear_flag) {
    __shared__ uint32_t h[WAVES][RADIX];
    // the first pass clears the out-of-grid flag that this step's gather sets (the previous
    // step's density pass, its only reader, has finished)
    if (clear_flag && blockIdx.x == 0 && threadIdx.x == 0) *clear_flag = 0u;
    for (int i = threadIdx.x; i < WAVES * RADIX; i += ST) (&h[0][0])[i] = 0;
    __syncthreads();
    const int w = threadIdx.x >> 6;
    const int64_t base = (int64_t)blockIdx.x * (ST * SI);
#pragma unroll
    for (int k = 0; k < SI; ++k) {
        int64_t idx = base + k * ST + threadIdx.x;
        if (idx < n) atomicAdd(&h[w][(keys[idx] >> shift) & mask], 1u);
    }
    __syncthreads();
    const int d = threadIdx.x;
    uint32_t s = 0;
#pragma unroll
    for (int i = 0; i < WAVES; ++i) s += h[i][d];
    hist[FEW ? (int64_t)blockIdx.x * RADIX + d : (int64_t)d * ntiles + blockIdx.x] = s;
}

__global__ __launch_bounds__(ST) void radix_scan_digits(uint32_t* __restrict__ hist, int ntiles,
                                                         uint32_t* __restrict__ digit_total) {
    __shared__ uint32_t lw[WAVES];
    uint32_t* row = hist + (int64_t)blockIdx.x * ntiles;
    uint32_t carry = 0;
    for (int base = 0; base < ntiles; base += ST) {
        const int i = base + threadIdx.x;
        uint32_t v = i < ntiles ? row[i] : 0u;
        uint32_t tot;
        uint32_t ex = block_excl_scan(v, lw, &tot);
        if (i < ntiles) row[i] = carry + ex;
        carry += tot;
    }
    if (threadIdx.x == 0) digit_total[blockIdx.x] = carry;
}

// GATHER (the last pass of the fused step): also gathers the state into cell order and, for
// the VOXEL formulation (C.formulation), reports a position outside the voxel grid in
// flags[kFlagOutOfGrid].
template <int SI, bool FEW, bool GATHER>
__global__ __launch_bounds__(ST) void radix_downsweep(const uint32_t* __restrict__ kin, const uint32_t* __restrict__ vin,
                                                       uint32_t* __restrict__ kout, uint32_t* __restrict__ vout, int n,
                                                       int shift, int bits, const uint32_t* __restrict__ hist,
                                                       const uint32_t* __restrict__ digit_total, int ntiles,
                                                       const float4* __restrict__ posB, const float4* __restrict__ velB,
                                                       const uint32_t* __restrict__ pidB, float4* __restrict__ posA,
                                                       float4* __restrict__ velA, uint32_t* __restrict__ pidA,
                                                       StepConsts C, uint32_t* __restrict__ flags) {
    constexpr int TILE = ST * SI;
    __shared__ uint32_t s_keys[TILE];
    __shared__ uint32_t s_vals[TILE];
    __shared__ uint32_t s_whist[WAVES][RADIX];
    __shared__ uint32_t s_tstart[RADIX];
    __shared__ uint32_t s_gbase[RADIX];
    __shared__ uint32_t s_lw[WAVES];

    const uint32_t mask = (1u << bits) - 1u;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int64_t base = (int64_t)blockIdx.x * TILE;

    for (int i = tid; i < WAVES * RADIX; i += ST) (&s_whist[0][0])[i] = 0;
    {
        uint32_t all = 0, before = 0;
        if constexpr (FEW) {
#pragma unroll 8
            for (int t = 0; t < ntiles; ++t) {
                const uint32_t v = hist[t * RADIX + tid];
                all += v;
                before += t < (int)blockIdx.x ? v : 0u;
            }
        } else {
            all = digit_total[tid];
            before = hist[(int64_t)tid * ntiles + blockIdx.x];
        }
        uint32_t tot;
        uint32_t ex = block_excl_scan(all, s_lw, &tot);  // synchronises: s_whist zeroed
        s_gbase[tid] = ex + before;
    }

    uint32_t key[SI], val[SI], rank[SI];
    const uint64_t lt = (1ull << lane) - 1ull;
#pragma unroll
    for (int k = 0; k < SI; ++k) {
        const int64_t idx = base + (int64_t)w * 64 * SI + k * 64 + lane;
        const bool valid = idx < n;
        key[k] = valid ? kin[idx] : 0u;
        val[k] = valid ? vin[idx] : 0u;
    }
#pragma unroll
    for (int k = 0; k < SI; ++k) {
        const int64_t idx = base + (int64_t)w * 64 * SI + k * 64 + lane;
        const bool valid = idx < n;
        const uint32_t d = (key[k] >> shift) & mask;
        uint64_t peers = __ballot(valid);
        for (int b = 0; b < bits; ++b) {
            const bool bit = (d >> b) & 1u;
            const uint64_t bal = __ballot(bit);
            peers &= bit ? bal : ~bal;
        }
        uint32_t r = 0;
        if (valid) {
            const uint32_t prefix = s_whist[w][d];
            const uint32_t below = (uint32_t)__popcll(peers & lt);
            r = prefix + below;
            if (below == 0) s_whist[w][d] = prefix + (uint32_t)__popcll(peers);
        }
        rank[k] = r;
    }
    __syncthreads();
    {
        const int d = tid;
        uint32_t run = 0;
#pragma unroll
        for (int i = 0; i < WAVES; ++i) {
            uint32_t t = s_whist[i][d];
            s_whist[i][d] = run;
            run += t;
        }
        uint32_t tot;
        s_tstart[d] = block_excl_scan(run, s_lw, &tot);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < SI; ++k) {
        const int64_t idx = base + (int64_t)w * 64 * SI + k * 64 + lane;
        if (idx < n) {
            const uint32_t d = (key[k] >> shift) & mask;
            const uint32_t p = s_tstart[d] + s_whist[w][d] + rank[k];
            s_keys[p] = key[k];
            s_vals[p] = val[k];
        }
    }
    __syncthreads();
    const int tile_n = (int)((n - base) < TILE ? (n - base) : TILE);
    // up to four keys' gathers in flight
    constexpr int GI = SI < 4 ? SI : 4;
    for (int i0 = tid; i0 < tile_n; i0 += ST * GI) {
        uint32_t vv[GI], g[GI];
#pragma unroll
        for (int u = 0; u < GI; ++u) {
            const int i = min(i0 + u * ST, tile_n - 1);
            const uint32_t kk = s_keys[i];
            const uint32_t d = (kk >> shift) & mask;
            vv[u] = s_vals[i];
            g[u] = s_gbase[d] + (uint32_t)i - s_tstart[d];
            if (i0 + u * ST < tile_n) {
                kout[g[u]] = kk;
                vout[g[u]] = vv[u];
            }
        }
        if constexpr (GATHER) {
            float4 p[GI], v[GI];
            uint32_t id[GI];
#pragma unroll
            for (int u = 0; u < GI; ++u) {
                p[u] = posB[vv[u]];
                v[u] = velB[vv[u]];
                id[u] = pidB[vv[u]];
            }
#pragma unroll
            for (int u = 0; u < GI; ++u) {
                if (i0 + u * ST >= tile_n) break;
                posA[g[u]] = p[u];
                velA[g[u]] = v[u];
                pidA[g[u]] = id[u];
                if (C.formulation == SPH_FORM_VOXEL && outside_voxel_grid(p[u].x, p[u].y, p[u].z, C))
                    flags[kFlagOutOfGrid] = 1u;
            }
        }
    }
}

// The tiles' digit counts.  tile_hist holds a tile per 2,048 keys; the counts of smaller tiles go to
// the NAIVE formulation's list words, which the sort's contexts leave alone: 1 KiB per 512 keys
// there, 4 B per particle.
uint32_t* tile_counts(const sph_ctx* c) {
    return (int64_t)c->num_tiles <= (c->n + 2047) / 2048 ? c->b.tile_hist : c->b.nn;
}

// One pass over the tiles.
template <int SI, bool FEW>
void launch_radix_pass(sph_ctx* c, int p, bool gather, const uint32_t* kin, const uint32_t* vin, uint32_t* kout,
                       uint32_t* vout, hipStream_t s) {
    const int n = (int)c->n, T = c->num_tiles, shift = c->pass_shift[p], bits = c->pass_bits[p];
    const Buffers& b = c->b;
    uint32_t* const counts = tile_counts(c);
    radix_upsweep<SI, FEW><<<T, ST, 0, s>>>(kin, n, shift, (1u << bits) - 1u, counts, T,
                                           p == 0 ? b.flags + kFlagOutOfGrid : nullptr);
    if (!FEW) radix_scan_digits<<<RADIX, ST, 0, s>>>(counts, T, b.digit_total);
    if (gather)
        radix_downsweep<SI, FEW, true><<<T, ST, 0, s>>>(kin, vin, kout, vout, n, shift, bits, counts,
                                                       b.digit_total, T, b.posB, b.velB, b.pidB, b.posA, b.velA,
                                                       b.pidA, c->sc, b.flags);
    else
        radix_downsweep<SI, FEW, false><<<T, ST, 0, s>>>(kin, vin, kout, vout, n, shift, bits, counts,
                                                        b.digit_total, T, nullptr, nullptr, nullptr, nullptr, nullptr,
                                                        nullptr, c->sc, nullptr);
}

}  // namespace

int radix_num_tiles(int64_t n) {
    const int64_t tile = (int64_t)ST * keys_per_thread(n);
    return (int)((n + tile - 1) / tile);
}

// Sorts (keyI, valI) into the radix ping-pong buffers.  When gather is set the last pass
// also writes posA/velA in sorted order; returns through c->sorted_keys/sorted_vals.
hipError_t launch_radix_sort_impl(sph_ctx* c, bool gather, hipStream_t s) {
    const uint32_t* kin = c->b.keyI;
    const uint32_t* vin = c->b.valI;
    if (c->n == 0) {
        c->sorted_keys = c->b.keyI;
        c->sorted_vals = c->b.valI;
        return hipGetLastError();
    }
    for (int p = 0; p < c->passes; ++p) {
        uint32_t* kout = c->b.keyS[p & 1];
        uint32_t* vout = c->b.valS[p & 1];
        const bool last = gather && p == c->passes - 1;
        const bool few = c->num_tiles <= kFewTiles;
        const int keys = keys_per_thread(c->n);
        const auto pass = few         ? launch_radix_pass<2, true>
                          : keys == 2 ? launch_radix_pass<2, false>
                          : keys == 4 ? launch_radix_pass<4, false>
                                      : launch_radix_pass<8, false>;
        pass(c, p, last, kin, vin, kout, vout, s);
        kin = kout;
        vin = vout;
    }
    c->sorted_keys = const_cast<uint32_t*>(kin);
    c->sorted_vals = const_cast<uint32_t*>(vin);
    return hipGetLastError();
}

}  // namespace sph
