// sph_cellsort.hip -- counting sort of the NAIVE formulation's cell keys for gfx950.
//
// The NAIVE path's keys are cell indices in [0, C) (clamped to the grid; bits 30-31 carry the
// particle's x slab in its cell), so the order the step needs -- by (cell, particle id), the
// order of the reference's stable sort of the voxel map (voxel_sph_strategy.py:81-89), or by
// (cell, slab, id) in the fused step -- is a counting sort by cell followed by that order
// within each cell.  The keys arrive in the state's current slot order (the previous step's cell
// order, see hash_particle), so neighbouring threads mostly hit the same or neighbouring
// cells.  Per step:
//   count    one thread per slot: rank = atomicAdd(&cnt[key], 1) (an arbitrary order among
//            the particles of a cell).  Between the steps of one multi-step call the previous
//            step's force pass has done this already as it wrote the keys (rank_in_cell), and
//            the sort starts at the scan
//   scan     exclusive prefix sum of cnt over all cells: tile sums (16-byte loads; a force
//            pass that counted with one lane per particle has added them up already, into
//            kTileSumCopies copies per tile), then each tile's offset is the sum of the tile
//            sums before it (added up by the tile's own workgroup when there are few tiles,
//            else by a one-workgroup scan first), then the tile is scanned; the result is
//            the cell start table cs[0..C] itself, and the tile scan resets cnt, and the
//            other array of tile sums, to zero for the next step
//   scatter  one thread per slot: tmp[cs[key] + rank] = slot
//   order    one thread per position: the particle there moves to cs[key] + (number of
//            particles of its cell with a smaller id), which is id order within the cell; the
//            sorted key is written there and either the slot (read by the separate reorder
//            pass of a staged step) or, in the fused step, the particle's gathered state.
//            With cells cut into x slabs (StepConsts::slab_shift) the fused step orders a
//            cell by (slab, id) instead, and the first particle of each cell stores the
//            offsets of its slabs in the high bits of the cell's table entry; the scan has
//            stored offset 0 there for the empty cells.  A staged step keeps the id order
//            (the reference's), and its table carries no offsets for occupied cells, which
//            the row walk then searches whole.
// The within-cell pass costs one comparison per particle of the cell, less than the density
// pass spends on the same cell.  The final order does not depend on the atomic order.
// The per-slot passes (count, scatter, order) map workgroups to slot ranges XCD by XCD as
// the density and force passes do (xcd_tile), so each XCD reads back from its own L2 the keys
// and state its force pass wrote (step 0.2245 -> 0.2226 ms on the 1M dam break).
#include <algorithm>

#include "sph_device.h"

namespace sph {
namespace {

constexpr int CT = 256;                        // threads per workgroup
constexpr int CTILE = 1 << kScanTileShift;     // cells per scan tile
constexpr int CI = CTILE / CT;                 // cells per thread in the scan
static_assert(CI == 16, "the scan's loads assume 16 cells per thread");
constexpr int CWAVES = CT / 64;
// up to this many tiles, each tile's workgroup sums the tile sums before it (at most 32
// loads per thread)
constexpr int kMergedTiles = 8192 / kTileSumCopies;

// The slab layout of the cell table (StepConsts::slab_shift .. start_mask).
struct SlabTable {
    int shift;
    int start_bits;
    int bits;
    int count_pos;
    int count_bits;
    uint32_t start_mask;
    // the fields of a cell with all its slab offsets 0 (an empty cell)
    __host__ __device__ uint32_t empty() const {
        uint32_t f = 0;
        for (int j = 1; j < (1 << shift); ++j) f |= 1u << (start_bits + bits * (j - 1));
        return f;
    }
};

// The fields of an occupied cell of count particles, b_j of them in slabs below j: the offsets of
// slabs 1 .. S - 1, each stored + 1, none if the largest does not fit; the count + 1 where it
// fits.
__device__ __forceinline__ uint32_t slab_fields(const SlabTable& T, uint32_t b1, uint32_t b2, uint32_t b3,
                                                uint32_t count) {
    const bool four = T.shift == 2;
    const uint32_t top = four ? b3 : b1;
    uint32_t fields = 0u;
    if (top + 1u <= (1u << T.bits) - 1u) {
        fields = (b1 + 1u) << T.start_bits;
        if (four) fields |= ((b2 + 1u) << (T.start_bits + T.bits)) | ((b3 + 1u) << (T.start_bits + 2 * T.bits));
    }
    if (T.count_bits > 0 && count + 1u <= (1u << T.count_bits) - 1u) fields |= (count + 1u) << T.count_pos;
    return fields;
}

constexpr uint32_t kIdMask = kCellKeyMask;  // particle ids are below 2^27

SlabTable slab_table(const StepConsts& S) {
    return SlabTable{S.slab_shift, S.start_bits, S.slab_bits, S.count_pos, S.count_bits, S.start_mask};
}

// One thread per slot; the ranks of rank_in_cell.
__global__ __launch_bounds__(CT) void cell_count_kernel(int n, const uint32_t* __restrict__ keyI,
                                                         uint32_t* __restrict__ cnt, uint32_t* __restrict__ rank) {
    const int i = xcd_tile(blockIdx.x, gridDim.x) * CT + threadIdx.x;
    const bool valid = i < n;
    const uint32_t r = rank_in_cell(valid ? keyI[i] & kCellKeyMask : 0xffffffffu, valid, cnt);
    if (valid) rank[i] = r;
}

__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t x) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    return x;
}

// Exclusive scan of one value per thread across the workgroup; *total receives the sum.
__device__ __forceinline__ uint32_t block_excl(uint32_t v, uint32_t* lw, uint32_t* total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint32_t x = wave_incl_scan(v);
    if (lane == 63) lw[w] = x;
    __syncthreads();
    uint32_t off = 0, tot = 0;
#pragma unroll
    for (int k = 0; k < CWAVES; ++k) {
        const uint32_t t = lw[k];
        off += k < w ? t : 0u;
        tot += t;
    }
    *total = tot;
    __syncthreads();
    return off + x - v;
}

constexpr int CV = CI / 4;  // 16-byte vectors per thread and tile

// Tile sums into part copy 0 (the scan that follows reads that copy only).
__global__ __launch_bounds__(CT) void cell_scan_reduce(const uint32_t* __restrict__ cnt, int m,
                                                        uint32_t* __restrict__ part) {
    __shared__ uint32_t lw[CWAVES];
    const int64_t base = (int64_t)blockIdx.x * CTILE;
    uint32_t s = 0;
    if (base + CTILE <= m) {  // base is a multiple of 4 cells: 16-byte aligned
        const uint4* c4 = reinterpret_cast<const uint4*>(cnt + base);
#pragma unroll
        for (int k = 0; k < CV; ++k) {
            const uint4 x = c4[k * CT + threadIdx.x];
            s += x.x + x.y + x.z + x.w;
        }
    } else {
        for (int k = 0; k < CI; ++k) {
            const int64_t c = base + k * CT + threadIdx.x;
            if (c < m) s += cnt[c];
        }
    }
    uint32_t tot;
    block_excl(s, lw, &tot);
    if (threadIdx.x == 0) part[blockIdx.x] = tot;
}

// One workgroup: exclusive scan of the tile sums (over their first `copies` copies) into
// copy 0, in chunks of CT with a carry.
__global__ __launch_bounds__(CT) void cell_scan_partials(uint32_t* __restrict__ part, int nparts, int copies) {
    __shared__ uint32_t lw[CWAVES];
    uint32_t carry = 0;
    for (int base = 0; base < nparts; base += CT) {
        const int i = base + threadIdx.x;
        uint32_t v = 0u;
        if (i < nparts)
            for (int k = 0; k < copies; ++k) v += part[(size_t)k * nparts + i];
        uint32_t tot;
        const uint32_t ex = block_excl(v, lw, &tot);
        if (i < nparts) part[i] = carry + ex;
        carry += tot;
    }
}

// Sum of the tile sums before tile b, over their first `copies` copies (the tile's offset
// when the tile sums were not scanned first).
__device__ __forceinline__ uint32_t tiles_before(const uint32_t* __restrict__ part, int b, int tiles, int copies,
                                                 uint32_t* lw) {
    uint32_t s = 0;
    for (int j = threadIdx.x; j < b; j += CT) {  // the copies of a tile in flight together
        uint32_t v[kTileSumCopies];
#pragma unroll
        for (int k = 0; k < kTileSumCopies; ++k) v[k] = k < copies ? part[(size_t)k * tiles + j] : 0u;
#pragma unroll
        for (int k = 0; k < kTileSumCopies; ++k) s += v[k];
    }
    uint32_t tot;
    block_excl(s, lw, &tot);
    return tot;
}

// The tile is read (and cnt cleared) with coalesced 16-byte accesses into LDS, each thread
// scans CI consecutive cells there, and cs is written back coalesced.  LDS index i is padded
// by i / 32 so that the thread-contiguous pass does not hit one bank.  The last tile also
// writes cs[m] = n.  MERGED: the first `copies` copies of part hold tile sums (all of them
// when a force pass added them up, copy 0 when cell_scan_reduce did; the offset is summed
// here); otherwise copy 0 of part holds the tiles' exclusive prefix sums.  Each workgroup also
// clears its tile's copies in next, the tile sums that the next force pass adds into.

__device__ __forceinline__ int cpad(int i) { return i + (i >> 5); }

template <bool MERGED>
__global__ __launch_bounds__(CT) void cell_scan_down(uint32_t* __restrict__ cnt, int m,
                                                      const uint32_t* __restrict__ part, uint32_t* __restrict__ next,
                                                      uint32_t* __restrict__ cs, uint32_t n, uint32_t empty,
                                                      int copies) {
    __shared__ uint32_t lw[CWAVES];
    __shared__ uint32_t tile[CTILE + CTILE / 32];
    const int64_t base = (int64_t)blockIdx.x * CTILE;
    if (threadIdx.x < kTileSumCopies) next[(size_t)threadIdx.x * gridDim.x + blockIdx.x] = 0u;
    const uint32_t offset = MERGED ? tiles_before(part, blockIdx.x, gridDim.x, copies, lw) : part[blockIdx.x];
    const bool full = base + CTILE <= m;  // base is a multiple of 4 cells: 16-byte aligned
    if (full) {
        uint4* c4 = reinterpret_cast<uint4*>(cnt + base);
#pragma unroll
        for (int k = 0; k < CV; ++k) {
            const int v = k * CT + threadIdx.x;
            const uint4 x = c4[v];
            c4[v] = make_uint4(0u, 0u, 0u, 0u);
            tile[cpad(4 * v)] = x.x;
            tile[cpad(4 * v + 1)] = x.y;
            tile[cpad(4 * v + 2)] = x.z;
            tile[cpad(4 * v + 3)] = x.w;
        }
    } else {
#pragma unroll
        for (int k = 0; k < CI; ++k) {
            const int j = k * CT + threadIdx.x;
            const int64_t c = base + j;
            uint32_t v = 0u;
            if (c < m) {
                v = cnt[c];
                cnt[c] = 0u;
            }
            tile[cpad(j)] = v;
        }
    }
    __syncthreads();
    const int j0 = threadIdx.x * CI;
    uint32_t s = 0;
#pragma unroll
    for (int k = 0; k < CI; ++k) s += tile[cpad(j0 + k)];
    uint32_t tot;
    uint32_t run = offset + block_excl(s, lw, &tot);  // synchronises
#pragma unroll
    for (int k = 0; k < CI; ++k) {
        const uint32_t v = tile[cpad(j0 + k)];
        tile[cpad(j0 + k)] = run | (v == 0u ? empty : 0u);
        run += v;
    }
    __syncthreads();
    if (full) {
        uint4* o4 = reinterpret_cast<uint4*>(cs + base);
#pragma unroll
        for (int k = 0; k < CV; ++k) {
            const int v = k * CT + threadIdx.x;
            o4[v] = make_uint4(tile[cpad(4 * v)], tile[cpad(4 * v + 1)], tile[cpad(4 * v + 2)], tile[cpad(4 * v + 3)]);
        }
    } else {
#pragma unroll
        for (int k = 0; k < CI; ++k) {
            const int j = k * CT + threadIdx.x;
            if (base + j < m) cs[base + j] = tile[cpad(j)];
        }
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) cs[m] = n;
}

__global__ __launch_bounds__(CT) void cell_scatter_kernel(int n, const uint32_t* __restrict__ keyI,
                                                           const uint32_t* __restrict__ rank,
                                                           const uint32_t* __restrict__ cs, uint32_t* __restrict__ tmp,
                                                           uint32_t start_mask) {
    const int i = xcd_tile(blockIdx.x, gridDim.x) * CT + threadIdx.x;
    if (i < n) tmp[(cs[keyI[i] & kCellKeyMask] & start_mask) + rank[i]] = (uint32_t)i;
}

template <bool GATHER>
__global__ __launch_bounds__(CT) void cell_order_kernel(int n, SlabTable T, const uint32_t* __restrict__ tmp,
                                                         const uint32_t* __restrict__ keyI, uint32_t* __restrict__ cs,
                                                         uint32_t* __restrict__ skey, uint32_t* __restrict__ sval,
                                                         const float4* __restrict__ posB,
                                                         const float4* __restrict__ velB,
                                                         const uint32_t* __restrict__ pidB, float4* __restrict__ posA,
                                                         float4* __restrict__ velA, uint32_t* __restrict__ pidA) {
    const int s = xcd_tile(blockIdx.x, gridDim.x) * CT + threadIdx.x;
    if (s >= n) return;
    const uint32_t slot = tmp[s];
    const uint32_t id = pidB[slot];
    const uint32_t kf = keyI[slot];
    const uint32_t k = kf & kCellKeyMask;
    // the first particle of cell k + 1 may be storing its slab offsets into cs[k + 1]
    const uint32_t a = cs[k] & T.start_mask, b = cs[k + 1] & T.start_mask;
    // the fused step's order within a cell is by (slab, id): ids are below 2^27, so the slab
    // bits of the key above the id order both
    const bool slabs = GATHER && T.shift > 0;
    const uint32_t own = slabs ? (kf & ~kCellKeyMask) | id : id;
    uint32_t r = 0, b1 = 0, b2 = 0, b3 = 0;  // b_j: particles of the cell in slabs below j
    for (uint32_t t = a; t < b; ++t) {
        const uint32_t st = tmp[t];
        if (slabs) {
            const uint32_t kt = keyI[st];
            const uint32_t q = kt >> kSlabKeyShift;
            r += ((kt & ~kCellKeyMask) | pidB[st]) < own ? 1u : 0u;
            b1 += q < 1u ? 1u : 0u;
            b2 += q < 2u ? 1u : 0u;
            b3 += q < 3u ? 1u : 0u;
        } else {
            r += pidB[st] < id ? 1u : 0u;
        }
    }
    const uint32_t f = a + r;
    if (slabs && r == 0u) {
        const uint32_t fields = slab_fields(T, b1, b2, b3, b - a);
        if (fields) cs[k] = a | fields;
    }
    skey[f] = k;
    if (!GATHER) sval[f] = slot;
    if (GATHER) {
        posA[f] = posB[slot];
        velA[f] = velB[slot];
        pidA[f] = id;
    }
}

// Few particles: the whole sort in one launch.  Every workgroup owns a contiguous range of cells:
// it reads all keys, counts those below its range (where its part of the order begins) and
// collects those in it, scans its cells' counts, places its particles cell by cell in LDS,
// orders each cell there and gathers its part of the state, and writes its part of the table.
// The passes above take five launches of about 4.4 us each at these sizes, whatever their work,
// and atomics in the force pass.  What bounds this one is one latency after another (keys, ids,
// state), and for many particles the keys' 4 n bytes in each workgroup.
// Where the particles crowd (a pile, a layer at one end of z), a range is cut into parts, which
// further workgroups take: each works the cut out for itself, from one key per thread, spread
// over all of them.  us per sort with the passes above / one workgroup per range / with the
// cut: 65,537 particles in the first cells of 1,048,576, 30 in each, 24 / 622 / 23, 500 in each
// 85 / 3,264 / 64; a layer of 5% of z, 19 / 40 / 19.  Particles that do not crowd pay 0.3 us
// (5,000) to 1 us (65,537) for the look at the sample.
// A range or part with more than `list` particles is collected in global memory (tmpE, tmpK)
// instead, by a second walk over the keys.  A cell of more than kHeavyCell particles is ordered
// through a bitmap of its (slab, id) in place of comparing each with each, which one workgroup
// alone would take long for (70,000 particles in one cell: 5e9 comparisons).
constexpr int OT = 1024;
constexpr int OWAVES = OT / 64;
constexpr int kOneGroups = 256;  // workgroups: one per CU
constexpr int kOneMost = 1 << 20;  // cells, at most
constexpr int kOneShares = 48;   // shares of all particles that ranges are measured by, at most ...
constexpr int kOneShare = 1024;  // ... and particles of one, at least
constexpr int kOneList = 3072;   // particles of a range or part kept in LDS ...
constexpr int kOneAll = 4096;    // ... all of them up to this many
constexpr int kOneLoads = 4;     // 16-byte key loads in flight per lane
constexpr int kHeavyCell = 512;
// us per step with the passes above / this one (30 neighbours, 4 lanes), in a corner of the box and all
// over it: 16,384 particles 39.9 / 32.3 and 40.0 / 32.2, 49,152 44.8 / 40.6 and 43.9 / 37.9, 65,537
// 48.8 / 47.1 and 46.1 / 42.0, 73,728 52.6 / 53.4 and 46.3 / 44.1
constexpr int64_t kOneSort = 73728;
constexpr int kHeavyMost = (int)(kOneSort / (kHeavyCell + 1)) + 1;  // heavy cells of a range, at most
inline __host__ __device__ int heavy_words(int n, bool slabs) { return ((slabs ? 4 : 1) * n + 31) / 32; }
inline __host__ __device__ int one_list(int n) { return n <= kOneAll ? kOneAll : kOneList; }
inline __host__ __device__ int one_shares(int n) { return n <= kOneAll ? 0 : min(kOneShares, n / kOneShare); }
// Parts of a range that holds `seen` of the OT sampled keys: one up to two shares of them, past that
// a part per share (rounded up), so that over all ranges the parts past the first are at most
// `shares`.
__device__ __forceinline__ uint32_t one_parts(uint32_t seen, int shares) {
    const uint32_t x = seen * (uint32_t)shares;
    return x > 2u * OT ? (x + OT - 1u) / OT : 1u;
}

// The range and the part of it that is the h-th of the parts past the first, from the sampled keys
// per range; range -1: there are fewer.  One wavefront, lane l the ranges 4 l .. 4 l + 3.
__device__ __forceinline__ void one_share(const uint32_t* hist, int ranges, int shares, int h, int* out) {
    static_assert(kOneGroups == 256, "four ranges per lane");
    const int lane = threadIdx.x & 63;
    uint32_t more[4], sum = 0u;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        more[u] = 4 * lane + u < ranges ? one_parts(hist[4 * lane + u], shares) - 1u : 0u;
        sum += more[u];
    }
    uint32_t first = wave_incl_scan(sum) - sum;
    if (lane == 63 && (uint32_t)h >= first + sum) out[0] = -1;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        if ((uint32_t)h >= first && (uint32_t)h < first + more[u]) {
            out[0] = 4 * lane + u;
            out[1] = h - (int)first + 1;
        }
        first += more[u];
    }
}

// SHARED: one_shares(n) > 0.
template <bool GATHER, bool SHARED>
__global__ __launch_bounds__(OT) void cell_sort_one_kernel(
    int n, int m, int per, int ranges, SlabTable T, const uint32_t* __restrict__ keyI,
    const uint32_t* __restrict__ pidB, uint32_t* __restrict__ cs, uint32_t* __restrict__ skey,
    uint32_t* __restrict__ sval, const float4* __restrict__ posB, const float4* __restrict__ velB,
    float4* __restrict__ posA, float4* __restrict__ velA, uint32_t* __restrict__ pidA, uint32_t* tmpE, uint32_t* tmpK) {
    extern __shared__ uint32_t s_one[];
    const int list = one_list(n), shares = one_shares(n);
    uint32_t* const start = s_one;          // per + 1: a cell's first place in the range
    uint32_t* const cur = start + per + 1;  // per: its count, its next free place, its table entry's fields
    uint32_t* const ordE = cur + per;       // list: the range's particles (slots) cell by cell
    uint32_t* const ordK = ordE + list;     // ... (slab, id) there
    uint32_t* const listE = ordK + list;    // ... as found
    uint32_t* const listK = listE + list;   // ... their keys
    uint32_t* const bits = listE;           // heavy_words, after that: a heavy cell's (slab, id)
    __shared__ uint32_t s_wave[OWAVES], s_count, s_below, s_heavy, s_cell[kHeavyMost], s_ones[OT];
    __shared__ uint32_t s_hist[kOneGroups], s_seen;
    __shared__ int s_share[2], s_lo, s_hi;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    auto cell_of = [&](uint32_t key) { return (int)(key & kCellKeyMask); };
    // this thread's sample of the keys: four neighbours share one of 256 places
    const int sample = SHARED ? cell_of(keyI[(tid / 4) * (n / 4) / (OT / 4) * 4 + tid % 4]) : 0;
    const uint4* const key4 = reinterpret_cast<const uint4*>(keyI);
    const int quads = n / 4;
    uint4 k[kOneLoads] = {};
    auto load = [&](int v0) {
#pragma unroll
        for (int u = 0; u < kOneLoads; ++u) k[u] = key4[min(v0 + u * OT, quads - 1)];
    };
    if (quads > 0) load(tid);  // while the samples are looked at
    for (int c = tid; c < per; c += OT) cur[c] = 0u;
    if (tid == 0) s_count = s_below = s_heavy = s_seen = 0u;
    const int block = xcd_tile(blockIdx.x, gridDim.x);
    int range = block, part = 0;
    if (SHARED && block >= ranges) {
        for (int r = tid; r < kOneGroups; r += OT) s_hist[r] = 0u;
        __syncthreads();
        atomicAdd(&s_hist[sample / per], 1u);
        __syncthreads();
        if (w == 0) one_share(s_hist, ranges, shares, block - ranges, s_share);
        __syncthreads();
        range = s_share[0];
        part = s_share[1];
        if (range < 0) return;
    }
    int lo = range * per, hi = min(lo + per, m);  // this range of cells
    auto mine = [&](int c) { return c >= lo && c < hi; };
    __syncthreads();
    if constexpr (SHARED) {
        const uint32_t found = (uint32_t)__popcll(__ballot(mine(sample)));
        if (lane == 0 && found) atomicAdd(&s_seen, found);
        __syncthreads();
        const uint32_t seen = s_seen, parts = one_parts(seen, shares);
        if (parts > 1u) {  // the part's: the cells before which its share of the range's samples lies
            const int cells = hi - lo;
            if (mine(sample)) atomicAdd(&cur[sample - lo], 1u);
            if (tid == 0) s_lo = s_hi = cells;
            __syncthreads();
            const int each = (cells + OT - 1) / OT;
            const int c0 = min(tid * each, cells), c1 = min(c0 + each, cells);
            uint32_t sum = 0u;
            for (int c = c0; c < c1; ++c) sum += cur[c];
            const uint32_t incl = wave_incl_scan(sum);
            if (lane == 63) s_wave[w] = incl;
            __syncthreads();
            uint32_t run = incl - sum;
            for (int j = 0; j < w; ++j) run += s_wave[j];
            const float rate = (float)parts / (float)seen;
            auto part_of = [&](uint32_t before) { return min((int)((float)before * rate), (int)parts - 1); };
            // the wavefront's first cell of this part or a later one, and of a later one
            auto bound = [&](int least, int* at) {
                const uint64_t found = __ballot(c0 < c1 && part_of(run + sum) >= least);
                if (!found || lane != __ffsll((unsigned long long)found) - 1) return;
                uint32_t before = run;
                int c = c0;
                while (c < c1 && part_of(before) < least) before += cur[c++];
                atomicMin(at, c);
            };
            if (part > 0) bound(part, &s_lo);
            bound(part + 1, &s_hi);
            __syncthreads();
            hi = lo + s_hi;
            lo += part > 0 ? s_lo : 0;
            for (int c = tid; c < cells; c += OT) cur[c] = 0u;
            __syncthreads();
        }
    }
    const int own = hi - lo;
    uint32_t below = 0u;
    auto take = [&](uint32_t key, int c, int e) {
        atomicAdd(&cur[c - lo], 1u);
        const uint32_t at = atomicAdd(&s_count, 1u);
        if (at < (uint32_t)list) {
            listE[at] = (uint32_t)e;
            listK[at] = key;
        }
    };
    // most quads hold no key of the range
    for (int v0 = tid; v0 < quads; v0 += kOneLoads * OT) {
        if (v0 != tid) load(v0);
#pragma unroll
        for (int u = 0; u < kOneLoads; ++u) {
            const int v = v0 + u * OT;
            if (v >= quads) break;
            const int c[4] = {cell_of(k[u].x), cell_of(k[u].y), cell_of(k[u].z), cell_of(k[u].w)};
            below += (c[0] < lo ? 1u : 0u) + (c[1] < lo ? 1u : 0u) + (c[2] < lo ? 1u : 0u) + (c[3] < lo ? 1u : 0u);
            if (mine(c[0]) || mine(c[1]) || mine(c[2]) || mine(c[3])) {
                if (mine(c[0])) take(k[u].x, c[0], 4 * v);
                if (mine(c[1])) take(k[u].y, c[1], 4 * v + 1);
                if (mine(c[2])) take(k[u].z, c[2], 4 * v + 2);
                if (mine(c[3])) take(k[u].w, c[3], 4 * v + 3);
            }
        }
    }
    for (int e = 4 * quads + tid; e < n; e += OT) {
        const uint32_t key = keyI[e];
        const int c = cell_of(key);
        below += c < lo ? 1u : 0u;
        if (mine(c)) take(key, c, e);
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) below += __shfl_xor(below, o);
    if (lane == 0 && below) atomicAdd(&s_below, below);
    __syncthreads();
    const uint32_t base = s_below, count = s_count;
    // exclusive scan of the counts, thread t the cells [t each, (t + 1) each)
    const int each = (own + OT - 1) / OT;
    const int c0 = min(tid * each, own), c1 = min(c0 + each, own);
    uint32_t sum = 0u;
    for (int c = c0; c < c1; ++c) sum += cur[c];
    const uint32_t incl = wave_incl_scan(sum);
    if (lane == 63) s_wave[w] = incl;
    __syncthreads();
    uint32_t run = incl - sum;
    for (int k = 0; k < w; ++k) run += s_wave[k];
    for (int c = c0; c < c1; ++c) {
        const uint32_t v = cur[c];
        start[c] = run;
        cur[c] = run;
        run += v;
        if (v > (uint32_t)kHeavyCell) s_cell[atomicAdd(&s_heavy, 1u)] = (uint32_t)c;
    }
    if (tid == 0) start[own] = count;
    __syncthreads();
    // the range's particles cell by cell in E and K, then each one's place in its cell: the number
    // of the cell's particles before it
    const bool slabs = GATHER && T.shift > 0;
    auto order = [&](uint32_t* E, uint32_t* K, bool listed) {
        auto place = [&](uint32_t key, uint32_t e) {
            const uint32_t at = atomicAdd(&cur[cell_of(key) - lo], 1u);
            E[at] = e;
            // ids are below 2^27, so the slab bits of a key above the id order both
            K[at] = (slabs ? key & ~kCellKeyMask : 0u) | pidB[e];
        };
        if (listed) {
            for (uint32_t at = tid; at < count; at += OT) place(listK[at], listE[at]);
        } else {
            for (int e = tid; e < n; e += OT) {
                const uint32_t key = keyI[e];
                if (mine(cell_of(key))) place(key, (uint32_t)e);
            }
            __threadfence_block();
        }
        __syncthreads();
        // particle E[at] of cell c: r of its particles come before it, b_j are in slabs below j
        auto put = [&](uint32_t at, int c, uint32_t r, uint32_t b1, uint32_t b2, uint32_t b3) {
            const uint32_t e = E[at], f = base + start[c] + r;
            if (slabs && r == 0u) cur[c] = slab_fields(T, b1, b2, b3, start[c + 1] - start[c]);
            skey[f] = (uint32_t)(c + lo);
            if (!GATHER) sval[f] = e;
            if (GATHER) {
                posA[f] = posB[e];
                velA[f] = velB[e];
                pidA[f] = K[at] & kIdMask;
            }
        };
        for (uint32_t at = tid; at < count; at += OT) {
            const uint32_t rank = K[at];
            const int c = cell_of(keyI[E[at]]) - lo;
            const uint32_t a = start[c], b = start[c + 1];
            if (b - a > (uint32_t)kHeavyCell) continue;
            uint32_t r = 0, b1 = 0, b2 = 0, b3 = 0;
            for (uint32_t t = a; t < b; ++t) {
                const uint32_t kt = K[t];
                r += kt < rank ? 1u : 0u;
                if (slabs) {
                    const uint32_t q = kt >> kSlabKeyShift;
                    b1 += q < 1u ? 1u : 0u;
                    b2 += q < 2u ? 1u : 0u;
                    b3 += q < 3u ? 1u : 0u;
                }
            }
            put(at, c, r, b1, b2, b3);
        }
        const int words = heavy_words(n, slabs), share = (words + OT - 1) / OT;
        auto place_of = [&](uint32_t k) { return (slabs ? (k >> kSlabKeyShift) * (uint32_t)n : 0u) + (k & kIdMask); };
        for (uint32_t h = 0; h < s_heavy; ++h) {
            const int c = (int)s_cell[h];
            const uint32_t a = start[c], b = start[c + 1];
            for (int x = tid; x < words; x += OT) bits[x] = 0u;
            __syncthreads();
            for (uint32_t t = a + tid; t < b; t += OT) {
                const uint32_t x = place_of(K[t]);
                atomicOr(&bits[x >> 5], 1u << (x & 31u));
            }
            __syncthreads();
            // ones before each thread's share of the words
            uint32_t ones = 0u;
            for (int x = tid * share; x < min((tid + 1) * share, words); ++x) ones += (uint32_t)__popc(bits[x]);
            const uint32_t upto = wave_incl_scan(ones);
            if (lane == 63) s_wave[w] = upto;
            __syncthreads();
            uint32_t first = upto - ones;
            for (int k = 0; k < w; ++k) first += s_wave[k];
            s_ones[tid] = first;
            __syncthreads();
            auto before = [&](uint32_t x) {
                const int word = (int)(x >> 5);
                if (word >= words) return b - a;
                uint32_t r = s_ones[word / share];
                for (int y = word / share * share; y < word; ++y) r += (uint32_t)__popc(bits[y]);
                return r + (uint32_t)__popc(bits[word] & ((1u << (x & 31u)) - 1u));
            };
            for (uint32_t t = a + tid; t < b; t += OT)
                put(t, c, before(place_of(K[t])), slabs ? before((uint32_t)n) : 0u,
                    slabs ? before(2u * (uint32_t)n) : 0u, slabs ? before(3u * (uint32_t)n) : 0u);
            __syncthreads();
        }
    };
    if (count <= (uint32_t)list) order(ordE, ordK, true);
    else order(tmpE + base, tmpK + base, false);
    __syncthreads();
    const uint32_t empty = T.empty();
    for (int c = tid; c < own; c += OT)
        cs[c + lo] = (base + start[c]) | (start[c] == start[c + 1] ? empty : slabs ? cur[c] : 0u);
    if (hi == m && tid == 0) cs[m] = (uint32_t)n;
}

inline int cblocks(int64_t n) { return (int)((n + CT - 1) / CT); }

}  // namespace

bool cell_sort_one(const sph_ctx* c) {
    return c->n <= kOneSort && c->sc.cs_cells <= kOneMost;
}

int64_t cell_scan_tiles(int64_t cells) { return (cells + CTILE - 1) / CTILE; }

// Sorted keys and slots go to keyS[1] / valS[1]; the cell table to cs.  counted: the
// per-cell counts and the ranks (in keyS[0]) of the current keys are there already, and with
// tile_sums_in_force also the tile sums (cell_part array part_phase) (launch_force with
// count; only on the global path, see count_in_force).  The scan clears the other array and
// part_phase names it afterwards.
hipError_t launch_cell_sort(sph_ctx* c, bool gather, hipStream_t s, bool counted) {
    const int n = (int)c->n;
    const int m = c->sc.cs_cells;
    const Buffers& b = c->b;
    uint32_t* rank = b.keyS[0];
    uint32_t* tmp = b.valS[0];
    const int tiles = (int)cell_scan_tiles(m);
    const SlabTable T = slab_table(c->sc);
    c->sorted_keys = b.keyS[1];
    c->sorted_vals = b.valS[1];
    if (cell_sort_one(c)) {
        const int shares = one_shares(n), most = kOneGroups - shares;
        const int per = std::max(1, (m + most - 1) / most), ranges = std::max(1, (m + per - 1) / per);
        const int groups = ranges + shares;
        const size_t lds = sizeof(uint32_t) * (2 * (size_t)per + 1 + 2 * one_list(n) +
                                               std::max(2 * one_list(n), heavy_words(n, gather && T.shift > 0)));
        const auto kernel =
            shares > 0 ? (gather ? cell_sort_one_kernel<true, true> : cell_sort_one_kernel<false, true>)
                       : (gather ? cell_sort_one_kernel<true, false> : cell_sort_one_kernel<false, false>);
        kernel<<<groups, OT, lds, s>>>(
            n, m, per, ranges, T, b.keyI, b.pidB, b.cs, b.keyS[1], b.valS[1], b.posB, b.velB, b.posA, b.velA, b.pidA,
            tmp, rank);
        return hipGetLastError();
    }
    const bool summed = counted && tile_sums_in_force(c);
    const int cur = summed ? c->part_phase : 0;
    uint32_t* part = b.cell_part + (size_t)cur * kTileSumCopies * tiles;
    uint32_t* next = b.cell_part + (size_t)(cur ^ 1) * kTileSumCopies * tiles;
    c->part_phase = cur ^ 1;
    if (n > 0 && !counted) cell_count_kernel<<<cblocks(n), CT, 0, s>>>(n, b.keyI, b.cell_cnt, rank);
    if (!summed) cell_scan_reduce<<<tiles, CT, 0, s>>>(b.cell_cnt, m, part);
    const int copies = summed ? kTileSumCopies : 1;
    if (tiles <= kMergedTiles) {
        cell_scan_down<true><<<tiles, CT, 0, s>>>(b.cell_cnt, m, part, next, b.cs, (uint32_t)n, T.empty(), copies);
    } else {
        cell_scan_partials<<<1, CT, 0, s>>>(part, tiles, copies);
        cell_scan_down<false><<<tiles, CT, 0, s>>>(b.cell_cnt, m, part, next, b.cs, (uint32_t)n, T.empty(), copies);
    }
    if (n > 0) {
        cell_scatter_kernel<<<cblocks(n), CT, 0, s>>>(n, b.keyI, rank, b.cs, tmp, T.start_mask);
        if (gather)
            cell_order_kernel<true><<<cblocks(n), CT, 0, s>>>(n, T, tmp, b.keyI, b.cs, b.keyS[1], b.valS[1], b.posB,
                                                               b.velB, b.pidB, b.posA, b.velA, b.pidA);
        else
            cell_order_kernel<false><<<cblocks(n), CT, 0, s>>>(n, T, tmp, b.keyI, b.cs, b.keyS[1], b.valS[1], nullptr,
                                                                nullptr, b.pidB, nullptr, nullptr, nullptr);
    }
    return hipGetLastError();
}

}  // namespace sph
