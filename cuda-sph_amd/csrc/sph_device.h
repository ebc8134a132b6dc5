// sph_device.h -- device helpers shared by the step kernels (sph_kernels.hip) and the
// reverse-mode kernels (sph_adjoint.hip).  The adjoint recomputes the force pass with the
// same code as the step, so its recomputed forward is bitwise the step's own.
#pragma once
#include <limits.h>
#include <math.h>

#include "sph_internal.h"

namespace sph {
namespace {

// Workgroup -> tile mapping that gives each of the 8 XCDs (one L2 each) a contiguous
// range of cell-ordered tiles, so neighbour reads of adjacent tiles hit the same L2.
// Workgroups are dispatched round-robin over XCDs: block b runs on XCD b % 8.
__device__ __forceinline__ int xcd_tile(int bid, int nb) {
    if (nb < 2 * kXcds) return bid;
    const int q = nb / kXcds, r = nb % kXcds;
    const int x = bid % kXcds, local = bid / kXcds;
    return x < r ? x * (q + 1) + local : r * (q + 1) + (x - r) * q + local;
}

// The mapping of the batched passes where StepConsts::spread says so: every XCD takes each eighth chunk
// of kBatchChunk tiles, so that the instances, whose particles cost up to 300 times as much in one as
// in another, are spread over all of them.  Contiguous eighths of the threads (xcd_tile) left the two
// densest of 64 boxes to three XCDs while the others ran out of work (4 steps, 5.98 ms against 4.88).
// Where all XCDs have as much to do, eighths keep an instance, and what the sort wrote of it, in
// one L2: 64 instances of 4,096 particles with 1,000 neighbours, 8 lanes, 1.25 ms per step against
// 1.72 in chunks, 8 of 60,000 with 30 neighbours 0.179 against 0.202.
constexpr int kBatchChunk = 16;
__device__ __forceinline__ int xcd_chunk_tile(int bid, int nb) {
    constexpr int round = kXcds * kBatchChunk;
    const int whole = nb / round * round;
    if (bid >= whole) return bid;  // the last, partial round
    const int x = bid % kXcds, local = bid / kXcds;
    return (local / kBatchChunk * kXcds + x) * kBatchChunk + local % kBatchChunk;
}

// Constants of the instance that owns particle slot i.  A plain step has one instance (the
// kernel argument itself).  In the batched form every instance owns a contiguous range of
// particle ids and, because its cell keys form a contiguous range too, the same range of
// cell-ordered slots; the range is found by binary search over the instance offsets.
template <bool BATCH>
__device__ __forceinline__ const StepConsts& inst_consts(const StepConsts& G, int i) {
    if constexpr (!BATCH) {
        return G;
    } else {
        int lo = 0, hi = G.n_inst;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (G.inst_first[mid] <= i) lo = mid;
            else hi = mid;
        }
        return G.inst_table[lo];
    }
}


// The value of lane (own lane) ^ O for O = 1, 2, 16 and, where every aligned group of O lanes holds
// one value, O = 4 and 8 (by mirroring: lane 7 - i and 15 - i of the row): as the steps of a sum
// over a group these need no LDS access up to 8, against a ds_bpermute and its address each.
// The sums come out as those of __shfl_xor, bit for bit.
template <int O>
__device__ __forceinline__ uint32_t lane_xor(uint32_t v) {
    if constexpr (O == 1) return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xb1, 0xf, 0xf, true);   // quad_perm 1 0 3 2
    else if constexpr (O == 2) return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4e, 0xf, 0xf, true);  // 2 3 0 1
    else if constexpr (O == 4) return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xf, 0xf, true);  // row_half_mirror
    else if constexpr (O == 8) return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xf, 0xf, true);  // row_mirror
    else if constexpr (O == 16) return (uint32_t)__builtin_amdgcn_ds_swizzle((int)v, 0x401f);  // xor 16 within 32
    else return (uint32_t)__shfl_xor((int)v, O);
}
// Combination of one value per lane over each group of L lanes, in all of them.
template <int L, typename F>
__device__ __forceinline__ uint32_t group_fold(uint32_t v, F&& f) {
    if constexpr (L > 1) v = f(v, lane_xor<1>(v));
    if constexpr (L > 2) v = f(v, lane_xor<2>(v));
    if constexpr (L > 4) v = f(v, lane_xor<4>(v));
    if constexpr (L > 8) v = f(v, lane_xor<8>(v));
    if constexpr (L > 16) v = f(v, lane_xor<16>(v));
    if constexpr (L > 32) v = f(v, lane_xor<32>(v));
    return v;
}
template <int L>
__device__ __forceinline__ float group_sum(float v) {
    return __uint_as_float(group_fold<L>(__float_as_uint(v), [](uint32_t a, uint32_t b) {
        return __float_as_uint(__uint_as_float(a) + __uint_as_float(b));
    }));
}

// Between the stores to LDS of some lanes of a wavefront and the loads of others, and back: a
// wavefront's LDS accesses are carried out in order, so nothing is waited for, but the compiler
// has to keep them in it.
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Raw buffer loads with 32-bit byte offsets: no 64-bit address arithmetic per access, and
// an offset past num_records reads zero instead of faulting.  Word 3 of the descriptor is
// the gfx9 value for untyped 32-bit-element buffers.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ float4 ld_f4(__amdgpu_buffer_rsrc_t r, uint32_t byte_off) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)byte_off, 0, 0);
    return make_float4(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]), __uint_as_float(v[3]));
}
__device__ __forceinline__ uint32_t ld_u32(__amdgpu_buffer_rsrc_t r, uint32_t byte_off) {
    return __builtin_amdgcn_raw_buffer_load_b32(r, (int)byte_off, 0, 0);
}

// ---------------------------------------------------------------------------------------
// Voxel keys.  Reference semantics (voxel_kernels.py:9-17, 88-105): per axis
// int32(x / voxel) truncated toward zero, flattened as x + y*Dx + z*Dx*Dy with wrapping
// int32 arithmetic and no clamping.  Grid semantics: the same but floor and clamped to the
// grid, which keeps every pair within h in neighbouring cells for any position.  Both are
// equal for 0 <= x < Dx*voxel, and both are exact: with power-of-two voxels x * (1/voxel)
// is exact in FP32; otherwise the quotient is formed in FP64 as the reference does.
// ---------------------------------------------------------------------------------------
__device__ __forceinline__ int grid_coord(float x, int d, const StepConsts& C) {
    float q;
    if (C.pow2) q = floorf(x * C.inv_cell[d]);
    else q = (float)floor((double)x / C.dcell[d]);
    q = fminf(fmaxf(q, 0.0f), (float)(C.dims[d] - 1));  // NaN -> 0
    return (int)q;
}

__device__ __forceinline__ int32_t ref_coord(float x, int d, const StepConsts& C) {
    if (C.pow2) return __float2int_rz(x * C.inv_cell[d]);
    return __double2int_rz((double)x / C.dcell[d]);
}

__device__ __forceinline__ uint32_t sort_key(float x, float y, float z, const StepConsts& C) {
    if (C.ref_keys) {
        uint32_t vx = (uint32_t)ref_coord(x, 0, C), vy = (uint32_t)ref_coord(y, 1, C),
                 vz = (uint32_t)ref_coord(z, 2, C);
        uint32_t key = vx + vy * (uint32_t)C.dims[0] + vz * (uint32_t)C.dims[0] * (uint32_t)C.dims[1];
        return key ^ 0x80000000u;  // signed order as unsigned
    }
    const int cx = grid_coord(x, 0, C);
    uint32_t key = (uint32_t)(C.cell_off + cx + C.dims[0] * (grid_coord(y, 1, C) + C.dims[1] * grid_coord(z, 2, C)));
    if (C.slab_shift > 0) {
        // the x slab within the cell: floor(S x / edge) - S cx, clamped to the cell's slabs
        // (the edge cells' outer slabs extend to infinity, NaN -> 0); exact for power-of-two
        // edges, and monotone in x otherwise
        const float S = (float)(1 << C.slab_shift);
        const float q = floorf(x * C.inv_cell[0] * S) - S * (float)cx;
        key |= (uint32_t)fminf(fmaxf(q, 0.0f), S - 1.0f) << kSlabKeyShift;
    }
    return key;
}

// The start of a cell held by a cell-table entry, and the offset + 1 of slab k (1 .. S - 1)
// from it (0 for k = 0, and 0 when not known); see StepConsts::slab_shift.
__device__ __forceinline__ uint32_t table_start(uint32_t w, const StepConsts& C) { return w & C.start_mask; }
__device__ __forceinline__ uint32_t slab_field(uint32_t w, uint32_t k, const StepConsts& C) {
    // the three fields with a zero field for slab 0 below them (start_bits is above slab_bits):
    // no select for k = 0, and no 32-bit product (a quarter-rate instruction)
    static_assert(kSlabBits == 3, "3 k from a shift and an add");
    const uint32_t fields = (w >> (C.start_bits - kSlabBits)) & C.field_mask;
    return __builtin_amdgcn_ubfe(fields, k + 2u * k, kSlabBits);
}

// bucket of a sort key in the cell table: -1 below the grid, n_cells above it
__device__ __forceinline__ int key_bucket(uint32_t ukey, const StepConsts& C) {
    if (!C.ref_keys) return (int)ukey;
    const int32_t s = (int32_t)(ukey ^ 0x80000000u);
    return s < 0 ? -1 : (s >= C.n_cells ? C.n_cells : s);
}

__device__ __forceinline__ bool finite3(float x, float y, float z) {
    return isfinite(x) && isfinite(y) && isfinite(z);
}

// Sort input of the next step.  SLOT_KEYS (the NAIVE formulation's counting sort): the key
// of the particle in posB slot `slot`, indexed by the slot, so the keys stay in the current
// cell order (coalesced stores; the sort's atomics and scatters touch neighbouring cells).
// Otherwise (the radix sort, which must see particle-id order to be stable by id): key and
// slot indexed by particle id.
// Returns the key.
template <bool SLOT_KEYS>
__device__ __forceinline__ uint32_t hash_particle(const StepConsts& C, float x, float y, float z, uint32_t pid,
                                                  uint32_t slot, uint32_t* __restrict__ keyI,
                                                  uint32_t* __restrict__ valI, uint32_t* __restrict__ flags) {
    const uint32_t key = sort_key(x, y, z, C);
    if constexpr (SLOT_KEYS) {
        keyI[slot] = key;
    } else {
        keyI[pid] = key;
        valI[pid] = slot;
    }
    if (!finite3(x, y, z)) atomicAdd(flags + kFlagNonFinite, 1u);
    return key;
}

// Rank of a key among the equal keys counted into cnt (the counting sort's per-cell
// counts): rank = atomicAdd(&cnt[key], 1), in an arbitrary order among the particles of a
// cell.  Consecutive slots are often in the same cell, so a wavefront's lanes come in runs
// of equal keys: the first lane of each run adds the run's length with one atomic and the
// run's lanes take consecutive ranks from the returned base.  The lanes that hold a key
// (valid) must be a prefix of the wavefront, and every active lane must call this together.
__device__ __forceinline__ uint32_t rank_in_cell(uint32_t key, bool valid, uint32_t* __restrict__ cnt) {
    const int lane = threadIdx.x & 63;
    const uint32_t prev = __shfl_up(key, 1);
    const bool head = valid && (lane == 0 || prev != key);
    const uint64_t heads = __ballot(head);
    const uint64_t valids = __ballot(valid);
    const uint64_t upto = lane == 63 ? ~0ull : ((1ull << (lane + 1)) - 1ull);
    const int first = 63 - __clzll((long long)(heads & upto));  // first lane of this lane's run
    const uint64_t above = heads & ~upto;
    // first lane of the next run, or one past the last valid lane
    const int next = above ? __ffsll((unsigned long long)above) - 1 : 64 - __clzll((long long)valids);
    uint32_t base = 0;
    if (head) base = atomicAdd(&cnt[key], (uint32_t)(next - lane));
    base = __shfl(base, first);
    return base + (uint32_t)(lane - first);
}

// Adds each active lane's cell to the sum of its scan tile, the counting sort's tile sums:
// part[cell >> kScanTileShift] of the copy that part points to.  The lanes with the first
// remaining lane's tile add their number with one atomic, until none is left: the keys of a
// wavefront are nearly in cell order, so that is mostly one atomic per wavefront.  Every
// active lane must call this together (the loop is uniform across the wavefront).
__device__ __forceinline__ void add_to_tile_sums(uint32_t cell, uint32_t* __restrict__ part) {
    const uint32_t tile = cell >> kScanTileShift;
    bool pending = true;
    for (uint64_t left = __ballot(1); left != 0; left = __ballot(pending)) {
        const int lead = __ffsll((unsigned long long)left) - 1;
        const uint32_t t = (uint32_t)__builtin_amdgcn_readlane((int)tile, lead);
        const bool mine = pending && tile == t;
        const uint64_t same = __ballot(mine);
        if ((int)(threadIdx.x & 63) == lead) atomicAdd(&part[t], (uint32_t)__popcll(same));
        pending = pending && !mine;
    }
}

// VOXEL formulation: whether a finite position lies outside the voxel grid, i.e. its key
// (truncated voxel index per axis, voxel_kernels.py:9-17) leaves [0, dims) on some axis and
// so wraps onto the key of another voxel or off the table.  Positions in (-voxel, 0) truncate
// into voxel 0 and count as inside (the density pass treats voxel 0 as open below).
// Non-finite positions count as inside: no pair test ever accepts them.
__device__ __forceinline__ bool outside_voxel_grid(float x, float y, float z, const StepConsts& C) {
    if (!finite3(x, y, z)) return false;
    const int32_t vx = ref_coord(x, 0, C), vy = ref_coord(y, 1, C), vz = ref_coord(z, 2, C);
    return vx < 0 || vx >= C.dims[0] || vy < 0 || vy >= C.dims[1] || vz < 0 || vz >= C.dims[2];
}

// ---------------------------------------------------------------------------------------
// Neighbour candidates of the NAIVE formulation.  For each row of cells (y, z) whose slab
// comes within h of the particle, the x cells are those overlapping [x - e, x + e] with
// e = sqrt(h^2 - dy^2 - dz^2); cells of one row are consecutive keys, so the candidates
// of a row are one contiguous range cs[first]..cs[last+1].  Boundary cells extend to
// infinity (positions outside the grid are clamped into them).  The search radius carries
// a small margin; the exact test r^2 <= h^2 is applied to each candidate.
// ---------------------------------------------------------------------------------------
// The rows of cells that the sphere of radius h_search around a particle reaches, in
// increasing cell order (cz, then cy): a row is the run of cells along x that the sphere's
// chord through the nearest point of the row's (y, z) slab covers, taken in x slabs of the
// cells (StepConsts::slab_shift; whole cells when the cells are not cut), so that its
// candidates are one contiguous range of the cell order.  The position is clamped into the
// grid first; an edge cell holds the particles beyond it, so a particle outside the grid
// gets a superset of its rows.  The margin of h_search over h covers the rounding of this
// float arithmetic (a slab it adds or drops holds only particles beyond h).
struct RowGrid {
    float gx, gy, gz, fx, hs2, mx, sinv;  // fx, mx: x in slabs; sinv: slabs per unit length
    int ylo, yhi, zlo, zhi;

    __device__ __forceinline__ RowGrid(float px, float py, float pz, const StepConsts& C) {
        const float hs = C.h_search;
        hs2 = hs * hs;
        const float S = (float)(1 << C.slab_shift);
        const float my = (float)(C.dims[1] - 1), mz = (float)(C.dims[2] - 1);
        gx = fminf(fmaxf(px, 0.0f), (float)C.dims[0] * C.cell[0]);  // NaN -> 0
        gy = fminf(fmaxf(py, 0.0f), (my + 1.0f) * C.cell[1]);
        gz = fminf(fmaxf(pz, 0.0f), (mz + 1.0f) * C.cell[2]);
        ylo = (int)__builtin_amdgcn_fmed3f((gy - hs) * C.inv_cell[1], 0.0f, my);
        yhi = (int)__builtin_amdgcn_fmed3f((gy + hs) * C.inv_cell[1], 0.0f, my);
        zlo = (int)__builtin_amdgcn_fmed3f((gz - hs) * C.inv_cell[2], 0.0f, mz);
        zhi = (int)__builtin_amdgcn_fmed3f((gz + hs) * C.inv_cell[2], 0.0f, mz);
        sinv = C.inv_cell[0] * S;
        fx = gx * sinv;
        mx = (float)C.dims[0] * S - 1.0f;
    }

    // distance from the particle to the slab [c s, (c + 1) s), zero inside it
    __device__ __forceinline__ static float slab(float g, int c, float s) {
        const float f = (float)c;
        return fmaxf(fmaxf(fmaf(f, s, -g), fmaf(-f, s, g - s)), 0.0f);
    }

    // h_search^2 less the squared distance to the slab of cz
    __device__ __forceinline__ float rest_z(int cz, const StepConsts& C) const {
        const float ez = slab(gz, cz, C.cell[2]);
        return fmaf(-ez, ez, hs2);
    }

    // the row at cy of the slab of cz (rz: rest_z(cz)): its first x slab q0 and one past its
    // last, q1, counted from the row's first cell; false if the sphere misses the row's slab
    __device__ __forceinline__ bool row(int cy, float rz, const StepConsts& C, uint32_t& q0, uint32_t& q1) const {
        const float ey = slab(gy, cy, C.cell[1]);
        const float rem = fmaf(-ey, ey, rz);
        if (!(rem >= 0.0f)) return false;
        const float ex = __builtin_amdgcn_sqrtf(rem) * sinv;
        q0 = (uint32_t)(int)__builtin_amdgcn_fmed3f(fx - ex, 0.0f, mx);
        q1 = (uint32_t)(int)__builtin_amdgcn_fmed3f(fx + ex, 0.0f, mx) + 1u;
        return true;
    }

    // the candidates [k0, k1) of slabs q0 .. q1 - 1 of the row whose first cell is row0, from
    // the cell-table entries of the cell holding q0 and of the cell holding q1 (the next
    // cell's start when q1 is a cell's first slab), ld(c) reading entry c
    template <typename LD>
    __device__ __forceinline__ static void range(int row0, uint32_t q0, uint32_t q1, const StepConsts& C, LD&& ld,
                                                 uint32_t& k0, uint32_t& k1) {
        const int sh = C.slab_shift;
        const uint32_t m = (1u << sh) - 1u;
        const int e = row0 + (int)(q1 >> sh);
        const uint32_t a = ld(row0 + (int)(q0 >> sh)), b = ld(e);
        const uint32_t fa = slab_field(a, q0 & m, C), fb = slab_field(b, q1 & m, C);
        k0 = table_start(a, C) + (fa ? fa - 1u : 0u);
        k1 = table_start(b, C) + (fb ? fb - 1u : 0u);
        // the end lies inside a cell whose slab offsets are not known: the whole cell, from its
        // count if the entry keeps it, else from the next cell's start
        if ((q1 & m) != 0u && fb == 0u) {
            const uint32_t nb = C.count_bits ? __builtin_amdgcn_ubfe(b, (uint32_t)C.count_pos, (uint32_t)C.count_bits) : 0u;
            k1 = nb ? table_start(b, C) + nb - 1u : table_start(ld(e + 1), C);
        }
    }
};

template <typename LD, typename F>
__device__ __forceinline__ void for_each_row(float px, float py, float pz, const StepConsts& C, LD&& ld, F&& f) {
    const RowGrid R(px, py, pz, C);
    for (int cz = R.zlo; cz <= R.zhi; ++cz) {
        const float rz = R.rest_z(cz, C);
        int row0 = C.cell_off + C.dims[0] * (R.ylo + C.dims[1] * cz);
        for (int cy = R.ylo; cy <= R.yhi; ++cy, row0 += C.dims[0]) {
            uint32_t q0, q1;
            if (R.row(cy, rz, C, q0, q1)) {
                uint32_t k0, k1;
                RowGrid::range(row0, q0, q1, C, ld, k0, k1);
                f(k0, k1);
            }
        }
    }
}

// Where the scan of a particle's candidates starts: at the first candidate k in the row of cells
// (cy, cz), or, without a list, at its first row (cy = cz = INT_MIN stands for it).
struct ListTail {
    uint32_t k = 0u;
    int cy = INT_MIN, cz = INT_MIN;
    ListTail() = default;
    // after its last listed neighbour, in the row that holds it (grid_coord gives the cell that
    // it was sorted by)
    __device__ __forceinline__ ListTail(uint32_t last, float4 q, const StepConsts& C)
        : k(last + 1u), cy(grid_coord(q.y, 1, C)), cz(grid_coord(q.z, 2, C)) {}
};

template <typename F>
__device__ __forceinline__ void for_each_candidate(float px, float py, float pz, const StepConsts& C,
                                                   const uint32_t* __restrict__ cs, F&& f) {
    for_each_row(px, py, pz, C, [&](int c) { return cs[c]; }, [&](uint32_t k0, uint32_t k1) {
        for (uint32_t k = k0; k < k1; ++k) f(k);
    });
}

// The rows [k0, k1) of a group's L lanes (k0 <= k1) laid end to end in lane order: the row of lane l
// has the places [start, start + k1 - k0) of `total`, and window() gives lane l the candidate at
// place `at` + l, for at = 0, L, ... in turn with one `seen` (past the last place: anything).
template <int L>
struct RowWindows {
    static_assert(L == 32, "starts are bits of one word");
    uint32_t total, start, l;
    uint32_t shift;  // of the l-th row that is not empty: k0 less start
    int gbase;
    bool any;
    __device__ __forceinline__ RowWindows(uint32_t k0, uint32_t k1, uint32_t lane, int base) : l(lane), gbase(base) {
        const uint32_t len = k1 - k0;
        any = len != 0u;
        uint32_t sum = len;
#pragma unroll
        for (int o = 1; o < L; o <<= 1) {
            const uint32_t y = __shfl_up(sum, o, L);
            if ((int)l >= o) sum += y;
        }
        total = __shfl(sum, L - 1, L);
        start = sum - len;
        // the rows that are not empty to the first lanes
        const uint32_t full = (uint32_t)(__ballot(any) >> gbase);
        const uint32_t before = (uint32_t)__popc(full & ((1u << l) - 1u));
        const uint32_t to = any ? before : (uint32_t)__popc(full) + l - before;
        shift = (uint32_t)__builtin_amdgcn_ds_permute((gbase + (int)to) * 4, (int)(k0 - start));
    }
    // seen: rows that start before the window
    __device__ __forceinline__ uint32_t window(uint32_t& seen, uint32_t at) const {
        const uint32_t rel = start - at;
        const uint32_t starts = group_fold<L>(any && rel < (uint32_t)L ? 1u << rel : 0u,
                                              [](uint32_t x, uint32_t y) { return x | y; });
        const uint32_t row = seen + (uint32_t)__popc(starts & ((2u << l) - 1u)) - 1u;
        seen += (uint32_t)__popc(starts);
        return (uint32_t)__shfl((int)shift, gbase + (int)row) + at + l;
    }
};

// for_each_row for a group of L lanes sharing one particle (groups aligned in the
// wavefront, l the lane's index in its group): the particle's (cy, cz) pairs are numbered
// t = 0, 1, ... in for_each_row's order, lane l works out the rows of pairs l, l + L, ...
// (geometry and cell-table entries), and the group then takes the rows' candidates in order,
// L at a time and a row's rest by itself: f(k, q, valid) is called by all lanes of the group
// together, lane l with the candidate k = k0 + l + L m of the row and q = pos[k] (valid: k lies
// in the row).  The next batch's positions are loaded before f gets this one's, so a group does
// not wait for each batch in turn.  With 32 lanes, which rows rarely fill, the rows of one pass
// over t are laid end to end and taken L at a time across their bounds; a lane finds its row from
// the places where rows start, without LDS memory (20-step gradients of 16,384 particles
// 1.575 -> 1.51 ms; with 16 lanes it lost 6% over the 64-box batch).
// AT_ONCE > 0: each row is taken by itself, AT_ONCE batches of it loaded together.
// From the tail's start on, without the candidates before the tail's first.  rows(k0, k1) gets the
// lane's own row ranges.
template <int L, int AT_ONCE = 0, typename RowF, typename F>
__device__ __forceinline__ void for_each_batch(float px, float py, float pz, const StepConsts& C,
                                               __amdgpu_buffer_rsrc_t rcs, __amdgpu_buffer_rsrc_t rpos, uint32_t l,
                                               RowF&& rows, F&& f, ListTail tail = ListTail()) {
    const int gbase = (int)((threadIdx.x & 63u) & ~(uint32_t)(L - 1));
    const RowGrid R(px, py, pz, C);
    const int ny = R.yhi - R.ylo + 1;
    const int npairs = ny * (R.zhi - R.zlo + 1);
    const float inv_ny = 1.0f / (float)ny;
    constexpr uint64_t group = L == 64 ? ~0ull : (1ull << (L & 63)) - 1ull;
    for (int t0 = ny * (max(tail.cz, R.zlo) - R.zlo) + max(tail.cy, R.ylo) - R.ylo; t0 < npairs; t0 += L) {
        uint32_t a0 = 0u, a1 = 0u;
        const int t = t0 + (int)l;
        if (t < npairs) {
            const int q = (int)(((float)t + 0.5f) * inv_ny);  // exact: t and ny are small
            const int cz = R.zlo + q, cy = R.ylo + (t - q * ny);
            const int row0 = C.cell_off + C.dims[0] * (cy + C.dims[1] * cz);
            uint32_t q0, q1;
            if (R.row(cy, R.rest_z(cz, C), C, q0, q1)) {
                RowGrid::range(row0, q0, q1, C, [&](int c) { return ld_u32(rcs, (uint32_t)c * 4u); }, a0, a1);
                a0 = min(max(a0, tail.k), a1);
                if (a0 < a1) rows(a0, a1);
            }
        }
        uint64_t left = (__ballot(a0 < a1) >> gbase) & group;  // the rows that hold candidates
        if constexpr (L == 32) {
            const RowWindows<L> line(a0, a1, l, gbase);
            if (line.total == 0u) continue;
            uint32_t seen = 0u;
            uint32_t k = line.window(seen, 0u);
            float4 q = ld_f4(rpos, k * 16u);
            for (uint32_t at = 0u; at < line.total; at += L) {
                const uint32_t kc = k;
                const float4 qc = q;
                if (at + L < line.total) {
                    k = line.window(seen, at + L);
                    q = ld_f4(rpos, k * 16u);
                }
                f(kc, qc, at + l < line.total);
            }
            continue;
        }
        if constexpr (AT_ONCE == 1) {
            for (int j = 0; j < min(L, npairs - t0); ++j) {
                const uint32_t k0 = __shfl(a0, gbase + j), k1 = __shfl(a1, gbase + j);
                for (uint32_t b = k0; b < k1; b += L) {
                    const uint32_t k = b + l;
                    f(k, ld_f4(rpos, k * 16u), k < k1);
                }
            }
            continue;
        }
        if constexpr (AT_ONCE > 1) {
            while (left != 0ull) {
                const int j = gbase + __ffsll((unsigned long long)left) - 1;
                left &= left - 1ull;
                const uint32_t k0 = __shfl(a0, j) + l, k1 = __shfl(a1, j);
                for (uint32_t k = k0; k - l < k1; k += (uint32_t)(AT_ONCE * L)) {
                    float4 q[AT_ONCE];
#pragma unroll
                    for (int u = 0; u < AT_ONCE; ++u) q[u] = ld_f4(rpos, (k + (uint32_t)(u * L)) * 16u);
#pragma unroll
                    for (int u = 0; u < AT_ONCE; ++u) f(k + (uint32_t)(u * L), q[u], k + (uint32_t)(u * L) < k1);
                }
            }
            continue;
        }
        uint32_t b = 0u, e = 0u;
        auto next_row = [&]() {
            const int j = gbase + __ffsll((unsigned long long)left) - 1;
            left &= left - 1ull;
            b = __shfl(a0, j);
            e = __shfl(a1, j);
        };
        if (left == 0ull) continue;
        next_row();
        float4 q = ld_f4(rpos, min(b + l, e - 1u) * 16u);
        while (true) {
            const uint32_t k = b + l;
            const float4 qk = q;
            const bool valid = k < e;
            b += L;
            bool more = true;
            if (b >= e) {
                more = left != 0ull;
                if (more) next_row();
            }
            if (more) q = ld_f4(rpos, min(b + l, e - 1u) * 16u);
            f(k, qk, valid);
            if (!more) break;
        }
    }
}

// The batches that a scan of a particle's candidates in place of its list, by the force pass and the
// pullbacks, takes at once (for_each_batch): it meets rows of many batches, and few lanes wait on each
// load.  Step and 4-step gradients of a box with 300 and 250 neighbours, looking one batch ahead and
// with this, 2 lanes of 4,099 particles 413 -> 357 us and 8,192 4.11 -> 3.44 ms, 4 lanes 189 -> 170 and
// 2.10 -> 1.75, 8 lanes 102 -> 95 and 1.20 -> 1.09 (as many as one per lane before: 396 and 3.74, 191
// and 2.00, 108 and 1.22).
template <int L>
constexpr int kScanAtOnce = L <= 4 ? 3 : L == 8 ? 2 : 0;

__device__ __forceinline__ float lane_of(float v, int lane) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(v), lane));
}

// The candidate rows of the P particles that share a wavefront, 64 / P lanes each: a row runs from
// the first to the last x slab that any of them reaches, so that each candidate is loaded once
// and tested against all P.  The passes over dense particles are bound by the L1 data path (its
// return path was busy 98% of the time with a load per pair).  ok: all P lie within about a cell of
// each other and have at most 64 rows, one per lane.
// With 16 lanes only, which dense instances get (us per step, density and force, before and
// after: 51,680 particles of 2,626 neighbours 188 and 258 -> 137 and 211, 43,010 of 1,086 117 and
// 161 -> 67 and 94, the 64-box batch 606 and 702 -> 508 and 578).
// 8 lanes gained nothing (95,162 particles of 295 neighbours 115 and 154 -> 118 and 146, the force
// kernel at 77 registers) and lost in the density pass with 4 (142 -> 165).
template <int L>
constexpr bool kSharesRows = L == 16;

template <int P>
struct SharedRows {
    uint32_t k0 = 0u, k1 = 0u;  // the lane's row
    bool ok;

    __device__ __forceinline__ SharedRows(float4 p, const StepConsts& C, __amdgpu_buffer_rsrc_t rcs) {
        const RowGrid R(p.x, p.y, p.z, C);
        int ylo = R.ylo, yhi = R.yhi, zlo = R.zlo, zhi = R.zhi;
        float xlo = R.fx, xhi = R.fx;
#pragma unroll
        for (int j = 0; j < P; ++j) {
            const int at = j * (64 / P);
            ylo = min(ylo, __builtin_amdgcn_readlane(R.ylo, at));
            yhi = max(yhi, __builtin_amdgcn_readlane(R.yhi, at));
            zlo = min(zlo, __builtin_amdgcn_readlane(R.zlo, at));
            zhi = max(zhi, __builtin_amdgcn_readlane(R.zhi, at));
            xlo = fminf(xlo, lane_of(R.fx, at));
            xhi = fmaxf(xhi, lane_of(R.fx, at));
        }
        const int ny = yhi - ylo + 1, rows = ny * (zhi - zlo + 1);
        const bool near = yhi - ylo <= R.yhi - R.ylo + 1 && zhi - zlo <= R.zhi - R.zlo + 1 &&
                          xhi - xlo <= (float)(2 << C.slab_shift);
        ok = __ballot(near && rows <= 64) == ~0ull;
        if (!ok) return;
        const int t = (int)(threadIdx.x & 63u);
        const int cz = zlo + t / ny, cy = ylo + t % ny;
        uint32_t q0 = 0xffffffffu, q1 = 0u;
#pragma unroll
        for (int j = 0; j < P; ++j) {
            const int at = j * (64 / P);
            const RowGrid one(lane_of(p.x, at), lane_of(p.y, at), lane_of(p.z, at), C);
            uint32_t a, b;
            if (t < rows && one.row(cy, one.rest_z(cz, C), C, a, b)) {
                q0 = min(q0, a);
                q1 = max(q1, b);
            }
        }
        if (q0 < q1)
            RowGrid::range(C.cell_off + C.dims[0] * (cy + C.dims[1] * cz), q0, q1, C,
                           [&](int c) { return ld_u32(rcs, (uint32_t)c * 4u); }, k0, k1);
    }

    // f(k, ld(k), valid) by all 64 lanes together, lane l with the candidates k0 + l + 64 m of
    // each row; the next batch is loaded before f gets this one's
    template <typename LD, typename F>
    __device__ __forceinline__ void walk(LD&& ld, F&& f) const {
        const uint32_t l = threadIdx.x & 63u;
        uint64_t left = __ballot(k0 < k1);
        if (left == 0ull) return;
        uint32_t b, e;
        auto next_row = [&]() {
            const int j = __ffsll((unsigned long long)left) - 1;
            left &= left - 1ull;
            b = (uint32_t)__builtin_amdgcn_readlane((int)k0, j);
            e = (uint32_t)__builtin_amdgcn_readlane((int)k1, j);
        };
        next_row();
        auto next = ld(min(b + l, e - 1u));
        while (true) {
            const uint32_t k = b + l;
            const bool valid = k < e;
            const auto now = next;
            b += 64u;
            bool more = true;
            if (b >= e) {
                more = left != 0ull;
                if (more) next_row();
            }
            if (more) next = ld(min(b + l, e - 1u));
            f(k, now, valid);
            if (!more) break;
        }
    }
};

// ---------------------------------------------------------------------------------------
// Wall collision.  Box: base_kernels.py:75-98.  Pipe: base_kernels.py:56-72, 101-127 and
// util_kernels.py:38-204, in FP32, with the particle's own xoroshiro128+ stream.
// ---------------------------------------------------------------------------------------
__device__ __forceinline__ void collide_box(const StepConsts& C, float& x, float& v, int d) {
    bool bounced = false;
    if (x < 0.0f) { x = C.box_lo_target; bounced = true; }
    if (x > C.space[d]) { x = C.box_hi_target[d]; bounced = true; }
    if (bounced) { v *= -1.0f; v *= C.damp; }
}

struct Vec3 { float x, y, z; };
__device__ __forceinline__ float len3(Vec3 a) { return sqrtf(a.x * a.x + a.y * a.y + a.z * a.z); }
__device__ __forceinline__ float dot3(Vec3 a, Vec3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }

__device__ int pipe_find_segment(const PipeTable& T, int rows, float x) {
    for (int j = 0; j < rows - 1; ++j)
        if (T.row[j][0] <= x && x < T.row[j + 1][0]) return j;
    return -1;
}

__device__ float pipe_radius(const PipeTable& T, float x, int seg) {
    const float r0 = T.row[seg][3], r1 = T.row[seg + 1][3], len = T.row[seg][4];
    if (r0 == r1) return r0;
    if (r0 < r1) {
        const float delta = x - T.xbeg[seg];
        const float tl = len * r0 / (r1 - r0);
        return r0 * (1.0f + delta / tl);
    }
    const float delta = T.xbeg[seg] + len - x;
    const float tl = len * r1 / (r0 - r1);
    return r1 * (1.0f + delta / tl);
}

__device__ bool pipe_out(const PipeTable& T, Vec3 p, int seg) {
    const float yn = p.y - T.row[seg][1], zn = p.z - T.row[seg][2];
    return sqrtf(yn * yn + zn * zn) > pipe_radius(T, p.x, seg);
}

__device__ void pipe_solve_collision(const PipeTable& T, Vec3& p, Vec3& v, int seg) {
    const float sr = T.row[seg][3], er = T.row[seg + 1][3];
    const float yn = p.y - T.row[seg][1], zn = p.z - T.row[seg][2];
    const float hh = sqrtf(yn * yn + zn * zn);
    // calc_edge_vector (util_kernels.py:152-171)
    Vec3 first{T.row[seg][0], yn / hh * sr, zn / hh * sr};
    const Vec3 second{T.row[seg + 1][0], yn / hh * er, zn / hh * er};
    const Vec3 edge{second.x - first.x, second.y - first.y, second.z - first.z};
    first.y += T.row[seg][1];
    first.z += T.row[seg][2];
    // calc_dt (util_kernels.py:113-121) with calc_distance_to_pipe (:124-135)
    const float sl = len3(v), el = len3(edge);
    const Vec3 pv{first.x - p.x, first.y - p.y, first.z - p.z};
    const Vec3 cr{edge.y * pv.z - edge.z * pv.y, edge.z * pv.x - edge.x * pv.z, edge.x * pv.y - edge.y * pv.x};
    const float dist = len3(cr) / el;
    // sin of the angle between v and the wall line.  The reference writes sqrt(1 - cos^2)
    // (util_kernels.py:118); for a particle sliding along a conical wall cos is within 1e-8
    // of 1, which FP32 rounds above 1 (sqrt of a negative: NaN).  |v x edge| / (|v| |edge|)
    // is the same quantity and stays accurate at small angles.
    const Vec3 ve{v.y * edge.z - v.z * edge.y, v.z * edge.x - v.x * edge.z, v.x * edge.y - v.y * edge.x};
    const float sin_a = len3(ve) / (sl * el);
    const float dt = -(dist / (sin_a + 0.001f)) / sl;
    const Vec3 cp{p.x + v.x * dt, p.y + v.y * dt, p.z + v.z * dt};
    // reflection (util_kernels.py:191-199)
    if (sr == er) {
        v.y = -v.y;
        v.z = -v.z;
    } else {
        const float c = dot3(edge, v) / (el * sl);
        const Vec3 sv{2.0f * edge.x / el * c * sl, 2.0f * edge.y / el * c * sl, 2.0f * edge.z / el * c * sl};
        v = Vec3{sv.x - v.x, sv.y - v.y, sv.z - v.z};
    }
    const Vec3 dd{p.x - cp.x, p.y - cp.y, p.z - cp.z};
    const float way = len3(dd);
    const float svl = len3(v);
    p = Vec3{cp.x + v.x * way / svl, cp.y + v.y * way / svl, cp.z + v.z * way / svl};
}

// xoroshiro128+ (Blackman & Vigna 2016; rotations 55, 14, 36) and the 53-bit uniform of
// numba.cuda.random.xoroshiro128p_uniform_float64, rounded once to FP32.
__device__ __forceinline__ uint64_t rotl64(uint64_t x, int k) { return (x << k) | (x >> (64 - k)); }
__device__ __forceinline__ uint64_t xoro_next(uint64_t& s0, uint64_t& s1) {
    const uint64_t a = s0;
    uint64_t b = s1;
    const uint64_t result = a + b;
    b ^= a;
    s0 = rotl64(a, 55) ^ b ^ (b << 14);
    s1 = rotl64(b, 36);
    return result;
}
__device__ __forceinline__ float xoro_uniform(uint64_t& s0, uint64_t& s1) {
    return (float)(double)(xoro_next(s0, s1) >> 11) * 0x1p-53f;
}

__device__ void collide_pipe(const StepConsts& C, const PipeTable& T, Vec3& p, Vec3& v, uint64_t* __restrict__ rng,
                             uint32_t pid) {
    const int rows = C.pipe_rows;
    const int seg = pipe_find_segment(T, rows, p.x);
    if (seg == -1) {
        // put_particle_at_pipe_begin (base_kernels.py:115-127)
        if (p.x < 0.0f) {
            p.x = -p.x;
            v.x = -v.x;
            if (pipe_out(T, p, 0)) pipe_solve_collision(T, p, v, 0);
        } else {
            p.x = 0.0f;
            // rand_position_inside_pipe (base_kernels.py:101-112); a pipe that does not start
            // at x <= 0 has no segment here and the reference reads past its table, so this
            // uses segment 0 instead
            int s0g = pipe_find_segment(T, rows, p.x);
            if (s0g < 0) s0g = 0;
            const float R = pipe_radius(T, p.x, s0g);
            uint64_t a = rng[2 * (uint64_t)pid], b = rng[2 * (uint64_t)pid + 1];
            const float r = R * sqrtf(xoro_uniform(a, b));
            const float theta = xoro_uniform(a, b) * 2.0f * 3.14159265358979f;
            rng[2 * (uint64_t)pid] = a;
            rng[2 * (uint64_t)pid + 1] = b;
            p.y = T.row[0][1] + r * cosf(theta);
            p.z = T.row[0][2] + r * sinf(theta);
        }
    } else if (pipe_out(T, p, seg)) {
        pipe_solve_collision(T, p, v, seg);
    }
}

// Symplectic Euler (base_kernels.py:30-53) before the wall collision: result force f,
// new velocity v and new position x.
struct Integrated {
    Vec3 f, v, x;
};
__device__ __forceinline__ Integrated integrate_particle(const StepConsts& C, float4 p, float4 v, float rho, Vec3 P,
                                                         Vec3 V) {
    Integrated r;
    r.f = Vec3{C.ext[0] + -P.x + V.x, C.ext[1] + -P.y + V.y, C.ext[2] + -P.z + V.z};
    r.v = Vec3{v.x + r.f.x / rho * C.dt, v.y + r.f.y / rho * C.dt, v.z + r.f.z / rho * C.dt};
    r.x = Vec3{p.x + r.v.x * C.dt, p.y + r.v.y * C.dt, p.z + r.v.z * C.dt};
    return r;
}

// Whether collide_box moves component d of a position x (the same two tests).
__device__ __forceinline__ bool box_bounced(const StepConsts& C, float x, int d) {
    const bool below = x < 0.0f;
    return below || (below ? C.box_lo_target : x) > C.space[d];
}

// Symplectic Euler (base_kernels.py:30-53), collision, output in the same sorted slot of
// posB/velB, hash of the new position for the next step (SLOT_KEYS: see hash_particle);
// returns the key.
template <int MODE, bool SLOT_KEYS>
__device__ __forceinline__ uint32_t finish_particle(const StepConsts& C, int i, float4 p, float4 v, uint32_t pid,
                                                    float rho, Vec3 P, Vec3 V, float4* __restrict__ posOut,
                                                    float4* __restrict__ velOut, uint32_t* __restrict__ pidOut,
                                                    uint32_t* __restrict__ keyI, uint32_t* __restrict__ valI,
                                                    uint64_t* __restrict__ rng, const PipeTable* __restrict__ pipe,
                                                    float4* __restrict__ dbgP, float4* __restrict__ dbgV,
                                                    float4* __restrict__ dbgF, uint32_t* __restrict__ flags) {
    const Integrated I = integrate_particle(C, p, v, rho, P, V);
    const float fx = I.f.x, fy = I.f.y, fz = I.f.z;
    Vec3 vv = I.v, pp = I.x;
    if (MODE == SPH_MODE_PIPE) {
        collide_pipe(C, *pipe, pp, vv, rng, pid);
    } else {
        collide_box(C, pp.x, vv.x, 0);
        collide_box(C, pp.y, vv.y, 1);
        collide_box(C, pp.z, vv.z, 2);
    }
    posOut[i] = make_float4(pp.x, pp.y, pp.z, rho);
    velOut[i] = make_float4(vv.x, vv.y, vv.z, 0.0f);
    pidOut[i] = pid;
    if (dbgP) {
        dbgP[i] = make_float4(P.x, P.y, P.z, 0.0f);
        dbgV[i] = make_float4(V.x, V.y, V.z, 0.0f);
        dbgF[i] = make_float4(fx, fy, fz, 0.0f);
    }
    return hash_particle<SLOT_KEYS>(C, pp.x, pp.y, pp.z, pid, (uint32_t)i, keyI, valI, flags);
}

// |d|^2 with its roundings spelled out: the compiler fuses the plain sum of squares around
// different products in different copies of a loop, and the neighbour relation must be the same
// from both particles, the sums the same from every kernel that forms them.
__device__ __forceinline__ float norm2(float dx, float dy, float dz) {
    return __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
}

// Neighbour lists.  Slots t and t + 1 (t even) of particle i share the 32-bit word (t / 2) * n
// + i, so a lane reads two slots per load and consecutive particles' words are contiguous.  A
// slot holds the low 16 bits of the neighbour's cell-ordered index minus the particle's own;
// the word nn[i] says how they are completed:
//   <= kListCap   the count; every neighbour lies within [i - 2^15, i + 2^15), so any slot can
//                 be decoded by itself (list_decode).
//   kSeqList set  built with one lane per particle where neighbours lie farther: the count in the
//                 low kSeqCountBits bits, above them how far before i its first candidate lies.
//                 Indices increase along the list by less than 2^16 from one neighbour to the
//                 next, so a walk from the first candidate on restores them (SeqWalk).  A 4.2M
//                 particle dam break, whose layers of cells hold 33,000 particles each, left
//                 its particles to a rescan without this: force 1,115 us per launch.
//   <= kTailCount the count, more than there are slots: the first kListCap neighbours are listed,
//                 within the window; the others are among the candidates after the last of
//                 them, in its row of cells and the rows after it (ListTail).  A reader with one
//                 lane per particle scans all candidates instead: the walk's second loop costs
//                 the force pass registers it cannot spare (1M dam break, 59 -> 62 us).
//   else          no list: the particle's candidates are scanned again, by a reader with several
//                 lanes per particle also in place of a kSeqList walk.
constexpr uint32_t kSeqList = 0x80000000u;
constexpr uint32_t kNoList = 0x7fffffffu;
constexpr int kSeqCountBits = 10;
constexpr uint32_t kSeqMaxBack = 1u << (31 - kSeqCountBits);
constexpr uint32_t kListWindow = 1u << 15;
// Past twice the slots most candidates lie after the list: one scan of all is cheaper then (the
// dense instances of the 64-box batch, 2,000 neighbours: force 1,082 us against 1,162 with their
// lists walked first; the 16,384-particle box, 102 neighbours, at 32 lanes: force 15.0 us with the
// list against 19.6, pullback 26.8 against 32.4).
constexpr uint32_t kTailCount = 2u * (uint32_t)kListCap;
static_assert(kListCap < (1 << kSeqCountBits), "the count fits its field");
__device__ __forceinline__ uint32_t seq_head(uint32_t cnt, uint32_t back) {
    return kSeqList | (back << kSeqCountBits) | cnt;
}
__device__ __forceinline__ uint32_t list_count(uint32_t head) { return head & ((1u << kSeqCountBits) - 1u); }
// The neighbours of a kSeqList list in order: each is the next index after the last whose
// offset from i has the slot's low 16 bits.
struct SeqWalk {
    uint32_t d;  // offset of the last neighbour; at first, of the first candidate
    int i;
    __device__ __forceinline__ SeqWalk(uint32_t head, int i_) : d(0u - ((head & ~kSeqList) >> kSeqCountBits)), i(i_) {}
    __device__ __forceinline__ uint32_t next(uint32_t e) {
        d += (uint32_t)(uint16_t)(e - d);
        return (uint32_t)i + d;
    }
};
__device__ __forceinline__ ListEntry list_encode(uint32_t k, int i) { return (ListEntry)(uint16_t)((int)k - i); }
__device__ __forceinline__ uint32_t list_decode(ListEntry e, int i) { return (uint32_t)(i + (int)(int16_t)e); }
__device__ __forceinline__ size_t list_at(int n, int i, uint32_t t) {
    return ((size_t)(t >> 1) * (size_t)n + (size_t)i) * 2u + (t & 1u);
}

// Pressure and viscosity sums of one pair (naive_kernels.py:38-52, :70-77) without the
// constant factors.  q = (x, y, z, p) and vj = (vx, vy, vz, 1/rho) of the neighbour.
struct PairSums {
    float ax = 0.f, ay = 0.f, az = 0.f, bx = 0.f, by = 0.f, bz = 0.f;
    // self = the pair is the particle itself: 1/r is taken as 0, which makes both terms zero
    // (the pressure term carries a factor 1/r, the viscosity term a factor v_j - v_i = 0).
    // 1/r is the hardware reciprocal square root: rsqrtf gives the same for every r^2 above
    // the FP32 denormal range and only rescales below it (distances under 1e-19).
    __device__ __forceinline__ void add(const StepConsts& C, float4 p, float4 v, float4 q, float4 vj,
                                        bool self = false) {
        const float dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
        const float r2 = norm2(dx, dy, dz);
        const float rinv = self ? 0.0f : __builtin_amdgcn_rsqf(r2);
        const float hr = C.h - r2 * rinv;
        const float cp = (p.w + q.w) * vj.w * hr * hr * rinv;
        ax += cp * dx;
        ay += cp * dy;
        az += cp * dz;
        const float cv = hr * vj.w;
        bx += cv * (vj.x - v.x);
        by += cv * (vj.y - v.y);
        bz += cv * (vj.z - v.z);
    }
};

// List slots (and their neighbour gathers) in flight per lane in the force pass.
#ifndef SPH_FORCE_UNROLL
#define SPH_FORCE_UNROLL 4
#endif
constexpr int kForceUnroll = SPH_FORCE_UNROLL;

// Pressure and viscosity sums of particle i over its neighbour list (or, for a particle
// with more neighbours than list slots, a rescan of its candidates).  The list holds the
// particle itself; PairSums gives that pair a zero contribution.
__device__ __forceinline__ PairSums naive_pair_sums(const StepConsts& C, int i, int n, float4 p, float4 v,
                                                    const float4* __restrict__ pos, const float4* __restrict__ vel,
                                                    const uint32_t* __restrict__ cs, const ListEntry* __restrict__ nl,
                                                    const uint32_t* __restrict__ nn) {
    const __amdgpu_buffer_rsrc_t rpos = make_rsrc(pos, (uint32_t)n * 16u);
    const __amdgpu_buffer_rsrc_t rvel = make_rsrc(vel, (uint32_t)n * 16u);
    PairSums S;
    const uint32_t head = nn[i];
    const uint32_t cnt = list_count(head);
    // two slots per 32-bit load (list_at); the next four slots are loaded while this group's
    // neighbours are gathered, so each group waits on one memory latency
    static_assert(kForceUnroll == 4, "the force pass walks the list four slots at a time");
    auto walk = [&](auto&& decode) {
        const uint32_t* words = reinterpret_cast<const uint32_t*>(nl) + i;
        const size_t stride = (size_t)n;
        uint32_t t = 0;
        uint32_t wn0 = 0u, wn1 = 0u;
        if (cnt >= 4u) {
            wn0 = words[0];
            wn1 = words[stride];
        }
        for (; t + 4u <= cnt; t += 4u) {
            const uint32_t w0 = wn0, w1 = wn1;
            words += 2 * stride;
            if (t + 8u <= cnt) {
                wn0 = words[0];
                wn1 = words[stride];
            }
            uint32_t k[4];
            k[0] = decode(w0);
            k[1] = decode(w0 >> 16);
            k[2] = decode(w1);
            k[3] = decode(w1 >> 16);
            float4 q[4], w[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                q[u] = ld_f4(rpos, k[u] * 16u);
                w[u] = ld_f4(rvel, k[u] * 16u);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) S.add(C, p, v, q[u], w[u], k[u] == (uint32_t)i);
        }
        for (; t < cnt; t += 2u) {  // the last one to three slots, a word at a time
            const uint32_t wd = words[0];
            words += stride;
            const uint32_t k0 = decode(wd);
            S.add(C, p, v, ld_f4(rpos, k0 * 16u), ld_f4(rvel, k0 * 16u), k0 == (uint32_t)i);
            if (t + 1u < cnt) {
                const uint32_t k1 = decode(wd >> 16);
                S.add(C, p, v, ld_f4(rpos, k1 * 16u), ld_f4(rvel, k1 * 16u), k1 == (uint32_t)i);
            }
        }
    };
    if (head <= (uint32_t)kListCap) {
        walk([&](uint32_t e) { return list_decode((ListEntry)e, i); });
    } else if (head & kSeqList) {
        SeqWalk at(head, i);
        walk([&](uint32_t e) { return at.next(e); });
    } else {
        for_each_candidate(p.x, p.y, p.z, C, cs, [&](uint32_t k) {
            const float4 q = pos[k];
            const float dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
            if (norm2(dx, dy, dz) <= C.h2 && k != (uint32_t)i) S.add(C, p, v, q, vel[k]);
        });
    }
    return S;
}

// The sums of the 64 / L particles that share a wavefront, over rows that they share: every lane
// tests its candidate against each of them.
template <int L>
__device__ __forceinline__ PairSums shared_pair_sums(const SharedRows<64 / L>& rows, const StepConsts& C, int i,
                                                     float4 p, float4 v, __amdgpu_buffer_rsrc_t rpos,
                                                     __amdgpu_buffer_rsrc_t rvel) {
    constexpr int P = 64 / L;
    struct Pair { float4 q, v; };
    PairSums S[P];
    float4 ps[P], vs[P];  // the particles', the same in all lanes
    uint32_t is[P];
#pragma unroll
    for (int j = 0; j < P; ++j) {
        const int at = j * L;
        ps[j] = make_float4(lane_of(p.x, at), lane_of(p.y, at), lane_of(p.z, at), lane_of(p.w, at));
        vs[j] = make_float4(lane_of(v.x, at), lane_of(v.y, at), lane_of(v.z, at), 0.0f);
        is[j] = (uint32_t)__builtin_amdgcn_readlane(i, at);
    }
    rows.walk([&](uint32_t k) { return Pair{ld_f4(rpos, k * 16u), ld_f4(rvel, k * 16u)}; },
              [&](uint32_t k, const Pair& c, bool valid) {
#pragma unroll
                  for (int j = 0; j < P; ++j)
                      if (valid && norm2(ps[j].x - c.q.x, ps[j].y - c.q.y, ps[j].z - c.q.z) <= C.h2 && k != is[j])
                          S[j].add(C, ps[j], vs[j], c.q, c.v);
              });
    PairSums mine;
    const int own = (int)(threadIdx.x & 63u) / L;
#pragma unroll
    for (int j = 0; j < P; ++j) {
        const PairSums t{group_sum<64>(S[j].ax), group_sum<64>(S[j].ay), group_sum<64>(S[j].az),
                         group_sum<64>(S[j].bx), group_sum<64>(S[j].by), group_sum<64>(S[j].bz)};
        if (j == own) mine = t;
    }
    return mine;
}

// The same sums with L lanes per particle (L = 1 is naive_pair_sums): lane l of the group
// walks list slots l, l + L, ... (and, past the list, every L-th candidate of each row), and
// the partial sums are added across the group; every lane of the group returns the total.
template <int L>
__device__ __forceinline__ PairSums naive_pair_sums_lanes(const StepConsts& C, int i, uint32_t l, int n, float4 p,
                                                          float4 v, const float4* __restrict__ pos,
                                                          const float4* __restrict__ vel,
                                                          const uint32_t* __restrict__ cs,
                                                          const ListEntry* __restrict__ nl,
                                                          const uint32_t* __restrict__ nn) {
    if constexpr (L == 1) {
        return naive_pair_sums(C, i, n, p, v, pos, vel, cs, nl, nn);
    } else {
        const __amdgpu_buffer_rsrc_t rpos = make_rsrc(pos, (uint32_t)n * 16u);
        const __amdgpu_buffer_rsrc_t rvel = make_rsrc(vel, (uint32_t)n * 16u);
        PairSums S;
        const uint32_t head = nn[i];
        if constexpr (kSharesRows<L>) {
            if (__ballot(head == kNoList) == ~0ull) {
                const __amdgpu_buffer_rsrc_t rcs =
                    make_rsrc(cs, ((uint32_t)C.cell_off + (uint32_t)C.n_cells + 1u) * 4u);
                const SharedRows<64 / L> rows(p, C, rcs);
                if (rows.ok) return shared_pair_sums<L>(rows, C, i, p, v, rpos, rvel);
            }
        }
        const uint32_t cnt = head < kNoList ? min(head, (uint32_t)kListCap) : 0u;
        // the lane's next list slot is loaded while this slot's neighbour is gathered
        uint32_t kn = l < cnt ? list_decode(nl[list_at(n, i, l)], i) : 0u;
        for (uint32_t t = l; t < cnt; t += L) {
            const uint32_t k = kn;
            if (t + L < cnt) kn = list_decode(nl[list_at(n, i, t + L)], i);
            S.add(C, p, v, ld_f4(rpos, k * 16u), ld_f4(rvel, k * 16u), k == (uint32_t)i);
        }
        if (head > (uint32_t)kListCap) {
            const __amdgpu_buffer_rsrc_t rcs = make_rsrc(cs, ((uint32_t)C.cell_off + (uint32_t)C.n_cells + 1u) * 4u);
            ListTail tail;
            if (head < kNoList) {
                const uint32_t last = list_decode(nl[list_at(n, i, kListCap - 1)], i);
                tail = ListTail(last, ld_f4(rpos, last * 16u), C);
            }
            for_each_batch<L, kScanAtOnce<L>>(
                p.x, p.y, p.z, C, rcs, rpos, l, [](uint32_t, uint32_t) {},
                [&](uint32_t k, float4 q, bool valid) {
                    const float dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
                    if (valid && norm2(dx, dy, dz) <= C.h2 && k != (uint32_t)i)
                        S.add(C, p, v, q, ld_f4(rvel, k * 16u));
                },
                tail);
        }
        S.ax = group_sum<L>(S.ax);
        S.ay = group_sum<L>(S.ay);
        S.az = group_sum<L>(S.az);
        S.bx = group_sum<L>(S.bx);
        S.by = group_sum<L>(S.by);
        S.bz = group_sum<L>(S.bz);
        return S;
    }
}

// The sums of naive_pair_sums, to the same bits, by a group of L >= 8 lanes: the lanes work out the
// terms of L pairs, keep them in LDS, and lanes 0 .. 5 each add one component of them up in the
// list's (or the scan's) order.  buf: the group's kOrderedPairWords<L> words of LDS: per pair
// the two coefficients and the components they multiply, kept apart by an odd pitch so that
// the six lanes read six banks.
template <int L>
constexpr uint32_t kOrderedPitch = (uint32_t)L + 1u;
template <int L>
constexpr uint32_t kOrderedPairWords = 8u * kOrderedPitch<L>;
template <int L>
__device__ __forceinline__ PairSums naive_pair_sums_ordered(const StepConsts& C, int i, uint32_t l, int n, float4 p,
                                                            float4 v, const float4* __restrict__ pos,
                                                            const float4* __restrict__ vel,
                                                            const uint32_t* __restrict__ cs,
                                                            const ListEntry* __restrict__ nl,
                                                            const uint32_t* __restrict__ nn, float* buf) {
    static_assert(L >= 8, "six lanes add");
    const __amdgpu_buffer_rsrc_t rpos = make_rsrc(pos, (uint32_t)n * 16u);
    const __amdgpu_buffer_rsrc_t rvel = make_rsrc(vel, (uint32_t)n * 16u);
    constexpr uint32_t kPitch = kOrderedPitch<L>;
    const int gbase = (int)((threadIdx.x & 63u) & ~(uint32_t)(L - 1));
    const uint32_t comp = l < 6u ? l : 5u;
    const float* const coef = buf + (comp < 3u ? 0u : kPitch);
    const float* const part = buf + (2u + comp) * kPitch;
    float acc = 0.0f;
    // the terms of one pair (PairSums::add) into place `at`
    auto keep = [&](float4 q, float4 vj, bool self, uint32_t at) {
        const float dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
        const float r2 = norm2(dx, dy, dz);
        const float rinv = self ? 0.0f : __builtin_amdgcn_rsqf(r2);
        const float hr = C.h - r2 * rinv;
        buf[at] = (p.w + q.w) * vj.w * hr * hr * rinv;
        buf[kPitch + at] = hr * vj.w;
        buf[2u * kPitch + at] = dx;
        buf[3u * kPitch + at] = dy;
        buf[4u * kPitch + at] = dz;
        buf[5u * kPitch + at] = vj.x - v.x;
        buf[6u * kPitch + at] = vj.y - v.y;
        buf[7u * kPitch + at] = vj.z - v.z;
    };
    auto add = [&](uint32_t count) {
        wave_lds_order();
        for (uint32_t t = 0; t < count; ++t) acc += coef[t] * part[t];
        wave_lds_order();
    };
    const uint32_t head = nn[i];
    const uint32_t cnt = head < kNoList ? min(head, (uint32_t)kListCap) : 0u;
    uint32_t kn = l < cnt ? list_decode(nl[list_at(n, i, l)], i) : (uint32_t)i;
    for (uint32_t t = 0; t < cnt; t += L) {
        const uint32_t k = kn;
        const float4 q = ld_f4(rpos, k * 16u), w = ld_f4(rvel, k * 16u);
        if (t + L + l < cnt) kn = list_decode(nl[list_at(n, i, t + L + l)], i);
        keep(q, w, k == (uint32_t)i, l);
        add(min((uint32_t)L, cnt - t));
    }
    if (head > (uint32_t)kListCap) {
        const __amdgpu_buffer_rsrc_t rcs = make_rsrc(cs, ((uint32_t)C.cell_off + (uint32_t)C.n_cells + 1u) * 4u);
        constexpr uint64_t group = L == 64 ? ~0ull : (1ull << (L & 63)) - 1ull;
        ListTail tail;
        if (head < kNoList) {
            const uint32_t last = list_decode(nl[list_at(n, i, kListCap - 1)], i);
            tail = ListTail(last, ld_f4(rpos, last * 16u), C);
        }
        for_each_batch<L>(
            p.x, p.y, p.z, C, rcs, rpos, l, [](uint32_t, uint32_t) {},
            [&](uint32_t k, float4 q, bool valid) {
                const float dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
                const bool hit = valid && norm2(dx, dy, dz) <= C.h2 && k != (uint32_t)i;
                const uint64_t gm = (__ballot(hit) >> gbase) & group;
                if (hit) keep(q, ld_f4(rvel, k * 16u), false, (uint32_t)__popcll(gm & ((1ull << l) - 1ull)));
                add((uint32_t)__popcll(gm));
            },
            tail);
    }
    PairSums S;
    S.ax = __shfl(acc, gbase);
    S.ay = __shfl(acc, gbase + 1);
    S.az = __shfl(acc, gbase + 2);
    S.bx = __shfl(acc, gbase + 3);
    S.by = __shfl(acc, gbase + 4);
    S.bz = __shfl(acc, gbase + 5);
    return S;
}

}  // namespace
}  // namespace sph
