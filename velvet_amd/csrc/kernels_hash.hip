// Spatial-hash build for gfx950: cell hash, stable LSD radix sort, cell start/end and the
// cached neighbour table (Velvet/SpatialHashGPU.cu:13-196).
//
// Segments of up to 2^17 particles are built by cell ranges (k_hash_part). The others are sorted in one
// device-wide pass sequence. Keys are the per-segment hash (< M of that
// segment), values the local particle index. Sort tiles never straddle segments and the
// digit histograms are laid out (segment, digit, tile), so one exclusive scan over the whole
// histogram gives every (segment, digit, tile) its global output offset: the segments come
// out sorted independently, in place, without sorting on segment bits. Ranking inside a tile
// is stable (each wave a contiguous chunk, in wave order; inside a chunk 64 keys at a time by
// wave ballots, in order), so the result equals a stable sort by hash within each segment -- the
// contract of the reference's
// cub::DeviceRadixSort::SortPairs call (Velvet/SpatialHashGPU.cu:133-157).
#include <hip/hip_runtime.h>

#include <cstddef>
#include <mutex>
#include <type_traits>

#include "launch.hpp"
#include "vec.hpp"
#include "vtx_device.hpp"

namespace vtx {


// HashCoords (Velvet/SpatialHashGPU.cu:18-22): 32-bit wrap-around products, then
// abs(h % M). |h % M| == |h| mod M for C's truncating remainder, and the unsigned remainder of
// a <= 2^31 takes one product with m = floor(2^32 / M) (mod_constant): a/M - a m / 2^32 < a / 2^32 <= 1/2,
// so the quotient's floor is right or one too small, and one subtraction mends it.
constexpr uint32_t HX = 92837111u, HY = 689287499u, HZ = 283923481u;

__device__ __forceinline__ uint32_t hash_reduce(uint32_t h, uint32_t M, uint32_t m) {
    const uint32_t a = (int32_t)h < 0 ? 0u - h : h;
    const uint32_t r = a - __umulhi(a, m) * M;
    return min(r, r - M);
}

__device__ __forceinline__ uint32_t hash_coords(int32_t x, int32_t y, int32_t z, uint32_t M, uint32_t m) {
    return hash_reduce(((uint32_t)x * HX) ^ ((uint32_t)y * HY) ^ ((uint32_t)z * HZ), M, m);
}

// ComputeIntCoord (Velvet/SpatialHashGPU.cu:13-16): floor of a correctly rounded binary32
// quotient (the library is built with -fhip-fp32-correctly-rounded-divide-sqrt).
__device__ __forceinline__ int32_t int_coord(float v, float cell) {
    return (int32_t)floorf(__fdiv_rn(v, cell));
}

// The cell of a position, as hashed: ComputeIntCoord plus the grid shift (0 on the reference grid,
// VTX_HASH_SHIFT on a tuned one) with 32-bit wrap-around. t = v times the cell's reciprocal (1 ulp) is
// within 2^-22 |t| of the quotient, so where t is more than 2^-20 |t| away from an integer its floor is
// the rounded quotient's; the division runs for the rest (large, on a cell's face, not finite). A key
// takes 50 VALU issue slots instead of 85.
__device__ __forceinline__ void cell_coords(float4 p, float cell, uint32_t shift, int32_t& x, int32_t& y, int32_t& z) {
    const float inv = __builtin_amdgcn_rcpf(cell);
    const float tx = p.x * inv, ty = p.y * inv, tz = p.z * inv;
    const float fx = floorf(tx), fy = floorf(ty), fz = floorf(tz);
    const float gx = fabsf(tx - fx - 0.5f), gy = fabsf(ty - fy - 0.5f), gz = fabsf(tz - fz - 0.5f);
    constexpr float E = 9.5367431640625e-07f;   // 2^-20
    const bool clear = (gx < 0.5f - E * fabsf(tx)) & (gy < 0.5f - E * fabsf(ty)) & (gz < 0.5f - E * fabsf(tz));
    int32_t cx = (int32_t)fx, cy = (int32_t)fy, cz = (int32_t)fz;
    if (!clear) {
        cx = int_coord(p.x, cell);
        cy = int_coord(p.y, cell);
        cz = int_coord(p.z, cell);
    }
    x = (int32_t)((uint32_t)cx + shift);
    y = (int32_t)((uint32_t)cy + shift);
    z = (int32_t)((uint32_t)cz + shift);
}

__device__ __forceinline__ uint32_t position_key(float4 p, float cell, uint32_t shift, uint32_t M, uint32_t m) {
    int32_t x, y, z;
    cell_coords(p, cell, shift, x, y, z);
    return hash_coords(x, y, z, M, m);
}

__device__ __forceinline__ uint32_t seg_shift(const SegDev& sg) {
    return (sg.flags & VTX_SEG_HASH_SHIFT) ? VTX_HASH_SHIFT : 0u;
}

// ComputeParticleHash_Kernel (Velvet/SpatialHashGPU.cu:34-42) over predicted positions.
// Segments that k_hash_part builds get theirs where it reads them: dst = the side its results go to.
__global__ __launch_bounds__(VTX_TILE) void k_hash_keys(DevState d, int in, int dst) {
    const TileDev t = d.tiles[tile_of(d.remap)];
    if (threadIdx.x >= t.count) return;
    const SegDev sg = d.segs[t.seg];
    const uint32_t g = t.begin + threadIdx.x;
    const bool part = sg.flags & VTX_SEG_HASH_PART;
    if (part && !(sg.flags & VTX_SEG_HASH_KEYED)) return;
    if (!part) d.vals[0][g] = g - sg.pbase;
    if (!(sg.flags & VTX_SEG_SELFCOL)) {
        d.keys[0][g] = 0;      // segment without self-collision: sorted as one cell, unused
        return;
    }
    const float4 p = d.P[in][g];
    const uint32_t sh = seg_shift(sg);
    d.keys[part ? dst ^ 1 : 0][g] = position_key(p, sg.cell, sh, sg.M, sg.mod);
}

// Digit histogram of one sort tile (count keys from `keys`): the count of digit g goes to
// out[g * stride].
__device__ __forceinline__ void tile_hist(const uint32_t* __restrict__ keys, uint32_t count, int shift,
                                          uint32_t* __restrict__ out, uint32_t stride) {
    __shared__ uint32_t cnt[256];
    cnt[threadIdx.x] = 0;
    __syncthreads();
    for (uint32_t r = 0; r < VTX_SORT_ITEMS; r++) {
        const uint32_t i = r * VTX_TILE + threadIdx.x;
        if (i < count) atomicAdd(&cnt[(keys[i] >> shift) & 255u], 1u);
    }
    __syncthreads();
    out[threadIdx.x * stride] = cnt[threadIdx.x];
}

// Per-tile digit histogram into hist[hbase + digit * ntiles + tidx].
__global__ __launch_bounds__(VTX_TILE) void k_sort_hist(DevState d, int src, int shift) {
    const SortTileDev t = d.stiles[blockIdx.x];
    tile_hist(d.keys[src] + t.begin, t.count, shift, d.hist + t.hbase + t.tidx, t.ntiles);
}

// Wave-level exclusive scan helpers (wave64).
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v) {
    const uint32_t lane = threadIdx.x & 63u;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t u = __shfl_up(v, o, 64);
        if (lane >= (uint32_t)o) v += u;
    }
    return v;
}

// Block (256 threads) exclusive scan; returns the exclusive prefix, *total the block sum.
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t* total, uint32_t* sh) {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t incl = wave_incl_scan(v);
    if (lane == 63) sh[wave] = incl;
    __syncthreads();
    uint32_t off = 0, tot = 0;
#pragma unroll
    for (uint32_t w = 0; w < VTX_TILE / 64; w++) {
        const uint32_t s = sh[w];
        off += (w < wave) ? s : 0u;
        tot += s;
    }
    __syncthreads();
    *total = tot;
    return off + incl - v;
}

// Device-wide exclusive scan of hist[0..n) in two launches: block sums, then each block adds
// the sums of the blocks before it (a block reduction over at most a few hundred sums) and
// scans its own elements.
__global__ __launch_bounds__(VTX_TILE) void k_scan_reduce(uint32_t* __restrict__ a, uint32_t n,
                                                          uint32_t* __restrict__ part) {
    __shared__ uint32_t sh[VTX_TILE / 64];
    const uint32_t base = blockIdx.x * VTX_SCAN_BLOCK;
    uint32_t s = 0;
    for (uint32_t r = 0; r < VTX_SCAN_BLOCK / VTX_TILE; r++) {
        const uint32_t i = base + r * VTX_TILE + threadIdx.x;
        if (i < n) s += a[i];
    }
    uint32_t total;
    block_excl_scan(s, &total, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = total;
}

__global__ __launch_bounds__(VTX_TILE) void k_scan_apply(uint32_t* __restrict__ a, uint32_t n,
                                                         const uint32_t* __restrict__ part) {
    __shared__ uint32_t sh[VTX_TILE / 64];
    const uint32_t base = blockIdx.x * VTX_SCAN_BLOCK;
    uint32_t carry = 0;
    for (uint32_t b0 = 0; b0 < blockIdx.x; b0 += VTX_TILE) {   // sums of the earlier blocks
        const uint32_t b = b0 + threadIdx.x;
        uint32_t total;
        block_excl_scan(b < blockIdx.x ? part[b] : 0u, &total, sh);
        carry += total;
    }
    for (uint32_t r = 0; r < VTX_SCAN_BLOCK / VTX_TILE; r++) {
        const uint32_t i = base + r * VTX_TILE + threadIdx.x;
        const uint32_t v = i < n ? a[i] : 0u;
        uint32_t total;
        const uint32_t ex = block_excl_scan(v, &total, sh);
        if (i < n) a[i] = carry + ex;
        carry += total;
    }
}

// Stable scatter of one sort tile (count keys and values from kin / vin). Wave w owns the tile's
// contiguous chunk w of count / 4 keys: it counts its chunk's digits with LDS atomics (order does
// not matter), each digit's start then runs through the waves in order from the tile's base
// (digit g of the tile starts at output position scanned[g * stride] + bias), and each wave
// scatters its chunk in order, 64 keys at a time ranked by ballots over the 8 digit bits, moving
// its own per-digit offsets on: chunks in wave order and keys in chunk order keep the sort
// stable, with two workgroup barriers per tile.
__device__ __forceinline__ void tile_scatter(const uint32_t* __restrict__ kin, const uint32_t* __restrict__ vin,
                                             uint32_t count, int shift, const uint32_t* __restrict__ scanned,
                                             uint32_t stride, uint32_t bias, uint32_t* __restrict__ kout,
                                             uint32_t* __restrict__ vout) {
    constexpr uint32_t NW = VTX_TILE / 64;
    __shared__ uint32_t wcnt[NW][256];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t chunk = (count + NW - 1) / NW;
    const uint32_t c0 = min(wave * chunk, count), c1 = min(c0 + chunk, count);
    uint32_t* __restrict__ hw = wcnt[wave];
    for (uint32_t k = lane; k < 256; k += 64) hw[k] = 0;
    __builtin_amdgcn_wave_barrier();
    for (uint32_t i = c0 + lane; i < c1; i += 64) atomicAdd(&hw[(kin[i] >> shift) & 255u], 1u);
    __syncthreads();
    {   // thread tid = digit: the waves' starts in wave order
        uint32_t run = scanned[tid * stride] + bias;
#pragma unroll
        for (uint32_t w = 0; w < NW; w++) {
            const uint32_t c = wcnt[w][tid];
            wcnt[w][tid] = run;
            run += c;
        }
    }
    __syncthreads();
    const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    for (uint32_t r0 = c0; r0 < c1; r0 += 64) {
        const uint32_t i = r0 + lane;
        const bool valid = i < c1;
        const uint32_t key = valid ? kin[i] : 0u;
        const uint32_t val = valid ? vin[i] : 0u;
        const uint32_t dg = (key >> shift) & 255u;
        uint64_t peers = __builtin_amdgcn_ballot_w64(valid);
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const uint32_t m = (uint32_t)((int32_t)(dg << (31 - b)) >> 31);   // bit b as 0 / ~0
            const uint64_t bal = __builtin_amdgcn_ballot_w64(m != 0u);
            peers &= ~(bal ^ ((uint64_t)m << 32 | m));                        // lanes whose bit b is this lane's
        }
        const uint32_t rank = (uint32_t)__popcll(peers & lt);
        const uint32_t at = hw[dg];
        if (valid) {
            kout[at + rank] = key;
            vout[at + rank] = val;
        }
        __builtin_amdgcn_wave_barrier();
        if (valid && rank == 0) hw[dg] = at + (uint32_t)__popcll(peers);
        __builtin_amdgcn_wave_barrier();
    }
}

__global__ __launch_bounds__(VTX_TILE) void k_sort_scatter(DevState d, int src, int shift) {
    const SortTileDev t = d.stiles[blockIdx.x];
    tile_scatter(d.keys[src] + t.begin, d.vals[src] + t.begin, t.count, shift, d.hist + t.hbase + t.tidx, t.ntiles,
                 t.bias, d.keys[src ^ 1], d.vals[src ^ 1]);
}

__global__ void k_fill_u32(uint32_t* __restrict__ a, uint32_t n, uint32_t v) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) a[i] = v;
}

// Mark every cell of every self-colliding segment empty: lane i of a segment clears cells
// i, i + n, i + 2n, ... < M (the reference's memset, Velvet/SpatialHashGPU.cu:185).
__global__ __launch_bounds__(VTX_TILE) void k_clear_cells(DevState d) {
    const TileDev t = d.tiles[tile_of(d.remap)];
    if (threadIdx.x >= t.count) return;
    const SegDev sg = d.segs[t.seg];
    if (!(sg.flags & VTX_SEG_SELFCOL) || (sg.flags & VTX_SEG_HASH_PART)) return;
    uint2* __restrict__ cells = d.cells + sg.tbase;
    for (uint32_t i = t.begin - sg.pbase + threadIdx.x; i < sg.M; i += sg.n) cells[i] = make_uint2(VTX_INVALID, VTX_INVALID);
}

// FindCellStart_Kernel (Velvet/SpatialHashGPU.cu:44-77) per segment with local sorted
// positions (cells were filled with ~0u: empty), plus the inverse permutation (particle ->
// sorted position) in the sort's free key buffer, from which k_sorted_records writes the
// sorted records in particle order, and the number of cells in a sample (SearchRule), left in the sort's free
// value buffer.
__global__ __launch_bounds__(VTX_TILE) void k_cell_bounds(DevState d, int in, int src) {
    const TileDev t = d.tiles[tile_of(d.remap)];
    if (threadIdx.x >= t.count) return;
    const SegDev sg = d.segs[t.seg];
    if (!(sg.flags & VTX_SEG_SELFCOL) || (sg.flags & VTX_SEG_HASH_PART)) return;
    const uint32_t g = t.begin + threadIdx.x;
    const uint32_t local = g - sg.pbase;
    const uint32_t* __restrict__ sk = d.keys[src];
    const uint32_t key = sk[g];
    uint2* __restrict__ cells = d.cells + sg.tbase;
    if (local == 0) {
        cells[key].x = 0;
    } else {
        const uint32_t prev = sk[g - 1];
        if (key != prev) {
            cells[key].x = local;
            cells[prev].y = local;
        }
    }
    if (local == sg.n - 1) cells[key].y = sg.n;
    d.keys[src ^ 1][sg.pbase + d.vals[src][g]] = local;
    if (t.begin == sg.pbase && sg.n > VTX_SEARCH_SAMPLED) {   // the first tile, full: cells of the sample
        constexpr uint32_t R = VTX_SEARCH_SAMPLE / VTX_TILE;
        __shared__ uint32_t wsum[VTX_TILE / 64];
        uint32_t k[R], next[R], count = 0;
#pragma unroll
        for (uint32_t r = 0; r < R; r++) {
            k[r] = sk[sg.pbase + r * VTX_TILE + local];
            next[r] = sk[sg.pbase + r * VTX_TILE + local + 1];
        }
#pragma unroll
        for (uint32_t r = 0; r < R; r++) count += (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(k[r] != next[r]));
        if ((local & 63u) == 0) wsum[local >> 6] = count;
        __syncthreads();
        if (local == 0) d.vals[src ^ 1][sg.pbase] = wsum[0] + wsum[1] + wsum[2] + wsum[3];
    }
}

// The sorted copies for the neighbour search, written from particle order: coalesced reads of the
// predicted and initial positions, one scattered 32-B record per particle (a gather in sorted
// order reads two scattered 16-B halves instead). w of the position copy carries the particle's
// local index (the inverse mass is not needed there). inv = the inverse permutation k_cell_bounds
// left in the sort's free key buffer.
__global__ __launch_bounds__(VTX_TILE) void k_sorted_records(DevState d, int in, int src) {
    const TileDev t = d.tiles[tile_of(d.remap)];
    if (threadIdx.x >= t.count) return;
    const SegDev sg = d.segs[t.seg];
    if (!(sg.flags & VTX_SEG_SELFCOL) || (sg.flags & VTX_SEG_HASH_PART)) return;
    const uint32_t g = t.begin + threadIdx.x;
    const size_t o = 2 * (size_t)(sg.pbase + d.keys[src ^ 1][g]);
    const float4 q = d.P[in][g];
    d.sPX[o] = make_float4(q.x, q.y, q.z, __uint_as_float(g - sg.pbase));
    d.sPX[o + 1] = d.X0[g];
}

template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ uint32_t dpp0(uint32_t v) {   // the source lane's v, 0 where there is none
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false);
}

// Inclusive sum over lanes 0..31 (lanes 32..63: over themselves), inclusive sum and maximum over the wave.
__device__ __forceinline__ uint32_t scan32_add(uint32_t v) {
    v += dpp0<0x111>(v);          // row_shr:1, 2, 4, 8
    v += dpp0<0x112>(v);
    v += dpp0<0x114>(v);
    v += dpp0<0x118>(v);
    return v + dpp0<0x142, 0xa>(v);   // row_bcast:15
}

__device__ __forceinline__ uint32_t scan64_add(uint32_t v) {
    v = scan32_add(v);
    return v + dpp0<0x143, 0xc>(v);   // row_bcast:31
}

__device__ __forceinline__ uint32_t scan64_max(uint32_t v) {
    v = max(v, dpp0<0x111>(v));
    v = max(v, dpp0<0x112>(v));
    v = max(v, dpp0<0x114>(v));
    v = max(v, dpp0<0x118>(v));
    v = max(v, dpp0<0x142, 0xa>(v));
    return max(v, dpp0<0x143, 0xc>(v));   // row_bcast:31
}

// Order LDS accesses of the lanes of one wave (a wave's LDS operations execute in order).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The whole spatial-hash build of one segment of at most VTX_HASH_PART_N particles in one launch (after
// k_hash_keys, see VTX_HASH_PART_KEYS): the table's cells are cut into ranges, and a workgroup builds one
// range on its own. It runs over the keys of all particles, counts those in its range per cell in LDS and
// those below the range (the range's first sorted position), scans the counts, puts the range's particles
// into their cells in any order and finds each one's place inside its cell by counting the cell's smaller
// indices: a stable sort by key, so the same table and records as the device-wide path. Counting a cell
// of c particles costs c^2, so a range with a cell of more than VTX_HASH_HEAVY sorts its list in LDS
// instead, or, if it holds more than the list or few keys are to be run over (VTX_HASH_SORT_MIN: a sort takes
// 13 us, two runs over 1,600 keys 1, over 24,100 3), places such cells by two runs over the keys in index order
// for up to 256 of them at a time (hash_part_runs), so that no input costs quadratic time: 131,072 objects
// with their search, in cells of 100 / 140 / 300 / 2,000 / 6,000: 66 / 80 / 93 / 101 / 166 us, in a table of
// 1,000 cells 94 us (device-wide sort 112 / 111 / 110 / 107 / 104, 96; two runs for each crowded cell 67 / 652 /
// 455 / 265 / 167, 461). All in one cell is one workgroup's work: 330 us (77; 441).
// Bound by latency: a launch's 2.6 us, then the chain range record, keys, LDS counts, scan, placement,
// gathered records, and from 2^15 particles on the two runs over the keys. No workgroup waits for another,
// where the dozen launches of a device-wide sort did and one workgroup per segment with a radix sort in
// LDS took one CU for the whole of it: 4,608 particles 20 -> 8.5 us (one workgroup), 16,384 55 -> 14.4
// (one workgroup; k_hash_keys included, as below), 22,500 49 -> 16 (device-wide), 65,536 73 -> 25,
// 131,044 in a frame of four builds 492 -> 354, 16 cloths of 65,536 1338 -> 1122 a frame of four builds.
struct alignas(16) HashPartLds {           // cnt is read and written four words at a time
    uint32_t cnt[VTX_HASH_PART_CELLS];      // per cell of the range: count, start, end (exclusive)
    uint32_t list[VTX_HASH_PART_LIST + 3];  // the range's particles by cell: cell << 20 | index
    uint32_t heavy[VTX_HASH_PART_N / VTX_HASH_HEAVY];
    uint32_t wsum[16], nheavy, below;
};
static_assert(offsetof(HashPartLds, cnt) % 16 == 0, "cnt is accessed in 16-byte units");

// Whether the wave's lanes (all active) have hit and one value: 64 LDS additions to one word go one by one.
__device__ __forceinline__ bool wave_of(uint32_t k, bool hit) {
    return __builtin_amdgcn_ballot_w64(hit && k == __builtin_amdgcn_readfirstlane(k)) == ~0ull;
}

// Ascending bitonic sort of a[0..m), m a power of two of at least 1. Thread t exchanges a pair 2^b apart;
// for pairs up to 64 apart a wave's threads stay within 128 words of their own, so steps of such pairs
// follow each other without a workgroup barrier.
template <uint32_t BT>
__device__ __forceinline__ void sort_list(uint32_t* a, uint32_t m) {
    for (uint32_t k = 2; k <= m; k <<= 1)
        for (uint32_t j = k >> 1; j; j >>= 1) {
            for (uint32_t t = threadIdx.x; t < m >> 1; t += BT) {
                const uint32_t i = (t & ~(j - 1u)) << 1 | (t & (j - 1u));
                const uint32_t x = a[i], y = a[i | j];
                if ((x > y) == !(i & k)) {
                    a[i] = y;
                    a[i | j] = x;
                }
            }
            if (j > 64u || (j == 1u && k >= 128u)) __syncthreads();   // the next step's pairs: j / 2 or k apart
            else wave_lds_sync();
        }
    __syncthreads();
}

// The cells of more than VTX_HASH_HEAVY particles of a range that holds more than its list, up to 256 (512)
// of them at a time: wave w takes the w-th part of the particles in order, counts its particles per cell,
// then places them behind those of the waves before it, 64 at a time ranked by ballots over the cell's number.
// U times 64 keys are in flight. L.heavy: the cells with their first places.
template <uint32_t BT, uint32_t U, class S>
__device__ __forceinline__ void hash_part_runs(const S& s, uint32_t n, uint32_t lo, uint32_t C, uint32_t base,
                                               uint32_t nheavy, HashPartLds& L) {
    constexpr uint32_t NW = BT / 64, HB = VTX_HASH_PART_LIST / NW;
    constexpr int BITS = HB == 256 ? 8 : 9;
    static_assert(HB == 1u << BITS, "a cell's number among HB");
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    __syncthreads();                                        // the cells' bounds are read
    for (uint32_t k = tid; k < C; k += BT) L.cnt[k] = VTX_INVALID;
    __syncthreads();
    for (uint32_t h = tid; h < nheavy; h += BT) L.cnt[L.heavy[h] & 0xFFFu] = h;
    uint32_t* const hw = L.list + wave * HB;
    const uint32_t chunk = (n + NW - 1) / NW, b = min(wave * chunk, n), e = min(b + chunk, n);
    const uint64_t lt = (1ull << lane) - 1ull;
    for (uint32_t h0 = 0; h0 < nheavy; h0 += HB) {
        const uint32_t nb = min(HB, nheavy - h0);
        for (uint32_t q = lane; q < HB; q += 64) hw[q] = 0;
        __syncthreads();
        uint32_t kk[U], q[U];                               // keys; the cells' numbers, nb or more: none
        const auto load = [&](uint32_t i0) {
#pragma unroll
            for (uint32_t u = 0; u < U; u++) kk[u] = s.key(min(i0 + 64 * u + lane, n - 1u));
#pragma unroll
            for (uint32_t u = 0; u < U; u++) {
                const uint32_t k = kk[u] - lo;
                q[u] = VTX_INVALID;
                if (i0 + 64 * u + lane < e && k < C) q[u] = L.cnt[k] - h0;
            }
        };
        for (uint32_t i0 = b; i0 < e; i0 += 64 * U) {
            load(i0);
#pragma unroll
            for (uint32_t u = 0; u < U; u++)
                if (wave_of(q[u], q[u] < nb)) {
                    if (lane == 0) atomicAdd(&hw[q[u]], 64u);
                } else if (q[u] < nb) {
                    atomicAdd(&hw[q[u]], 1u);
                }
        }
        __syncthreads();
        for (uint32_t h = tid; h < nb; h += BT) {
            uint32_t run = base + (L.heavy[h0 + h] >> 12);
            for (uint32_t w = 0; w < NW; w++) {
                const uint32_t c = L.list[w * HB + h];
                L.list[w * HB + h] = run;
                run += c;
            }
        }
        __syncthreads();
        for (uint32_t i0 = b; i0 < e; i0 += 64 * U) {
            load(i0);
            uint32_t at[U];
#pragma unroll
            for (uint32_t u = 0; u < U; u++) {
                const bool hit = q[u] < nb;
                const uint64_t hits = __builtin_amdgcn_ballot_w64(hit);
                if (!hits) continue;
                const uint32_t f = (uint32_t)__builtin_amdgcn_readlane((int)q[u], __builtin_ctzll(hits));
                uint64_t peers = hits;
                if (hits & ~__builtin_amdgcn_ballot_w64(q[u] == f))   // more than one cell
#pragma unroll
                    for (int c = 0; c < BITS; c++) {
                        const uint32_t m = (uint32_t)((int32_t)(q[u] << (31 - c)) >> 31);   // bit c as 0 / ~0
                        peers &= ~(__builtin_amdgcn_ballot_w64(m != 0u) ^ ((uint64_t)m << 32 | m));
                    }
                const uint32_t rank = (uint32_t)__popcll(peers & lt);
                at[u] = hw[hit ? q[u] : 0u] + rank;
                wave_lds_sync();
                if (hit && rank == 0) hw[q[u]] = at[u] + (uint32_t)__popcll(peers);
                wave_lds_sync();
            }
            float4 p[U], x[U];
#pragma unroll
            for (uint32_t u = 0; u < U; u++)
                if (q[u] < nb) s.get(i0 + 64 * u + lane, p[u], x[u]);
#pragma unroll
            for (uint32_t u = 0; u < U; u++)
                if (q[u] < nb) s.put(at[u], kk[u], i0 + 64 * u + lane, p[u], x[u]);
        }
        __syncthreads();
    }
}

// S: the particles (key(i), put(g, key, i) for sorted position g, cell(k, begin, end)).
template <uint32_t BT, bool KEYED, class S>
__device__ __forceinline__ void hash_part(const S& s, uint32_t n, uint32_t lo, uint32_t C, uint32_t* __restrict__ spill,
                                          HashPartLds& L) {
    constexpr uint32_t NW = BT / 64, U = 8, Q = VTX_HASH_PART_CELLS / (4 * BT);
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
#pragma unroll
    for (uint32_t q = 0; q < Q; q++) reinterpret_cast<uint4*>(L.cnt)[q * BT + tid] = make_uint4(0u, 0u, 0u, 0u);
    if (tid == 0) L.nheavy = L.below = 0u;
    __syncthreads();
    // counts
    uint32_t kk[U], below = 0;
    const uint32_t rounds = KEYED ? n : 1u;
    for (uint32_t i0 = 0; i0 < rounds; i0 += U * BT) {
        s.template load<BT, U>(i0 + tid, kk);
#pragma unroll
        for (uint32_t u = 0; u < U; u++) {
            if (i0 + u * BT >= n) break;
            const bool valid = i0 + u * BT + tid < n;
            below += valid && kk[u] < lo;
            kk[u] = valid ? kk[u] - lo : VTX_INVALID;
            if (kk[u] < C) atomicAdd(&L.cnt[kk[u]], 1u);
        }
    }
    below = scan64_add(below);
    if (lane == 63 && below) atomicAdd(&L.below, below);
    __syncthreads();
    // exclusive scan, consecutive cells per thread
    uint4 c4[Q];
    uint32_t sum = 0;
#pragma unroll
    for (uint32_t q = 0; q < Q; q++) {
        const uint4 c = c4[q] = reinterpret_cast<const uint4*>(L.cnt)[Q * tid + q];
        sum += c.x + c.y + c.z + c.w;
        if (max(max(c.x, c.y), max(c.z, c.w)) > VTX_HASH_HEAVY) {
            const uint32_t k = 4 * (Q * tid + q);
            if (c.x > VTX_HASH_HEAVY) L.heavy[atomicAdd(&L.nheavy, 1u)] = k;
            if (c.y > VTX_HASH_HEAVY) L.heavy[atomicAdd(&L.nheavy, 1u)] = k + 1;
            if (c.z > VTX_HASH_HEAVY) L.heavy[atomicAdd(&L.nheavy, 1u)] = k + 2;
            if (c.w > VTX_HASH_HEAVY) L.heavy[atomicAdd(&L.nheavy, 1u)] = k + 3;
        }
    }
    const uint32_t incl = scan64_add(sum);
    if (lane == 63) L.wsum[wave] = incl;
    __syncthreads();
    static_assert(NW <= 16, "the waves' sums are scanned in rows of 16 lanes");
    uint32_t ws = (lane & 15u) < NW ? L.wsum[lane & 15u] : 0u;
    ws += dpp0<0x111>(ws);
    ws += dpp0<0x112>(ws);
    ws += dpp0<0x114>(ws);
    ws += dpp0<0x118>(ws);
    const uint32_t own = (uint32_t)__builtin_amdgcn_readlane((int)ws, 15);
    uint32_t off = incl - sum + (wave ? (uint32_t)__builtin_amdgcn_readlane((int)ws, (int)wave - 1) : 0u);
#pragma unroll
    for (uint32_t q = 0; q < Q; q++) {
        const uint4 c = c4[q];
        reinterpret_cast<uint4*>(L.cnt)[Q * tid + q] = make_uint4(off, off + c.x, off + c.x + c.y, off + c.x + c.y + c.z);
        off += c.x + c.y + c.z + c.w;
    }
    const uint32_t base = L.below, nheavy = L.nheavy;
    const uint32_t padded = own <= 1u ? 1u : 1u << (32 - __builtin_clz(own - 1u));   // list entries to sort
    __syncthreads();
    // the range's particles into their cells, in any order; more than fit go through global scratch. Crowded
    // cells are sorted with the list, or stay out of it (their places marked empty) and are placed afterwards
    constexpr uint32_t FLAG = 1u << 31;                     // in cnt: a crowded cell that has its end already
    const bool fits = own <= VTX_HASH_PART_LIST, runs = nheavy && (!fits || n <= VTX_HASH_SORT_MIN);
    const auto keep_out = [&](uint32_t* __restrict__ list) {
        constexpr uint32_t NH = (VTX_HASH_PART_N / VTX_HASH_HEAVY + BT - 1) / BT;
        uint32_t end[NH];
#pragma unroll
        for (uint32_t r = 0; r < NH; r++) {
            const uint32_t h = r * BT + tid, k = h < nheavy ? L.heavy[h] : 0u;
            end[r] = k + 1u < C ? L.cnt[k + 1u] : own;
        }
        __syncthreads();
#pragma unroll
        for (uint32_t r = 0; r < NH; r++) {
            const uint32_t h = r * BT + tid;
            if (h < nheavy) {
                const uint32_t k = L.heavy[h];
                L.heavy[h] = L.cnt[k] << 12 | k;            // with the cell's first place (< 2^17)
                L.cnt[k] = end[r] | FLAG;
            }
        }
        __syncthreads();
        for (uint32_t h = 0; h < nheavy; h++) {
            const uint32_t b = L.heavy[h] >> 12, e = L.cnt[L.heavy[h] & 0xFFFu] & ~FLAG;
            for (uint32_t g = b + tid; g < e; g += BT) list[g] = VTX_INVALID;
        }
    };
    const auto fill = [&](uint32_t* __restrict__ list, auto crowded) {
        for (uint32_t i0 = 0; i0 < rounds; i0 += U * BT) {
            if (KEYED && n > U * BT) s.template load<BT, U>(i0 + tid, kk);
#pragma unroll
            for (uint32_t u = 0; u < U; u++) {
                if (i0 + u * BT >= n) break;
                const uint32_t i = i0 + u * BT + tid;
                const uint32_t k = KEYED && n > U * BT ? (i < n ? kk[u] - lo : VTX_INVALID) : kk[u];
                if (k < C && !(crowded.value && L.cnt[k] >> 31)) list[atomicAdd(&L.cnt[k], 1u)] = k << 20 | i;
            }
        }
        __syncthreads();
    };
    // every particle behind the smaller ones of its cell; V entries of the list in flight
    const auto place = [&](const uint32_t* __restrict__ list, auto crowded, auto v_, auto clamp) {
        constexpr uint32_t V = v_.value;
        for (uint32_t g0 = tid; g0 < own; g0 += V * BT) {
            uint32_t ev[V];
#pragma unroll
            for (uint32_t v = 0; v < V; v++) ev[v] = list[V > 1 ? min(g0 + v * BT, own - 1u) : g0];
#pragma unroll
            for (uint32_t v = 0; v < V; v++) {
                const uint32_t e = ev[v], k = e >> 20;
                if ((V > 1 && g0 + v * BT >= own) || (crowded.value && e == VTX_INVALID)) continue;
                const uint32_t begin = k ? L.cnt[k - 1] & (crowded.value ? ~FLAG : ~0u) : 0u, end = L.cnt[k];
                uint32_t at = begin;
                for (uint32_t j = begin; j < end; j += 4) {   // what follows the cell in the list is larger than e
                    uint32_t o[4];
#pragma unroll
                    for (uint32_t u = 0; u < 4; u++) o[u] = list[clamp.value ? min(j + u, own - 1u) : j + u];
#pragma unroll
                    for (uint32_t u = 0; u < 4; u++) at += (!(clamp.value || crowded.value) || j + u < end) && o[u] < e;
                }
                s.put(base + at, lo + k, e & 0xFFFFFu);
            }
        }
    };
    constexpr std::integral_constant<uint32_t, 1> one{};
    constexpr std::integral_constant<uint32_t, 4> four{};
    constexpr std::true_type yes{};
    constexpr std::false_type no{};
    if (fits && tid < 3) L.list[own + tid] = VTX_INVALID;
    if (!fits) {
        keep_out(spill + base);
        fill(spill + base, yes);
        place(spill + base, yes, four, yes);
    } else if (!nheavy) {
        fill(L.list, no);
        place(L.list, no, one, no);
    } else if (runs) {
        keep_out(L.list);
        fill(L.list, yes);
        place(L.list, yes, one, no);
    } else {
        for (uint32_t g = own + tid; g < padded; g += BT) L.list[g] = VTX_INVALID;
        fill(L.list, no);
        sort_list<BT>(L.list, padded);
        for (uint32_t g = tid; g < own; g += BT) {
            const uint32_t e = L.list[g];
            s.put(base + g, lo + (e >> 20), e & 0xFFFFFu);
        }
    }
    for (uint32_t k = tid; k < C; k += BT) {
        const uint32_t begin = k ? L.cnt[k - 1] & ~FLAG : 0u, end = L.cnt[k] & ~FLAG;
        s.cell(lo + k, end > begin ? base + begin : VTX_INVALID, end > begin ? base + end : VTX_INVALID);
    }
    if (runs) hash_part_runs<BT, KEYED ? 4 : 2>(s, n, lo, C, base, nheavy, L);
}

// A segment's particles: float4 positions, keys from k_hash_keys or worked out here.
template <bool KEYED>
struct SegmentHash {
    const float4 *P, *X0;
    const uint32_t* keys;
    uint2* cells;
    float4* rec;
    uint32_t *ko, *vo;
    uint32_t mod;
    float size;
    uint32_t n, M, shift;
    __device__ __forceinline__ uint32_t of(float4 p) const {
        return position_key(p, size, shift, M, mod);
    }
    __device__ __forceinline__ uint32_t key(uint32_t i) const { return KEYED ? keys[i] : of(P[i]); }
    template <uint32_t BT, uint32_t U>
    __device__ __forceinline__ void load(uint32_t i, uint32_t (&k)[U]) const {
        if (KEYED) {
#pragma unroll
            for (uint32_t u = 0; u < U; u++) k[u] = keys[min(i + u * BT, n - 1u)];
            return;
        }
        float4 p[U];
#pragma unroll
        for (uint32_t u = 0; u < U; u++) {
            p[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (i + u * BT < n) p[u] = P[i + u * BT];
        }
#pragma unroll
        for (uint32_t u = 0; u < U; u++) {
            k[u] = VTX_INVALID;
            if (u * BT < n) k[u] = of(p[u]);
        }
    }
    __device__ __forceinline__ void get(uint32_t i, float4& p, float4& x) const {
        p = P[i];
        x = X0[i];
    }
    __device__ __forceinline__ void put(uint32_t g, uint32_t k, uint32_t i, float4 p, float4 x) const {
        ko[g] = k;
        vo[g] = i;
        rec[2 * (size_t)g] = make_float4(p.x, p.y, p.z, __uint_as_float(i));
        rec[2 * (size_t)g + 1] = x;
    }
    __device__ __forceinline__ void put(uint32_t g, uint32_t k, uint32_t i) const {
        float4 p, x;
        get(i, p, x);
        put(g, k, i, p, x);
    }
    __device__ __forceinline__ void cell(uint32_t k, uint32_t begin, uint32_t end) const { cells[k] = make_uint2(begin, end); }
};

template <uint32_t BT, bool KEYED>
__device__ __forceinline__ void hash_part_segment(const DevState& d, const HashPartDev& t, int in, int dst, HashPartLds& L) {
    SegmentHash<KEYED> s;
    s.P = d.P[in] + t.pbase;
    s.X0 = d.X0 + t.pbase;
    s.keys = d.keys[dst ^ 1] + t.pbase;
    s.cells = d.cells + t.tbase;
    s.rec = d.sPX + 2 * (size_t)t.pbase;
    s.ko = d.keys[dst] + t.pbase;
    s.vo = d.vals[dst] + t.pbase;
    s.mod = t.mod;
    s.size = t.cell;
    s.n = t.n;
    s.M = t.M;
    s.shift = t.shift;
    hash_part<BT, KEYED>(s, t.n, t.lo, t.cells, d.vals[dst ^ 1] + t.pbase, L);
}

template <uint32_t BT>
__global__ __launch_bounds__(BT, 8) void k_hash_part(DevState d, int in, int dst) {
    __shared__ HashPartLds lds;
    const HashPartDev t = d.hparts[tile_of(d.remap)];   // the ranges of a segment on one XCD: they read the same particles
    if (t.keyed) hash_part_segment<BT, true>(d, t, in, dst, lds);
    else hash_part_segment<BT, false>(d, t, in, dst, lds);
}

// CacheNeighbors_Kernel (Velvet/SpatialHashGPU.cu:79-130). Cells are visited x-, y-, z-nested;
// inside a cell in sorted order, at most max_nbr entries per cell and in total; the list ends
// with ~0u unless full. Squared distances are fmaf(dz,dz,fmaf(dy,dy,dx*dx)).
//
// A wave takes PW consecutive particles of the sorted order. Consecutive particles of one grid cell
// (a run) have the same 27 candidate ranges, so the ranges are looked up once per run (the wave's
// lanes share out the runs' cells), and the run's candidates are loaded once, one per lane: lane l
// holds candidate l of the concatenated ranges, and the wave tests a particle against 64 candidates at
// a time. The particle is wave-uniform (scalar loads); the accepted lanes take their places in the
// list from the test's ballot, which keeps the walk's order. One particle per lane instead, each
// lane walking its own 60 to 300 candidates one after the other, was bound by that chain at small
// sizes and by the vector cache at large ones (0.9 accesses a clock on every CU): 16,384 particles
// 88 -> 11.8 us, 65,536 particles 54.6 -> 16.9 us, 963,130 in 256 draped cloths 204.8 -> 106.7 us (a
// particle tests some 150 candidates at 15 VALU instructions per 64, and 6 more where one is accepted:
// 85% of its VALU issue time). A segment whose records outgrow the L2 is bound by fetching each cell's
// records again and again, as neighbours in the sorted order are no neighbours in space: 1,048,576 particles,
// 33.5 MB of records, fetch 1,605 MB a search at rest (242 us) and 1,083 MB in a pile (286 us; one particle
// per lane 759) (by particle index instead: neighbor_blocks).
struct NbSet {
    const float4* rec;    // sorted records: position with w = index at 2i, initial position at 2i + 1
    const uint2* cells;   // (start, end) per hash cell
    char* table;          // neighbour lists
    uint32_t mod;         // mod_constant(M)
    uint32_t n, M, K, shift;
    float cell, cell2, diam2;
    bool n16;             // 16-bit entries
};

// The lists' layout: entry k of particle i, CHUNK: chunks of four entries, chunk c at entry
// 4 (c n + i); else column-major at entry k n + i (the kernel-launch tier's layout). Entries are
// 32-bit or, for a segment with VTX_SEG_NBR16, 16-bit (the sentinel truncated to 0xffff).
template <bool CHUNK>
__device__ __forceinline__ void nb_put(const NbSet& a, uint32_t id, uint32_t k, uint32_t v) {
    const uint32_t esh = CHUNK && a.n16 ? 1u : 2u;
    const uint32_t row = CHUNK ? k >> 2 : k, stride = (CHUNK ? 4 * a.n : a.n);
    char* at = a.table + (((uint64_t)row * stride + (CHUNK ? 4 * id + (k & 3u) : id)) << esh);
    if (CHUNK && a.n16) *reinterpret_cast<uint16_t*>(at) = (uint16_t)v;
    else *reinterpret_cast<uint32_t*>(at) = v;
}

// How the search stores entries: chunks of 16-bit or 32-bit entries or the column-major layout, and whether
// a table's byte offsets fit 32 bits with 24-bit factors (n < 2^22).
enum NbStore { NB_CHUNK16, NB_CHUNK32, NB_COLUMN };

// nb_put with `row` = entries of a row (4 n or n) and at0 = the particle's first entry, both wave-uniform.
template <NbStore ST, bool SMALL>
__device__ __forceinline__ void nb_put_uniform(const NbSet& a, uint32_t id, uint32_t row, uint32_t at0, uint32_t k, uint32_t v) {
    if (!SMALL) {
        nb_put<ST != NB_COLUMN>(a, id, k, v);
        return;
    }
    uint32_t off;   // the compiler takes the 32-bit product otherwise, a quarter of the rate
    if (ST == NB_COLUMN) {
        asm("v_mul_u32_u24 %0, %2, %1" : "=v"(off) : "v"(k), "s"(row));
        off += at0;
    } else {
        asm("v_mul_u32_u24 %0, %2, %1" : "=v"(off) : "v"(k >> 2), "s"(row));
        off += at0 | (k & 3u);
    }
    if (ST == NB_CHUNK16) *reinterpret_cast<uint16_t*>(a.table + (off << 1)) = (uint16_t)v;
    else *reinterpret_cast<uint32_t*>(a.table + (off << 2)) = v;
}

// v with lane l's value replaced (x and l wave-uniform).
__device__ __forceinline__ uint32_t write_lane(uint32_t v, uint32_t x, uint32_t l) {
    asm("s_mov_b32 m0, %2\n\tv_writelane_b32 %0, %1, m0" : "+v"(v) : "s"(x), "s"(l) : "m0");
    return v;
}

// LDS of one wave of the search.
template <int PW>
struct NbLds {
    uint32_t range[PW * 27];   // per (run, cell): start | length << 25
    uint32_t cx[PW], cy[PW], cz[PW];   // per run: its cell's coordinates times the hash's factors
    uint32_t mark[64];
};

// A sorted record through the scalar cache (i wave-uniform).
__device__ __forceinline__ void ld_record_uniform(const float4* rec, uint32_t i, float4& p, float4& o) {
    typedef const float __attribute__((address_space(4))) cfloat;
    cfloat* q = (cfloat*)(uintptr_t)(rec + 2 * (size_t)i);
    p = make_float4(q[0], q[1], q[2], q[3]);
    o = make_float4(q[4], q[5], q[6], 0.f);
}

// The lists of cnt <= PW particles by the calling wave: the sorted positions from i0 on, or with LISTED
// lane m's i0.
template <int PW, NbStore ST, bool SMALL, bool LISTED>
__device__ __forceinline__ void neighbor_wave_as(const NbSet& a, uint32_t i0, uint32_t cnt, NbLds<PW>& L) {
#pragma clang fp contract(off)
    constexpr int NC = 2;                                   // candidate chunks held at a time
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t lt = (1ull << lane) - 1ull;
    // the wave's particles: cells, runs
    float4 me = make_float4(0.f, 0.f, 0.f, 0.f);
    if (lane < cnt) me = a.rec[2 * (size_t)(LISTED ? i0 : i0 + lane)];
    int32_t ix, iy, iz;
    cell_coords(me, a.cell, a.shift, ix, iy, iz);
    // every lane active in the exchange: one that sits out would hand its neighbour nothing
    const int32_t px = __shfl_up(ix, 1, 64), py = __shfl_up(iy, 1, 64), pz = __shfl_up(iz, 1, 64);
    const bool head = lane < cnt && ((lane == 0) | (px != ix) | (py != iy) | (pz != iz));
    const uint64_t heads = __builtin_amdgcn_ballot_w64(head);
    const uint32_t nruns = (uint32_t)__popcll(heads);
    if (head) {                                             // the cell as hashed, factor by factor
        const uint32_t r = (uint32_t)__popcll(heads & lt);
        L.cx[r] = (uint32_t)ix * HX;
        L.cy[r] = (uint32_t)iy * HY;
        L.cz[r] = (uint32_t)iz * HZ;
    }
    wave_lds_sync();
    // the runs' cell ranges: a half of the wave takes one run, a lane (of 27) always the same of its cells,
    // so that the lane's share of the hash's products is worked out once; four rounds' loads in flight
    const uint32_t q = lane & 31u, dx = (q * 57u) >> 9, yz = q - 9u * dx, dy = (yz * 11u) >> 5, dz = yz - 3u * dy;
    const uint32_t ox = (dx - 1u) * HX, oy = (dy - 1u) * HY, oz = (dz - 1u) * HZ;
    for (uint32_t r0 = 0; r0 < nruns; r0 += 8u) {
        uint64_t c[4];
#pragma unroll
        for (uint32_t u = 0; u < 4u; u++) {
            if (r0 + 2u * u >= nruns) break;
            const uint32_t r = min(r0 + 2u * u + (lane >> 5), nruns - 1u);
            const uint32_t hq = hash_reduce((L.cx[r] + ox) ^ (L.cy[r] + oy) ^ (L.cz[r] + oz), a.M, a.mod);
            c[u] = q < 27u ? *reinterpret_cast<const uint64_t*>(a.cells + hq) : 0ull;   // one 8-byte load
        }
#pragma unroll
        for (uint32_t u = 0; u < 4u; u++) {
            if (r0 + 2u * u >= nruns) break;
            const uint32_t r = r0 + 2u * u + (lane >> 5);
            const uint32_t st = (uint32_t)c[u], len = min((uint32_t)(c[u] >> 32) - st, a.K);
            if (q < 27u && r < nruns) L.range[r * 27u + q] = st == VTX_INVALID ? 0u : st | len << 25;
        }
    }
    wave_lds_sync();
    uint32_t kv = 0;                                        // lane m: entries of particle m
    const uint32_t row = ST == NB_COLUMN ? a.n : 4 * a.n;
    uint64_t rest = heads;
    for (uint32_t r = 0; r < nruns; r++) {
        const uint32_t m0 = (uint32_t)__builtin_ctzll(rest);
        rest &= rest - 1ull;
        const uint32_t m1 = rest ? (uint32_t)__builtin_ctzll(rest) : cnt;
        const uint32_t v = lane < 27u ? L.range[r * 27u + lane] : 0u;
        const uint32_t len = v >> 25, incl = scan32_add(len), excl = incl - len;
        const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 31);
        const uint32_t base = (v & 0x1FFFFFFu) - excl;      // candidate c of the cell: sorted position base + c
        for (uint32_t g0 = 0; g0 < total; g0 += 64u * NC) {
            float4 q[NC], x[NC];
#pragma unroll
            for (int h = 0; h < NC; h++) {
                const uint32_t c0 = g0 + 64u * h;
                q[h] = x[h] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (h && c0 >= total) continue;
                // the cell of each lane's candidate: every cell marks the lane of its first one
                L.mark[lane] = 0;
                wave_lds_sync();
                if (lane < 27u && len && incl > c0 && excl < c0 + 64u) L.mark[max(excl, c0) - c0] = lane + 1u;
                wave_lds_sync();
                const uint32_t own = scan64_max(L.mark[lane]);
                const uint32_t b = (uint32_t)__builtin_amdgcn_ds_bpermute((int)((own - 1u) << 2), (int)base);
                const uint32_t at = c0 + lane < total ? b + c0 + lane : 0u;
                q[h] = a.rec[2 * (size_t)at];
                x[h] = a.rec[2 * (size_t)at + 1];
                if (c0 + lane >= total) q[h].x = __builtin_nanf("");
                wave_lds_sync();
            }
            // lanes without a candidate are farther than any distance; the particle itself is told by its index
            for (uint32_t m = m0; m < m1; m++) {
                float4 p, o;
                ld_record_uniform(a.rec, LISTED ? (uint32_t)__builtin_amdgcn_readlane((int)i0, (int)m) : i0 + m, p, o);
                const uint32_t id = __float_as_uint(p.w);
                uint32_t k = (uint32_t)__builtin_amdgcn_readlane((int)kv, (int)m);
#pragma unroll
                for (int h = 0; h < NC; h++) {
                    if (h && g0 + 64u * h >= total) continue;
                    const float dx = p.x - q[h].x, dy = p.y - q[h].y, dz = p.z - q[h].z;
                    const float d2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
                    const float ex = o.x - x[h].x, ey = o.y - x[h].y, ez = o.z - x[h].z;
                    const float e2 = __builtin_fmaf(ez, ez, __builtin_fmaf(ey, ey, ex * ex));
                    const uint64_t mask = __builtin_amdgcn_ballot_w64(d2 < a.cell2) &
                                          __builtin_amdgcn_ballot_w64(e2 > a.diam2) &
                                          __builtin_amdgcn_ballot_w64(__float_as_uint(q[h].w) != id);
                    if (!mask) continue;
                    const uint32_t e = __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                                                 __builtin_amdgcn_mbcnt_lo((uint32_t)mask, k));
                    if (__builtin_amdgcn_inverse_ballot_w64(mask) && e < a.K)
                        nb_put_uniform<ST, SMALL>(a, id, row, ST == NB_COLUMN ? id : 4 * id, e, __float_as_uint(q[h].w));
                    k = min(k + (uint32_t)__popcll(mask), a.K);
                }
                kv = write_lane(kv, k, m);
            }
        }
    }
    // a full list has no sentinel
    if (lane < cnt && kv < a.K) nb_put<ST != NB_COLUMN>(a, __float_as_uint(me.w), kv, VTX_INVALID);
}

template <int PW, bool CHUNK, bool LISTED = false>
__device__ __forceinline__ void neighbor_wave(const NbSet& a, uint32_t i0, uint32_t cnt, NbLds<PW>& L) {
    if (CHUNK && a.n16) neighbor_wave_as<PW, NB_CHUNK16, true, LISTED>(a, i0, cnt, L);   // n < 2^16
    else if (a.n < (1u << 22)) neighbor_wave_as<PW, CHUNK ? NB_CHUNK32 : NB_COLUMN, true, LISTED>(a, i0, cnt, L);
    else neighbor_wave_as<PW, CHUNK ? NB_CHUNK32 : NB_COLUMN, false, LISTED>(a, i0, cnt, L);
}

// The search by particle index (search_rule), for segments whose records outgrow the L2. In sorted order
// the waves that run at one time have no cells in common, as neighbouring hashes are no neighbours in space.
// Here a wave takes whole blocks of cells by index: neighbours in a cloth's index order are neighbours in
// space, and a tile's wave and those beside it (on one XCD) share cells. A block is what a bucket holds of an
// aligned run of PW sorted positions; the one of its particles that leads it is drawn by a hash of its first
// position, so that of several layers not the lowest does all the work. inv: particle -> sorted position.
// A draped 1,048,576-particle cloth on grid 1 fetches 440 MB instead of 1,605: 243 -> 154 us a search, 1.78 ->
// 1.61 ms a frame; on the reference grid, whose mirrored cells share buckets, 245 -> 198 us. A pile loses,
// 319 -> 497 us, as the waves are uneven and fetches are not what bounds it.
template <int PW>
__device__ __forceinline__ void neighbor_blocks(const NbSet& a, const uint32_t* __restrict__ inv,
                                                const float4* __restrict__ P, uint32_t first, uint32_t cnt, NbLds<PW>& L) {
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t begin = 0, len = 0;
    if (lane < cnt) {
        const uint32_t pos = inv[first + lane];
        const uint2 c = a.cells[position_key(P[first + lane], a.cell, a.shift, a.M, a.mod)];
        begin = max(c.x, pos & ~(PW - 1u));
        const uint32_t n = min(c.y, (pos & ~(PW - 1u)) + PW) - begin;
        if (c.x <= pos && pos < c.y && pos == begin + (((begin * 2654435761u) >> 16) * n >> 16)) len = n;   // len <= PW
    }
    const uint32_t incl = scan32_add(len), excl = incl - len;
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 31);
    for (uint32_t b = 0; b < total; b += PW) {
        L.mark[lane] = 0;
        wave_lds_sync();
        if (len && incl > b && excl < b + PW) L.mark[max(excl, b) - b] = lane + 1u;
        wave_lds_sync();
        const uint32_t own = scan64_max(L.mark[lane]);
        const uint32_t at = (uint32_t)__builtin_amdgcn_ds_bpermute((int)((own - 1u) << 2), (int)(begin - excl));
        wave_lds_sync();
        neighbor_wave<PW, true, true>(a, at + b + lane, min((uint32_t)PW, total - b), L);
        wave_lds_sync();
    }
}

// The search over the segments' particle tiles (a tile's sorted positions): 4 PW particles per
// workgroup of four waves.
template <int PW, bool BY_INDEX>
__global__ __launch_bounds__(256) void k_neighbors(DevState d, int in, const uint32_t* __restrict__ inv,
                                                   const uint32_t* __restrict__ sample, SearchRule rule) {
    __shared__ NbLds<PW> lds[4];
    const uint32_t b = tile_of(d.remap), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr uint32_t S = VTX_TILE / (4 * PW);                 // workgroups per tile
    const TileDev t = d.tiles[b / S];
    const uint32_t first = ((b % S) * 4 + wave) * PW;
    const SegDev& sg = d.segs[t.seg];
    if (first >= t.count || !(sg.flags & VTX_SEG_SELFCOL)) return;
    NbSet a;
    a.rec = d.sPX + 2 * (size_t)sg.pbase;
    a.cells = d.cells + sg.tbase;
    a.table = reinterpret_cast<char*>(d.nbr + ((uint64_t)sg.nbase_hi << 32 | sg.nbase_lo));
    a.mod = sg.mod;
    a.n = sg.n;
    a.M = sg.M;
    a.K = sg.max_nbr;
    a.shift = seg_shift(sg);
    a.cell = sg.cell;
    a.cell2 = sg.cell2;
    a.diam2 = sg.diam2;
    a.n16 = sg.flags & VTX_SEG_NBR16;
    const uint32_t i = t.begin - sg.pbase + first, cnt = min((uint32_t)PW, t.count - first);
    if (BY_INDEX && search_by_index(rule, sg.n, sg.flags) && (!rule.cells || sample[sg.pbase] >= rule.cells))
        neighbor_blocks<PW>(a, inv + sg.pbase, d.P[in] + sg.pbase, i, cnt, lds[wave]);
    else
        neighbor_wave<PW, true>(a, i, cnt, lds[wave]);
}

// ---------------------------------------------------------------- kernel-launch tier
// HashObjects on raw device arrays (Velvet/SpatialHashGPU.cu:159-196, SpatialHashGPU.cuh:17-25):
// one object set, positions and initial positions as packed xyz triples (glm::vec3), the
// sort's key/value ping-pong partly in the caller's particle_hash / particle_index and partly in
// a workspace, which also holds the interleaved cell table and the 32-B sorted records that
// the walk reads (one cache line per candidate).

__device__ __forceinline__ float4 ld_xyz(const float* __restrict__ a, uint32_t i, float w) {
    return make_float4(a[3 * (size_t)i], a[3 * (size_t)i + 1], a[3 * (size_t)i + 2], w);
}

// ComputeParticleHash_Kernel (Velvet/SpatialHashGPU.cu:34-42).
__global__ __launch_bounds__(VTX_TILE) void k_raw_keys(const float* __restrict__ pos, uint32_t n, float cell,
                                                       uint32_t M, uint32_t mod, uint32_t* __restrict__ keys,
                                                       uint32_t* __restrict__ vals) {
    const uint32_t i = blockIdx.x * VTX_TILE + threadIdx.x;
    if (i >= n) return;
    const float4 p = ld_xyz(pos, i, 0.f);
    keys[i] = position_key(p, cell, 0u, M, mod);
    vals[i] = i;
}

// Sort tile b covers keys [b * VTX_SORT_TILE, ...); its digit g count sits at hist[g * ntiles + b].
__global__ __launch_bounds__(VTX_TILE) void k_raw_sort_hist(const uint32_t* __restrict__ keys, uint32_t n, int shift,
                                                            uint32_t* __restrict__ hist) {
    const uint32_t b = blockIdx.x, begin = b * VTX_SORT_TILE;
    tile_hist(keys + begin, min(n - begin, (uint32_t)VTX_SORT_TILE), shift, hist + b, gridDim.x);
}

__global__ __launch_bounds__(VTX_TILE) void k_raw_sort_scatter(const uint32_t* __restrict__ kin,
                                                               const uint32_t* __restrict__ vin, uint32_t n,
                                                               int shift, const uint32_t* __restrict__ hist,
                                                               uint32_t* __restrict__ kout, uint32_t* __restrict__ vout) {
    const uint32_t b = blockIdx.x, begin = b * VTX_SORT_TILE;
    tile_scatter(kin + begin, vin + begin, min(n - begin, (uint32_t)VTX_SORT_TILE), shift, hist + b, gridDim.x, 0u,
                 kout, vout);
}

// FindCellStart_Kernel (Velvet/SpatialHashGPU.cu:44-77) into the interleaved table (cells were
// filled with ~0u), plus the sorted records.
__global__ __launch_bounds__(VTX_TILE) void k_raw_cell_bounds(const uint32_t* __restrict__ skeys,
                                                              const uint32_t* __restrict__ svals, uint32_t n,
                                                              const float* __restrict__ pos,
                                                              const float* __restrict__ pos0,
                                                              uint2* __restrict__ cells, float4* __restrict__ rec) {
    const uint32_t g = blockIdx.x * VTX_TILE + threadIdx.x;
    if (g >= n) return;
    const uint32_t key = skeys[g];
    if (g == 0) {
        cells[key].x = 0;
    } else {
        const uint32_t prev = skeys[g - 1];
        if (key != prev) {
            cells[key].x = g;
            cells[prev].y = g;
        }
    }
    if (g == n - 1) cells[key].y = n;
    const uint32_t id = svals[g];
    rec[2 * (size_t)g] = ld_xyz(pos, id, __uint_as_float(id));
    rec[2 * (size_t)g + 1] = ld_xyz(pos0, id, 0.f);
}

// The same table, arrays and records by cell ranges (hash_part), straight from the positions or from the
// keys of k_raw_keys; the caller's cell arrays are written here too.
template <bool KEYED>
struct RawHash {
    const float *pos, *pos0;
    const uint32_t* keys;
    uint2* cells;
    float4* rec;
    uint32_t *ko, *vo, *start, *end;
    uint32_t mod;
    float size;
    uint32_t n, M;
    __device__ __forceinline__ uint32_t of(float4 p) const {
        return position_key(p, size, 0u, M, mod);
    }
    __device__ __forceinline__ uint32_t key(uint32_t i) const { return KEYED ? keys[i] : of(ld_xyz(pos, i, 0.f)); }
    template <uint32_t BT, uint32_t U>
    __device__ __forceinline__ void load(uint32_t i, uint32_t (&k)[U]) const {
        if (KEYED) {
#pragma unroll
            for (uint32_t u = 0; u < U; u++) k[u] = keys[min(i + u * BT, n - 1u)];
            return;
        }
        float4 p[U];
#pragma unroll
        for (uint32_t u = 0; u < U; u++) {
            p[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (i + u * BT < n) p[u] = ld_xyz(pos, i + u * BT, 0.f);
        }
#pragma unroll
        for (uint32_t u = 0; u < U; u++) {
            k[u] = VTX_INVALID;
            if (u * BT < n) k[u] = of(p[u]);
        }
    }
    __device__ __forceinline__ void get(uint32_t i, float4& p, float4& x) const {
        p = ld_xyz(pos, i, __uint_as_float(i));
        x = ld_xyz(pos0, i, 0.f);
    }
    __device__ __forceinline__ void put(uint32_t g, uint32_t k, uint32_t i, float4 p, float4 x) const {
        ko[g] = k;
        vo[g] = i;
        rec[2 * (size_t)g] = p;
        rec[2 * (size_t)g + 1] = x;
    }
    __device__ __forceinline__ void put(uint32_t g, uint32_t k, uint32_t i) const {
        float4 p, x;
        get(i, p, x);
        put(g, k, i, p, x);
    }
    __device__ __forceinline__ void cell(uint32_t k, uint32_t b, uint32_t e) const {
        cells[k] = make_uint2(b, e);
        start[k] = b;
        end[k] = e;
    }
};

template <bool KEYED>
__global__ __launch_bounds__(VTX_HASH_PART_BT, 8) void k_raw_hash_part(RawHash<KEYED> s, uint32_t width, uint32_t* spill) {
    __shared__ HashPartLds lds;
    const uint32_t lo = blockIdx.x * width;
    hash_part<VTX_HASH_PART_BT, KEYED>(s, s.n, lo, min(width, s.M - lo), spill, lds);
}

// CacheNeighbors_Kernel (Velvet/SpatialHashGPU.cu:79-130).
template <int PW>
__global__ __launch_bounds__(256) void k_raw_neighbors(const float4* __restrict__ rec, const uint2* __restrict__ cells,
                                                       uint32_t* __restrict__ nbr, uint32_t n, float cell, float cell2,
                                                       float diam2, uint32_t M, uint32_t mod, uint32_t K) {
    __shared__ NbLds<PW> lds[4];
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t first = (blockIdx.x * 4 + wave) * PW;
    if (first >= n) return;
    const NbSet a{rec, cells, reinterpret_cast<char*>(nbr), mod, n, M, K, 0u, cell, cell2, diam2, false};
    neighbor_wave<PW, false>(a, first, min((uint32_t)PW, n - first), lds[wave]);
}

// The interleaved table to the caller's cell_start / cell_end (empty cells: ~0u in both).
__global__ __launch_bounds__(VTX_TILE) void k_raw_split_cells(const uint2* __restrict__ cells, uint32_t M,
                                                              uint32_t* __restrict__ start, uint32_t* __restrict__ end) {
    for (uint32_t i = blockIdx.x * VTX_TILE + threadIdx.x; i < M; i += gridDim.x * VTX_TILE) {
        const uint2 c = cells[i];
        start[i] = c.x;
        end[i] = c.y;
    }
}

// Particles per wave of the neighbour search. Up to 2^17 particles in a launch a wave takes 8: the chip's 8,192
// waves are not all busy, and a wave's particles go one after the other (measured, us per search, 8 /
// 32 particles a wave: 16,384 particles 11.8 / 27.9, 65,536 17.1 / 29.7). Above, 32: the lookups of a
// run and its candidates' loads serve more particles (963,130 particles in 256 cloths 164.9 / 129.9;
// a pile of 1,048,576 runs long lists either way, 268 / 293).
static bool search_small(uint32_t particles) { return particles <= (1u << 17); }

size_t hash_workspace_bytes(uint32_t n, uint32_t M) {
    const size_t tiles = (n + VTX_SORT_TILE - 1) / VTX_SORT_TILE;
    const size_t nhist = 256 * tiles, nparts = (nhist + VTX_SCAN_BLOCK - 1) / VTX_SCAN_BLOCK;
    auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
    return up(32 * (size_t)n) + up(8 * (size_t)M) + up(8 * (size_t)n) + up(4 * nhist) + up(4 * nparts);
}

hipError_t hash_objects(const HashObjectsArgs& a, void* workspace, hipStream_t s) {
    const uint32_t n = a.num_objects, M = a.table_size;
    auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
    char* w = static_cast<char*>(workspace);
    float4* rec = reinterpret_cast<float4*>(w);
    w += up(32 * (size_t)n);
    uint2* cells = reinterpret_cast<uint2*>(w);
    w += up(8 * (size_t)M);
    uint32_t* kalt = reinterpret_cast<uint32_t*>(w);
    uint32_t* valt = kalt + n;
    w += up(8 * (size_t)n);
    const uint32_t tiles = (n + VTX_SORT_TILE - 1) / VTX_SORT_TILE;
    uint32_t* hist = reinterpret_cast<uint32_t*>(w);
    w += up(4 * (size_t)256 * tiles);
    uint32_t* part = reinterpret_cast<uint32_t*>(w);

    const uint32_t blocks = (n + VTX_TILE - 1) / VTX_TILE;
    const uint32_t mod = mod_constant(M);
    const auto search = [&] {
        const auto nb = [&](auto kernel, uint32_t pw) {
            hipLaunchKernelGGL(kernel, dim3((n + 4 * pw - 1) / (4 * pw)), dim3(256), 0, s, (const float4*)rec,
                               (const uint2*)cells, a.neighbors, n, a.cell_spacing, a.cell_spacing2,
                               a.particle_diameter2, M, mod, a.max_num_neighbors);
        };
        if (search_small(n)) nb(k_raw_neighbors<8>, 8);
        else nb(k_raw_neighbors<32>, 32);
    };
    if (n && hash_by_ranges(n, M)) {   // one or two launches instead of up to sixteen
        const uint32_t width = hash_part_width(n, M, VTX_HASH_PART_SHARE), parts = (M + width - 1) / width;
        const auto build = [&](auto keyed) {
            constexpr bool K = decltype(keyed)::value;
            const RawHash<K> h{a.positions, a.original_positions, kalt, cells, rec, a.particle_hash, a.particle_index,
                               a.cell_start, a.cell_end, mod, a.cell_spacing, n, M};
            hipLaunchKernelGGL((k_raw_hash_part<K>), dim3(parts), dim3(VTX_HASH_PART_BT), 0, s, h, width, valt);
        };
        if (n > VTX_HASH_PART_KEYS) {
            hipLaunchKernelGGL(k_raw_keys, dim3(blocks), dim3(VTX_TILE), 0, s, a.positions, n, a.cell_spacing, M, mod,
                               kalt, valt);
            build(std::true_type{});
        } else {
            build(std::false_type{});
        }
        search();
        return hipGetLastError();
    }

    // stable LSD radix sort on ceil(log2 M) bits (Velvet/SpatialHashGPU.cu:179), 8 per pass;
    // the keys start on the side that makes the last pass end in the caller's arrays
    const uint32_t bits = M > 1 ? 32u - (uint32_t)__builtin_clz(M - 1u) : 0u;
    const int passes = (int)((bits + 7) / 8);
    uint32_t* k[2] = {a.particle_hash, kalt};
    uint32_t* v[2] = {a.particle_index, valt};
    int src = passes & 1;
    if (n) hipLaunchKernelGGL(k_raw_keys, dim3(blocks), dim3(VTX_TILE), 0, s, a.positions, n, a.cell_spacing, M, mod,
                              k[src], v[src]);
    for (int pass = 0; pass < passes && n; pass++) {
        hipLaunchKernelGGL(k_raw_sort_hist, dim3(tiles), dim3(VTX_TILE), 0, s, (const uint32_t*)k[src], n, 8 * pass,
                           hist);
        hipError_t e = launch_scan(hist, 256 * tiles, part, s);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_raw_sort_scatter, dim3(tiles), dim3(VTX_TILE), 0, s, (const uint32_t*)k[src],
                           (const uint32_t*)v[src], n, 8 * pass, (const uint32_t*)hist, k[src ^ 1], v[src ^ 1]);
        src ^= 1;
    }
    hipError_t e = launch_fill_u32(reinterpret_cast<uint32_t*>(cells), 2 * M, VTX_INVALID, s);
    if (e != hipSuccess) return e;
    if (n) {
        hipLaunchKernelGGL(k_raw_cell_bounds, dim3(blocks), dim3(VTX_TILE), 0, s, (const uint32_t*)a.particle_hash,
                           (const uint32_t*)a.particle_index, n, a.positions, a.original_positions, cells, rec);
        search();
    }
    uint32_t sb = (M + VTX_TILE - 1) / VTX_TILE;
    if (sb > 4096) sb = 4096;
    if (sb) hipLaunchKernelGGL(k_raw_split_cells, dim3(sb), dim3(VTX_TILE), 0, s, (const uint2*)cells, M, a.cell_start,
                               a.cell_end);
    return hipGetLastError();
}

// Workspace of hash_objects_noalloc: a fixed device array, one copy per GPU, alive until the
// process ends. Host code never passes `scratch` itself to a kernel (on the host the name is a
// shadow, not a device address): each device's address comes from hipGetSymbolAddress, taken once
// per device with that device current, and only that address is used.
static __device__ __align__(256) unsigned char scratch[VTX_HASH_SCRATCH_BYTES];

#define VTX_SCRATCH_MAX_DEVICES 64
static std::mutex scratch_mu;
static void* scratch_ptr[VTX_SCRATCH_MAX_DEVICES];

static hipError_t scratch_address(void** out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= VTX_SCRATCH_MAX_DEVICES) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(scratch_mu);
    if (!scratch_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        if (!p) return hipErrorInvalidSymbol;
        scratch_ptr[dev] = p;
    }
    *out = scratch_ptr[dev];
    return hipSuccess;
}

hipError_t hash_objects_noalloc(const HashObjectsArgs& a, hipStream_t s) {
    if (hash_workspace_bytes(a.num_objects, a.table_size) > (size_t)VTX_HASH_SCRATCH_BYTES) return hipErrorInvalidValue;
    void* ws = nullptr;
    const hipError_t e = scratch_address(&ws);
    if (e != hipSuccess) return e;
    // every workspace part is written before it is read (records, cell table fill, sort
    // keys, histograms, scan partials), so nothing is cleared between calls
    return hash_objects(a, ws, s);
}

// ---------------------------------------------------------------- host launchers
hipError_t launch_hash_keys(const DevState& d, int in, int dst, hipStream_t s) {
    hipLaunchKernelGGL(k_hash_keys, dim3(d.ntiles), dim3(VTX_TILE), 0, s, d, in, dst);
    return hipGetLastError();
}

hipError_t launch_scan(uint32_t* a, uint32_t n, uint32_t* part, hipStream_t s) {
    const uint32_t nb = (n + VTX_SCAN_BLOCK - 1) / VTX_SCAN_BLOCK;
    if (!nb) return hipSuccess;
    hipLaunchKernelGGL(k_scan_reduce, dim3(nb), dim3(VTX_TILE), 0, s, a, n, part);
    hipLaunchKernelGGL(k_scan_apply, dim3(nb), dim3(VTX_TILE), 0, s, a, n, (const uint32_t*)part);
    return hipGetLastError();
}

hipError_t launch_sort_pass(const DevState& d, int src, int shift, hipStream_t s) {
    hipLaunchKernelGGL(k_sort_hist, dim3(d.nstiles), dim3(VTX_TILE), 0, s, d, src, shift);
    hipError_t e = launch_scan(d.hist + d.hbase0, d.nhist, d.part, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_sort_scatter, dim3(d.nstiles), dim3(VTX_TILE), 0, s, d, src, shift);
    return hipGetLastError();
}

hipError_t launch_fill_u32(uint32_t* a, uint32_t n, uint32_t v, hipStream_t s) {
    if (!n) return hipSuccess;
    uint32_t blocks = (n + 1023) / 1024;
    if (blocks > 2048) blocks = 2048;
    hipLaunchKernelGGL(k_fill_u32, dim3(blocks), dim3(1024), 0, s, a, n, v);
    return hipGetLastError();
}

hipError_t launch_hash_parts(const DevState& d, int in, int dst, hipStream_t s) {
    // a full chip: 512 threads a range hold half of the wave slots while they wait (512 cloths of 963,130
    // particles with three solvers overlapping, us a frame pair, 1024 / 512 threads: 3205 / 3175); a lone
    // cloth's ranges take 1024 (the chip is empty, more loads in flight)
    if (d.nhparts && (d.live & VTX_LIVE_FULL))
        hipLaunchKernelGGL(k_hash_part<VTX_HASH_PART_BT / 2>, dim3(d.nhparts), dim3(VTX_HASH_PART_BT / 2), 0, s, d, in, dst);
    else if (d.nhparts)
        hipLaunchKernelGGL(k_hash_part<VTX_HASH_PART_BT>, dim3(d.nhparts), dim3(VTX_HASH_PART_BT), 0, s, d, in, dst);
    return hipGetLastError();
}

hipError_t launch_clear_cells(const DevState& d, hipStream_t s) {
    hipLaunchKernelGGL(k_clear_cells, dim3(d.ntiles), dim3(VTX_TILE), 0, s, d);
    return hipGetLastError();
}

hipError_t launch_cell_bounds(const DevState& d, int in, int src, hipStream_t s) {
    hipLaunchKernelGGL(k_cell_bounds, dim3(d.ntiles), dim3(VTX_TILE), 0, s, d, in, src);
    hipLaunchKernelGGL(k_sorted_records, dim3(d.ntiles), dim3(VTX_TILE), 0, s, d, in, src);
    return hipGetLastError();
}

hipError_t launch_neighbors(const DevState& d, int in, int src, bool by_index, SearchRule rule, hipStream_t s) {
    const auto nb = [&](auto kernel, uint32_t pw) {
        hipLaunchKernelGGL(kernel, dim3(d.ntiles * (VTX_TILE / (4 * pw))), dim3(256), 0, s, d, in,
                           (const uint32_t*)d.keys[src ^ 1], (const uint32_t*)d.vals[src ^ 1], rule);   // k_cell_bounds' output
    };
    if (search_small(d.nparticles)) nb(k_neighbors<8, false>, 8);
    else if (by_index) nb(k_neighbors<32, true>, 32);
    else nb(k_neighbors<32, false>, 32);
    return hipGetLastError();
}

}  // namespace vtx
