// lf_kernels.hip -- CDNA4 (gfx950) kernels of one WCSPH substep over a pool
// of independent scenes.
//
// Pool: every per-particle array spans all particle slots of the pool.  A
// scene owns whole 512-slot chunks starting at slot `first` (its particles
// fill [first, first + count)) and a bucket range [cell_base, cell_base +
// ncells + 1): its grid cells and its out-of-grid bucket.  One exclusive scan
// runs over all buckets of the pool; a scene places its particles at
// first + (start[b] - start[cell_base]) + rank, so free slots and buckets
// between scenes, or scenes left out of a step, need no bookkeeping.  Every
// pass is one launch over all slots of the pool; a workgroup serves one scene
// and reads that scene's constants (Consts table) with scalar loads.  A
// single scene is a pool of one.
//
// Layout: every per-particle array is SoA float4 (16 B, one dwordx4 load):
//   P = (x, y, z, id bits)   V = (vx, vy, vz, 0)   A = (ax, ay, az, 0)
//   L = low-order position words: the position is the double-float P.xyz + L.xyz
//   D = (density, pressure, sound speed, 1/density)   N = (normal, 0)
// Ids are scene-local.  The sorted arrays are in (cell key, particle id)
// order; `start` holds the first slot of every bucket up to the pool's
// active span plus an end sentinel.
//
// The density pass tests every candidate of the clipped 27-cell stencil (nine
// contiguous x-row slot ranges) and records, per row, a 32/64-bit mask of the
// slots within a skin radius h_s >= h (of its first 96 slots; RowMasks).
// The normals, forces and XSPH passes walk those masks over packed neighbour
// data (XSPH when the substep's largest move proves them complete; otherwise
// it makes such masks from the moved positions) and re-test each pair; set
// bits are visited in slot order, so every pass sums the same neighbours in
// the same order as a full stencil scan, bit for bit.
//
// SPH here is a gather-bound stencil, not a dense contraction: the kernels
// are VALU/L1 work over the stencil walk and never use MFMA.

#include <hip/hip_ext.h>

#include <algorithm>

#include "lf_device.h"
#include "lf_kernels.h"

namespace lf {

// ---------------------------------------------------------------------------
// 1. hash + count (PointHashOperator, hash.cu:10-27; fill fluidsystem.cu:304).
// The value returned by the count atomic is the particle's provisional rank
// inside its bucket.  Particles arrive in the previous cell order, so runs of
// lanes share a bucket: each run issues one atomic for its length and hands
// out consecutive ranks.  Counts are zeroed by the previous substep's scan
// or scatter.
// Each thread takes kHashItems particles, kBlock slots apart, whose loads
// and count atomics are issued together (the pass is latency bound).
constexpr int kHashItems = 2;
__global__ __launch_bounds__(kBlock) void k_hash(const Consts *__restrict__ cs, const uint32_t *__restrict__ chunk,
                                                 const float4 *__restrict__ P, uint32_t *__restrict__ keys,
                                                 uint32_t *__restrict__ ranks, uint32_t *__restrict__ counts,
                                                 uint32_t *__restrict__ flags, uint32_t *__restrict__ moves,
                                                 uint32_t *__restrict__ nsegs) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *nsegs = 0u;  // large buckets of the substep, listed by k_scatter
    uint32_t slot0;
    const Consts *cp = block_scene<kBlock * kHashItems>(cs, chunk, slot0);
    if (!cp) return;
    const Consts &c = *cp;
    const int lane = threadIdx.x & 63;
    uint32_t i[kHashItems], b[kHashItems], base[kHashItems];
    int first[kHashItems], next[kHashItems];
    bool active[kHashItems];
    float4 p[kHashItems];
#pragma unroll
    for (int q = 0; q < kHashItems; ++q) {
        i[q] = slot0 + (uint32_t)(q * kBlock) + threadIdx.x;
        active[q] = i[q] < c.first + c.count;
        p[q] = active[q] ? P[i[q]] : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int q = 0; q < kHashItems; ++q) {
        if (i[q] == c.first) set_flag(flags, c.scene, kFragileByte, 0u);  // set by k_density
        if (i[q] - c.first < kMoveSlots) *move_slot(moves, c.scene, i[q] - c.first) = 0u;  // raised by k_gather
        b[q] = active[q] ? c.cell_base + bucket_of(c, p[q]) : 0xFFFFFFFFu;
        const uint32_t prev = __shfl_up(b[q], 1, 64);
        const bool head = lane == 0 || prev != b[q];
        const uint64_t heads = __ballot(head);
        const uint64_t upto = (lane == 63) ? ~0ull : ((1ull << (lane + 1)) - 1ull);
        first[q] = 63 - __clzll(heads & upto);
        const uint64_t above = heads & ~upto;
        next[q] = above ? __ffsll((unsigned long long)above) - 1 : 64;
    }
#pragma unroll
    for (int q = 0; q < kHashItems; ++q) {
        base[q] = 0u;
        if (active[q] && lane == first[q]) base[q] = atomicAdd(&counts[b[q]], (uint32_t)(next[q] - first[q]));
    }
#pragma unroll
    for (int q = 0; q < kHashItems; ++q) {
        const uint32_t bq = __shfl(base[q], first[q], 64);
        if (active[q]) {
            keys[i[q]] = b[q];
            ranks[i[q]] = bq + (uint32_t)(lane - first[q]);
        }
    }
}

// ---------------------------------------------------------------------------
// 2. cell start table: exclusive scan of the bucket counts
// (thrust::exclusive_scan, fluidsystem.cu:316), two phases over all buckets
// of the pool.

__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        uint32_t t = __shfl_up(v, o, 64);
        if (lane >= o) v += t;
    }
    return v;
}

__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t *sh, uint32_t &total) {
    const uint32_t incl = wave_incl_scan(v);
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 63) sh[w] = incl;
    __syncthreads();
    uint32_t off = 0, tot = 0;
#pragma unroll
    for (int k = 0; k < kBlock / 64; ++k) {
        const uint32_t t = sh[k];
        off += (k < w) ? t : 0u;
        tot += t;
    }
    __syncthreads();
    total = tot;
    return off + incl - v;
}

// The counts of one thread: kScanPerThread (= 4) consecutive buckets from
// `base`, one 16-byte load (tiles start at multiples of kScanTile, so base is
// 16-byte aligned) except in the last, partial tile.
__device__ __forceinline__ uint4 scan_load(const uint32_t *__restrict__ counts, uint32_t base, uint32_t m) {
    if (base + 4u <= m) return *reinterpret_cast<const uint4 *>(counts + base);
    return make_uint4(base < m ? counts[base] : 0u, base + 1u < m ? counts[base + 1u] : 0u,
                      base + 2u < m ? counts[base + 2u] : 0u, base + 3u < m ? counts[base + 3u] : 0u);
}

// Phase 1: the sum of each tile of kScanTile buckets.
__global__ __launch_bounds__(kBlock) void k_scan_sum(const uint32_t *__restrict__ counts, uint32_t m,
                                                     uint32_t *__restrict__ bsum) {
    __shared__ uint32_t sh[kBlock / 64];
    const uint4 v = scan_load(counts, blockIdx.x * kScanTile + threadIdx.x * kScanPerThread, m);
    uint32_t tot;
    (void)block_excl_scan(v.x + v.y + v.z + v.w, sh, tot);
    if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}

// Phase 1b, for more than kScanDirectTiles tiles: one workgroup turns the
// tile sums into exclusive prefixes in place, kScanTile of them per step.
__global__ __launch_bounds__(kBlock) void k_scan_tiles(uint32_t *__restrict__ bsum, uint32_t nb) {
    __shared__ uint32_t sh[kBlock / 64];
    uint32_t carry = 0;
    for (uint32_t t0 = 0; t0 < nb; t0 += kScanTile) {
        const uint32_t base = t0 + threadIdx.x * kScanPerThread;
        const uint4 v = scan_load(bsum, base, nb);
        uint32_t tot;
        const uint32_t run = carry + block_excl_scan(v.x + v.y + v.z + v.w, sh, tot);
        const uint32_t sv[4] = {run, run + v.x, run + v.x + v.y, run + v.x + v.y + v.z};
        for (uint32_t k = 0; k < 4u; ++k)
            if (base + k < nb) bsum[base + k] = sv[k];
        carry += tot;
    }
}

// Phase 2: each tile takes the sum of the tiles before it (prefixed: phase
// 1b's prefix; else it adds up their sums, at most kScanDirectTiles, cached),
// scans its own buckets, writes their starts and clears their counts for the
// next substep; the last tile writes the end sentinel start[m].
__global__ __launch_bounds__(kBlock) void k_scan_down(uint32_t *__restrict__ counts, uint32_t m,
                                                      const uint32_t *__restrict__ bsum, uint32_t nb,
                                                      int prefixed, uint32_t *__restrict__ start) {
    __shared__ uint32_t sh[kBlock / 64];
    uint32_t prefix;
    if (prefixed) {
        prefix = bsum[blockIdx.x];
    } else {
        uint32_t before = 0, t = threadIdx.x;
        for (; t + 3u * kBlock < blockIdx.x; t += 4u * kBlock)  // four loads in flight
            before += bsum[t] + bsum[t + kBlock] + bsum[t + 2u * kBlock] + bsum[t + 3u * kBlock];
        for (; t < blockIdx.x; t += kBlock) before += bsum[t];
        (void)block_excl_scan(before, sh, prefix);
    }
    const uint32_t base = blockIdx.x * kScanTile + threadIdx.x * kScanPerThread;
    const uint4 v = scan_load(counts, base, m);
    uint32_t tot;
    const uint32_t run = prefix + block_excl_scan(v.x + v.y + v.z + v.w, sh, tot);
    const uint4 st = make_uint4(run, run + v.x, run + v.x + v.y, run + v.x + v.y + v.z);
    if (base + 4u <= m) {
        *reinterpret_cast<uint4 *>(start + base) = st;
        *reinterpret_cast<uint4 *>(counts + base) = make_uint4(0u, 0u, 0u, 0u);
    } else {
        const uint32_t sv[4] = {st.x, st.y, st.z, st.w};
        for (uint32_t k = 0; k < 4u && base + k < m; ++k) {
            start[base + k] = sv[k];
            counts[base + k] = 0u;
        }
    }
    if (blockIdx.x == nb - 1u && threadIdx.x == 0) start[m] = prefix + tot;
}

// The scan of at most kScanOneTiles tiles of kScanOneTile buckets in one
// launch: each workgroup adds up the counts of every tile before its own
// (eight 16-byte loads in flight per thread) instead of waiting for a first
// launch to do so: a replayed substep of 2,000 particles 46.0 -> 44.4 us, of
// 60,000 (64,000 buckets) 64.5 -> 63.9; at 20 tiles the two ways are even.
// The counts are cleared by k_scatter, as other workgroups still read them
// here.
constexpr int kScanOneThreads = 1024;
constexpr uint32_t kScanOneTile = 4u * kScanOneThreads, kScanOneTiles = 16u;
__global__ __launch_bounds__(kScanOneThreads) void k_scan_one(const uint32_t *__restrict__ counts, uint32_t m,
                                                              uint32_t *__restrict__ start) {
    __shared__ uint32_t before_w[kScanOneThreads / 64], own_w[kScanOneThreads / 64];
    const uint32_t t = threadIdx.x, lane = t & 63u, w = t >> 6;
    const uint32_t base = blockIdx.x * kScanOneTile + 4u * t;
    const uint4 v = scan_load(counts, base, m);
    uint32_t before = 0u;
    for (uint32_t k0 = 0u; k0 < blockIdx.x; k0 += 8u) {  // tiles before this one: all whole
        uint4 x[8];
#pragma unroll
        for (uint32_t k = 0u; k < 8u; ++k) {
            const uint32_t tile = k0 + k < blockIdx.x ? k0 + k : 0u;
            x[k] = *reinterpret_cast<const uint4 *>(counts + tile * kScanOneTile + 4u * t);
        }
#pragma unroll
        for (uint32_t k = 0u; k < 8u; ++k)
            if (k0 + k < blockIdx.x) before += x[k].x + x[k].y + x[k].z + x[k].w;
    }
    const uint32_t own = v.x + v.y + v.z + v.w;
    const uint32_t incl = wave_incl_scan(own), all = wave_incl_scan(before);
    if (lane == 63u) {
        own_w[w] = incl;
        before_w[w] = all;
    }
    __syncthreads();
    uint32_t run = incl - own, total = 0u;
#pragma unroll
    for (uint32_t k = 0u; k < kScanOneThreads / 64; ++k) {
        run += before_w[k] + (k < w ? own_w[k] : 0u);
        total += before_w[k] + own_w[k];
    }
    const uint32_t sv[4] = {run, run + v.x, run + v.x + v.y, run + v.x + v.y + v.z};
    if (base + 4u <= m)
        *reinterpret_cast<uint4 *>(start + base) = make_uint4(sv[0], sv[1], sv[2], sv[3]);
    else
        for (uint32_t k = 0u; k < 4u && base + k < m; ++k) start[base + k] = sv[k];
    if (blockIdx.x == gridDim.x - 1u && t == 0u) start[m] = total;
}

// ---------------------------------------------------------------------------
// Slot of the first particle of pool bucket b of scene c:
//   first + (start[b] - start[cell_base]) = start[b] + shift.
__device__ __forceinline__ uint32_t slot_shift(const Consts &c, const uint32_t *__restrict__ start) {
    return c.first - start[c.cell_base];
}

// 3b. segments (buckets of more than kRankDirectMax particles) sorted by id
// in place: (slot_id, slot_src) of slots [lo, lo + size), by one workgroup of
// NT threads, segment after segment (k_sort_segments, after k_scatter): an LSD radix sort by 8 bits of the id
// per pass, through tmp (same slots) and back.  A pass counts the digits,
// then places the segment tile by tile (NT elements, in slot order): a
// member's new place is the digit's running base, plus that digit's count
// in the tile's earlier waves, plus its rank among the earlier lanes of its
// wave with the same digit (lanes matched by eight ballots), so every pass
// is stable.  Ids are unique within a scene.
__device__ __forceinline__ uint32_t seg_digit(uint32_t id, uint32_t shift) { return (id >> shift) & 0xFFu; }

template <int NT>
struct SegSortLds {
    uint32_t base[256];               // running start of each digit in the destination
    uint32_t wcnt[NT / 64][256];      // per wave: digit counts, then their prefix over waves
    uint32_t scan_tot[4];
};

template <int NT>
__device__ void sort_segments(SegSortLds<NT> &sh, const uint4 *__restrict__ segs, uint32_t nseg,
                              uint32_t *__restrict__ slot_id, uint32_t *__restrict__ slot_src,
                              uint2 *__restrict__ tmp) {
    static_assert(NT >= 256 && NT % 64 == 0, "the digit scan needs four waves");
    constexpr int kWaves = NT / 64;
    const uint32_t t = threadIdx.x, lane = t & 63u, w = t >> 6;
    const uint64_t below = (1ull << lane) - 1ull;
    for (uint32_t sg = 0; sg < nseg; ++sg) {
        const uint4 g = segs[sg];
        const uint32_t lo = g.x, n = g.y, passes = (g.z + 7u) / 8u;
        for (uint32_t p = 0; p < passes; ++p) {
            const bool from_tmp = (p & 1u) != 0u;
            const uint32_t shift = 8u * p;
            if (t < 256u) sh.base[t] = 0u;
            __syncthreads();
            for (uint32_t k = t; k < n; k += NT) {
                const uint32_t id = from_tmp ? tmp[lo + k].x : slot_id[lo + k];
                atomicAdd(&sh.base[seg_digit(id, shift)], 1u);
            }
            __syncthreads();
            // exclusive scan of the 256 digit counts (waves 0-3)
            uint32_t v = 0u, incl = 0u;
            if (t < 256u) {
                v = sh.base[t];
                incl = v;
#pragma unroll
                for (int o = 1; o < 64; o <<= 1) {
                    const uint32_t u = __shfl_up(incl, o, 64);
                    if ((int)lane >= o) incl += u;
                }
                if (lane == 63u) sh.scan_tot[w] = incl;
            }
            __syncthreads();
            if (t < 256u) {
                uint32_t off = 0u;
                for (uint32_t q = 0; q < w; ++q) off += sh.scan_tot[q];
                sh.base[t] = off + incl - v;
            }
            __syncthreads();
            for (uint32_t tile = 0; tile < n; tile += NT) {
                for (uint32_t q = t; q < kWaves * 256u; q += NT) (&sh.wcnt[0][0])[q] = 0u;
                __syncthreads();
                const uint32_t k = tile + t;
                const bool valid = k < n;
                uint2 e = make_uint2(0u, 0u);
                if (valid) e = from_tmp ? tmp[lo + k] : make_uint2(slot_id[lo + k], slot_src[lo + k]);
                const uint32_t d = seg_digit(e.x, shift);
                uint64_t peers = __ballot(valid);
#pragma unroll
                for (uint32_t bit = 0; bit < 8u; ++bit) {
                    const bool on = ((d >> bit) & 1u) != 0u;
                    const uint64_t m = __ballot(on);
                    peers &= on ? m : ~m;
                }
                const uint32_t rank = (uint32_t)__popcll(peers & below);
                if (valid && rank == 0u) sh.wcnt[w][d] = (uint32_t)__popcll(peers);
                __syncthreads();
                uint32_t tile_total = 0u;
                if (t < 256u) {  // prefix of digit t's counts over the waves
                    for (uint32_t q = 0; q < (uint32_t)kWaves; ++q) {
                        const uint32_t c = sh.wcnt[q][t];
                        sh.wcnt[q][t] = tile_total;
                        tile_total += c;
                    }
                }
                __syncthreads();
                if (valid) {
                    const uint32_t dst = lo + sh.base[d] + sh.wcnt[w][d] + rank;
                    if (from_tmp) {
                        slot_id[dst] = e.x;
                        slot_src[dst] = e.y;
                    } else {
                        tmp[dst] = e;
                    }
                }
                __syncthreads();
                if (t < 256u) sh.base[t] += tile_total;
                __syncthreads();
            }
        }
        if (passes & 1u) {  // the last pass wrote tmp
            for (uint32_t k = t; k < n; k += NT) {
                const uint2 e = tmp[lo + k];
                slot_id[lo + k] = e.x;
                slot_src[lo + k] = e.y;
            }
        }
        __syncthreads();
    }
}

// 3. provisional scatter: slot = bucket start + atomic rank.  The particle
// with rank 0 of a bucket of more than kRankDirectMax particles lists the
// bucket's slot range as a segment for k_sort_segments: (first slot, size,
// bits of the scene's largest id).  After a scan in one launch (k_scan_one,
// whose workgroups read each other's counts) it clears the counts [0, clear)
// for the next substep.
__global__ __launch_bounds__(kBlock) void k_scatter(const Consts *__restrict__ cs, const uint32_t *__restrict__ chunk,
                                                    const float4 *__restrict__ P, const uint32_t *__restrict__ keys,
                                                    const uint32_t *__restrict__ ranks,
                                                    const uint32_t *__restrict__ start,
                                                    uint32_t *__restrict__ slot_src, uint32_t *__restrict__ slot_id,
                                                    uint4 *__restrict__ segs, uint32_t *__restrict__ nsegs,
                                                    uint32_t *__restrict__ counts, uint32_t clear) {
    for (uint32_t k = blockIdx.x * kBlock + threadIdx.x; k < clear; k += gridDim.x * kBlock) counts[k] = 0u;
    uint32_t slot0;
    const Consts *cp = block_scene<kBlock>(cs, chunk, slot0);
    if (!cp) return;
    const uint32_t i = slot0 + threadIdx.x;
    if (i >= cp->first + cp->count) return;
    const uint32_t b = keys[i], r = ranks[i];
    const uint32_t lo = start[b] + slot_shift(*cp, start);
    const uint32_t s = lo + r;
    slot_src[s] = i;
    slot_id[s] = __float_as_uint(P[i].w);
    if (r == 0u) {
        const uint32_t size = start[b + 1] - start[b];
        if (size > kRankDirectMax) {
            const uint32_t bits = cp->count > 1u ? 32u - (uint32_t)__clz(cp->count - 1u) : 1u;
            segs[atomicAdd(nsegs, 1u)] = make_uint4(lo, size, bits, 0u);
        }
    }
}

// 3c. the listed segments, one workgroup each (grid stride over the list;
// a workgroup with no segment exits at once).  (A ticket taken by every
// workgroup of the scatter pass, to let its last workgroup sort, needs a
// device-scope fence per wave, which costs far more than this launch.)
constexpr int kSegThreads = 1024;
constexpr int kSegBlocks = 32;
__global__ __launch_bounds__(kSegThreads) void k_sort_segments(const uint4 *__restrict__ segs,
                                                               const uint32_t *__restrict__ nsegs,
                                                               uint32_t *__restrict__ slot_id,
                                                               uint32_t *__restrict__ slot_src,
                                                               uint2 *__restrict__ tmp) {
    __shared__ SegSortLds<kSegThreads> sh;
    const uint32_t nseg = *nsegs;
    for (uint32_t sg = blockIdx.x; sg < nseg; sg += gridDim.x)
        sort_segments<kSegThreads>(sh, segs + sg, 1u, slot_id, slot_src, tmp);
}

// 4. stable placement + payload gather (sort_by_key of Points, Velocity,
// Acceleration, fluidsystem.cu:309-313).  The final slot of a particle is
// its bucket start plus the number of bucket members with a smaller id, so
// the order is (key, id) whatever order the atomics handed out; a bucket of
// more than kRankDirectMax particles has been sorted by id in place
// (k_sort_segments), so there the provisional slot is the final one.  Position
// and velocity are copied to cell order (the neighbour passes gather them);
// the acceleration and the position's low word, which only the particle's
// own integration reads, stay where they are: order[f] records the state
// slot the particle in slot f came from.
__global__ __launch_bounds__(kBlock) void k_gather(const Consts *__restrict__ cs, const uint32_t *__restrict__ chunk,
                                                   const uint32_t *__restrict__ slot_src,
                                                   const uint32_t *__restrict__ slot_id,
                                                   const uint32_t *__restrict__ keys,
                                                   const uint32_t *__restrict__ start, const float4 *__restrict__ P,
                                                   const float4 *__restrict__ V,
                                                   float4 *__restrict__ Ps, float4 *__restrict__ Vs,
                                                   uint32_t *__restrict__ order, float *__restrict__ soa,
                                                   uint32_t nslots, uint8_t *__restrict__ near,
                                                   uint32_t *__restrict__ moves) {
    uint32_t slot0;
    const Consts *cp = block_scene<kBlock>(cs, chunk, slot0);
    if (!cp) return;
    const uint32_t s = slot0 + threadIdx.x;
    uint32_t q = 0u;
    if (s < cp->first + cp->count) {
        const uint32_t src = slot_src[s], id = slot_id[s];
        const uint32_t b = keys[src];
        const uint32_t shift = slot_shift(*cp, start);
        const uint32_t lo = start[b] + shift, hi = start[b + 1] + shift;
        uint32_t f = s;
        if (hi - lo <= kRankDirectMax) {
            // four members' ids loaded together per step
            uint32_t r = 0, t = lo;
            for (; t + 4u <= hi; t += 4u) {
                const uint32_t a0 = slot_id[t], a1 = slot_id[t + 1u], a2 = slot_id[t + 2u], a3 = slot_id[t + 3u];
                r += (a0 < id ? 1u : 0u) + (a1 < id ? 1u : 0u) + (a2 < id ? 1u : 0u) + (a3 < id ? 1u : 0u);
            }
            for (; t < hi; ++t) r += (slot_id[t] < id) ? 1u : 0u;
            f = lo + r;
        }
        const float4 p = P[src], v = V[src];
        Ps[f] = p;
        soa[f] = p.x;
        soa[nslots + f] = p.y;
        soa[2 * (size_t)nslots + f] = p.z;
        Vs[f] = v;
        order[f] = src;
        q = skin_quantum(*cp, v);
        if (s % kNearBlock == 0u) near[s / kNearBlock] = 0u;  // marked again by k_density
    }
    // The scene's largest move of the substep (XSPH skin): reduced over the
    // workgroup, then one atomicMax into the slot of the workgroup's index.
    __shared__ uint32_t wq[kBlock / 64];
    q = wave_max<10>(q);
    if ((threadIdx.x & 63u) == 0u) wq[threadIdx.x >> 6] = q;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t m = wq[0];
#pragma unroll
        for (int w = 1; w < kBlock / 64; ++w) m = m > wq[w] ? m : wq[w];
        atomicMax(move_slot(moves, cp->scene, blockIdx.x % kMoveSlots), m);
    }
}

// ---------------------------------------------------------------------------
// Neighbour rows.  The clipped 27-cell stencil of a cell is nine contiguous
// slot ranges (x-rows, z outer, y inner: the reference's visiting order of
// cells, fluidphysics.cu:30-53, up to the order inside a row).  rows9 issues
// the eighteen start-table loads together; rows outside the grid are empty.
// `start` is the scene's own table, `shift` its slot_shift.
__device__ __forceinline__ void rows9(const Consts &c, const uint32_t *__restrict__ start, uint32_t shift, float4 pc,
                                      uint32_t *b, uint32_t *e) {
    int cx, cy, cz;
    cell_xyz(c, pc, cx, cy, cz);
    const int x0 = cx > 0 ? cx - 1 : 0, x1 = cx < c.gx - 1 ? cx + 1 : c.gx - 1;
#pragma unroll
    for (int r = 0; r < 9; ++r) {
        const int z = cz + r / 3 - 1, y = cy + r % 3 - 1;
        const bool ok = z >= 0 && z < c.gz && y >= 0 && y < c.gy;
        const uint32_t row = (uint32_t)((ok ? z : cz) * c.gy + (ok ? y : cy)) * (uint32_t)c.gx;
        const uint32_t bb = start[row + (uint32_t)x0] + shift;
        const uint32_t ee = start[row + (uint32_t)x1 + 1u] + shift;
        b[r] = bb;
        e[r] = ok ? ee : bb;
    }
}

// The density pass records, per row, a mask of the row's slots within the
// skin radius (bit k = slot b[r] + k), a superset of the neighbours within h,
// which the callbacks re-test.  walk_masks visits the set bits in increasing
// slot order, the
// same order as a full scan; a row longer than 64 slots is scanned in full
// (walk_flat does better).  With use == false every row is scanned.  Each step takes
// up to W set bits of the row and issues all their candidates' loads (ld)
// before using them (fn, in slot order), so W gathers per lane are in flight
// at a time.  fn(cand, slot, ok) adds nothing when ok is false (a step with
// fewer set bits left passes its first slot again with ok = false and, as
// that candidate, whatever finite values the previous step loaded there);
// calling it unconditionally keeps the later candidates' loads ahead of the
// first candidate's arithmetic.
// The pair walk (PAIR) passes ok as the wave's lane mask, as the compare that
// gave it left it: a bool kept across the loads was turned into 0 / 1 in a
// register and compared again.
struct LaneMask {
    uint64_t lanes;
};
__device__ __forceinline__ uint64_t lane_mask(bool ok) { return lanes(ok); }
__device__ __forceinline__ uint64_t lane_mask(LaneMask ok) { return ok.lanes; }
template <int W, bool PAIR = false, class Ld, class Fn>
__device__ __forceinline__ void walk_masks(const uint32_t *b, const uint32_t *e, const RowMasks &mask, bool use,
                                           uint32_t nslots, uint32_t i, Ld &&ld, Fn &&fn) {
    uint64_t mk[9];
    // A step's candidates past the lane's last set bit (ok = false) load
    // nothing and keep the previous step's values (finite: zero at first).
    decltype(ld(0u)) a[W] = {};
#pragma unroll
    for (int r = 0; r < 9; ++r) {
        const uint32_t len = e[r] - b[r];
        const size_t at = (size_t)r * nslots + i;
        mk[r] = 0ull;
        if (use && len <= 32u) mk[r] = mask.w32[at];
        else if (use && len <= 64u) mk[r] = mask.w64[at];
    }
    if constexpr (PAIR) {
        // Where every row of the wave fits 32 slots, rows are walked in
        // pairs, row 2g's mask word and then row 2g + 1's, so a step's
        // padding is paid per pair, not per row.  Bits stay in slot order.
        // (Two 32-bit words and a count of the bits left take nine VALU
        // instructions a bit where a 64-bit stream took twelve, and no
        // spills: XSPH of the column 65.9 -> 64.8 us, of 262,144 spray
        // particles 23.2 -> 21.7.)
        bool lng = !use;
#pragma unroll
        for (int r = 0; r < 9; ++r) lng = lng || e[r] - b[r] > 32u;
        if (!__ballot(lng)) {
#pragma unroll
            for (int g = 0; g < 5; ++g) {
                const int r0 = 2 * g, r1 = 2 * g + 1;
                uint32_t lo = (uint32_t)mk[r0], hi = r1 < 9 ? (uint32_t)mk[r1] : 0u;
                const uint32_t b0 = b[r0], b1 = r1 < 9 ? b[r1] : 0u;
                int left = __popc(lo) + __popc(hi);
                while (left > 0) {
                    uint32_t j[W];
                    uint64_t ok[W];  // lane masks
#pragma unroll
                    for (int k = 0; k < W; ++k) {
                        ok[k] = k ? lanes(left > k) : ~0ull;
                        const bool first = lo != 0u;
                        const uint32_t w = first ? lo : hi;
                        const uint32_t next = w & (w - 1u);
                        j[k] = (first ? b0 : b1) + (uint32_t)__builtin_ctz(w);
                        lo = first ? next : 0u;
                        hi = first ? hi : next;
                    }
                    a[0] = ld(j[0]);
#pragma unroll
                    for (int k = 1; k < W; ++k)
                        if (left > k) a[k] = ld(j[k]);
#pragma unroll
                    for (int k = 0; k < W; ++k) fn(a[k], j[k], LaneMask{ok[k]});
                    left -= W;
                }
            }
            return;
        }
    }
#pragma unroll
    for (int r = 0; r < 9; ++r) {
        if (use && e[r] - b[r] <= 64u) {
            uint64_t m = mk[r];
            while (m) {
                uint32_t j[W];
                bool ok[W];
                j[0] = b[r] + (uint32_t)__ffsll((unsigned long long)m) - 1u;
                ok[0] = true;
                m &= m - 1ull;
#pragma unroll
                for (int k = 1; k < W; ++k) {
                    ok[k] = m != 0ull;
                    j[k] = ok[k] ? b[r] + (uint32_t)__ffsll((unsigned long long)m) - 1u : j[0];
                    m &= m - 1ull;  // stays 0 when it was 0
                }
                a[0] = ld(j[0]);
#pragma unroll
                for (int k = 1; k < W; ++k)
                    if (ok[k]) a[k] = ld(j[k]);
#pragma unroll
                for (int k = 0; k < W; ++k) fn(a[k], j[k], ok[k]);
            }
        } else {
            for (uint32_t j = b[r]; j < e[r]; ++j)
                if (j != i) fn(ld(j), j, true);
        }
    }
}

// Row r (wave-uniform) of the particle at pc: its first slot and its end,
// as rows9 gives them.
__device__ __forceinline__ uint2 row_span(const Consts &c, const uint32_t *__restrict__ start, uint32_t shift,
                                          float4 pc, uint32_t r) {
    int cx, cy, cz;
    cell_xyz(c, pc, cx, cy, cz);
    const int x0 = cx > 0 ? cx - 1 : 0, x1 = cx < c.gx - 1 ? cx + 1 : c.gx - 1;
    const int z = cz + (int)(r / 3u) - 1, y = cy + (int)(r % 3u) - 1;
    const bool ok = z >= 0 && z < c.gz && y >= 0 && y < c.gy;
    const uint32_t row = (uint32_t)((ok ? z : cz) * c.gy + (ok ? y : cy)) * (uint32_t)c.gx;
    const uint32_t bb = start[row + (uint32_t)x0] + shift;
    const uint32_t ee = start[row + (uint32_t)x1 + 1u] + shift;
    return make_uint2(bb, ok ? ee : bb);
}

// Long rows.  What the walks need to find a row's mask words without the
// row table in registers: the scene, its cell table, the pre-integration
// positions (also as planes) and the largest move, which gives the skin
// radius of the density pass; and, for XSPH in a scene whose masks are not
// complete, the integrated positions to test instead (moved; null elsewhere).
struct RowSource {
    const Consts &c;
    const uint32_t *__restrict__ st;
    uint32_t shift;
    const float4 *__restrict__ pos;  // pre-integration positions, cell order
    const float *__restrict__ soa;
    const uint32_t *__restrict__ moves;
    const float4 *__restrict__ moved;
};

// Mask word of up to 32 slots [s, s + n) (n of them, at most 32 used),
// tested against the skin radius exactly as the density pass tests them.
__device__ __forceinline__ uint32_t skin_word(const RowSource &src, uint32_t nslots, float4 pc, uint32_t s,
                                              uint32_t n, uint32_t i) {
    const __amdgpu_buffer_rsrc_t px = plane_buffer(src.soa, nslots), py = plane_buffer(src.soa + nslots, nslots),
                                 pz = plane_buffer(src.soa + 2 * (size_t)nslots, nslots);
    const float nh2s = -skin_h2s(src.c, skin_frac(scene_move_q(src.moves, src.c.scene)));
    const uint32_t off = s * (uint32_t)sizeof(float);
    uint32_t cur = 0u;
    auto test = [&](float qx, float qy, float qz) {
        const float dx = qx - pc.x, dy = qy - pc.y, dz = qz - pc.z;
        const float rs = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, __builtin_fmaf(dx, dx, nh2s)));
        cur = __builtin_amdgcn_alignbit(cur, __float_as_uint(rs), 31u);
    };
#pragma unroll 1
    for (uint32_t so = 0u; so < 32u * (uint32_t)sizeof(float); so += 4u * (uint32_t)sizeof(float)) {
        const float4 X = load4(px, off, so), Y = load4(py, off, so), Z = load4(pz, off, so);
        test(X.x, Y.x, Z.x);
        test(X.y, Y.y, Z.y);
        test(X.z, Y.z, Z.z);
        test(X.w, Y.w, Z.w);
    }
    uint32_t m = __brev(cur);
    if (n < 32u) m &= (1u << n) - 1u;
    const uint32_t k = i - s;  // the particle itself is no candidate
    if (k < 32u) m &= ~(1u << k);
    return m;
}

// Mask word of up to 32 slots [s, s + n) by the integrated positions: those
// within h (the pair test of the XSPH walk itself).
__device__ __forceinline__ uint32_t moved_word(const RowSource &src, uint32_t s, uint32_t n, uint32_t i) {
    uint32_t cur = 0u;
    if (n > 32u) n = 32u;
    const float4 xi = at32(src.moved, i);
#pragma unroll 1
    for (uint32_t g = 0u; g < n; g += 4u) {
        float4 q[4];
#pragma unroll
        for (uint32_t k = 0u; k < 4u; ++k) q[k] = at32(src.moved, g + k < n ? s + g + k : s);
#pragma unroll
        for (uint32_t k = 0u; k < 4u; ++k)
            cur |= g + k < n && dist2(xi, q[k]) <= src.c.h2 ? 1u << (g + k) : 0u;
    }
    const uint32_t k = i - s;  // the particle itself is no candidate
    if (k < 32u) cur &= ~(1u << k);
    return cur;
}

// The stored mask of a row's first 64 slots by one unconditional 8-byte load:
// from the 64-bit array for a row of more than 32 slots, else from the 32-bit
// array, whose allocation is padded so that the word after the last entry is
// readable (that second word is dropped).
__device__ __forceinline__ uint64_t row_mask64(const RowMasks &mask, size_t at, uint32_t len) {
    const char *p = len > 32u ? reinterpret_cast<const char *>(mask.w64 + at)
                              : reinterpret_cast<const char *>(mask.w32 + at);
    uint64_t v;
    __builtin_memcpy(&v, p, sizeof(v));
    return len > 32u ? v : (v & 0xFFFFFFFFull);
}

// Fills the lane's column of the flattened walk's table with its next
// pseudo-rows, from word `word` of row `row` on (both wave-uniform, left at
// the first pseudo-row that did not fit), and returns how many it stored.
// The first three words of a row come from the density pass's masks; later
// ones (rows of more than 96 slots) are tested again here, 7 VALU
// instructions a candidate against the 25 to 60 of the walk it spares.  Row
// bounds and words are loaded anew for each batch, two rows and one row
// ahead of their use, instead of being held in registers through the walk.
// With src.moved every word is tested on the integrated positions.
template <int BS>
__device__ __forceinline__ uint32_t fill_long(uint2 *__restrict__ tab, const RowSource &src, const RowMasks &mask,
                                              uint32_t nslots, uint32_t i, uint32_t &row, uint32_t &word) {
    const uint32_t t = threadIdx.x;
    struct Span {
        uint32_t s, len;
    };
    struct Words {
        uint64_t w01;
        uint32_t w2;
    };
    const float4 pc = at32(src.pos, i);
    const auto span = [&](uint32_t r) {
        const uint2 x = row_span(src.c, src.st, src.shift, pc, r < 9u ? r : 8u);
        return Span{x.x, x.y - x.x};
    };
    const auto words = [&](uint32_t r, uint32_t len) {
        const size_t at = (size_t)(r < 9u ? r : 8u) * nslots + i;
        return Words{row_mask64(mask, at, len), mask.w32[at]};  // w2: slots 64..95 of a row of more than 64
    };
    Span cur = span(row), nxt = span(row + 1u);
    Words w = words(row, cur.len);
    uint32_t cnt = 0u, used = 0u;
#pragma unroll 1
    while (row < 9u) {
        const Words wn = words(row + 1u, nxt.len);
        const Span nn = span(row + 2u);
#pragma unroll 1
        for (; __ballot(cur.len > 32u * word); ++word) {
            if (used == (uint32_t)kFlatEntries) return cnt;
            const bool in = cur.len > 32u * word;
            uint32_t m = word == 0u ? (uint32_t)w.w01 : word == 1u ? (uint32_t)(w.w01 >> 32) : w.w2;
            if (src.moved)
                m = in ? moved_word(src, cur.s + 32u * word, cur.len - 32u * word, i) : 0u;
            else if (word >= 3u)
                m = in ? skin_word(src, nslots, pc, cur.s + 32u * word, cur.len - 32u * word, i) : 0u;
            if (in && m != 0u) {
                tab[cnt * BS + t] = make_uint2(m, cur.s + 32u * word);
                ++cnt;
            }
            ++used;
        }
        word = 0u;
        ++row;
        cur = nxt;
        w = wn;
        nxt = nn;
    }
    return cnt;
}

// Visits the set bits of the lane's first cnt table entries, W per step.
template <int BS, int W, class Ld, class Fn>
__device__ __forceinline__ void walk_table(const uint2 *__restrict__ tab, uint32_t cnt, Ld &&ld, Fn &&fn) {
    const uint32_t t = threadIdx.x;
    const uint2 e0 = tab[t];
    uint32_t m = cnt > 0u ? e0.x : 0u, base = e0.y;
    uint2 nx = tab[BS + t];  // entry nxt as read: used only if nxt < cnt
    uint32_t nxt = 1u;
    auto advance = [&]() {  // the current pseudo-row is used up: take entry nxt, fetch the one after
        m = nxt < cnt ? nx.x : 0u;
        base = nx.y;
        ++nxt;
        nx = tab[(nxt < (uint32_t)kFlatEntries ? nxt : 0u) * BS + t];
    };
    decltype(ld(0u)) a[W] = {};  // as in walk_masks: ok = false loads nothing
    while (m) {
        uint32_t j[W];
        bool ok[W];
        j[0] = base + (uint32_t)__builtin_ctz(m);
        ok[0] = true;
        m &= m - 1u;
        if (!m) advance();
#pragma unroll
        for (int k = 1; k < W; ++k) {  // once a bit is missing, so are the rest
            ok[k] = m != 0u;
            j[k] = ok[k] ? base + (uint32_t)__builtin_ctz(m) : j[0];
            if (ok[k]) {
                m &= m - 1u;
                if (!m) advance();
            }
        }
        a[0] = ld(j[0]);
#pragma unroll
        for (int k = 1; k < W; ++k)
            if (ok[k]) a[k] = ld(j[k]);
#pragma unroll
        for (int k = 0; k < W; ++k) fn(a[k], j[k], ok[k]);
    }
}

// Flattened walk of the nine rows' masks.  Iterating row by row costs every
// row the longest run of any lane in the wave; one stream of set bits over
// all rows costs only the largest total.  Each lane splits its rows into
// pseudo-rows of at most 32 slots (a row of 33..64 slots is two: its 64-bit
// mask's low and high words, the second starting 32 slots later), compacts
// the non-empty ones, (mask, first slot), into its own column of the
// workgroup's LDS table tab[kFlatEntries][BS] and walks them in row order,
// W set bits per step (consecutive bits may come from adjacent pseudo-rows):
// the W candidates' loads are all issued before the first is used, so W
// gathers per lane are in flight.  The next entry is fetched one entry
// ahead, so a row change does not wait on LDS.  Visits the same slots in the
// same order as walk_masks.
//
// A wave in which a lane has a row of more than 64 slots, or more than
// kFlatEntries non-empty pseudo-rows, fills and walks its table several times
// (fill_long).  Such rows are everyday in the default double dam break (h is
// 2.3 particle spacings there: rows of up to 81 slots at rest density) and in
// compressed fluid; while their waves scanned those rows slot by slot, one
// dependent load each, normals / forces / XSPH of the 200,000-particle double
// dam with every force term took 172 / 366 / 175 us late in the splash and
// 91 / 178 / 106 early, against 73 / 203 / 158 and 39 / 127 / 55 this way;
// rows of 192 slots (100,000 particles at h/4): forces and XSPH 371 / 308 us
// against 167 / 143.  Near-isolated waves (WL = 0) keep the slot-by-slot
// scan: they hardly ever have such rows, and the batches would cost their
// walk registers.  Returns false, having visited nothing, in that case and
// when (need_long) no lane of the wave has a row of more than 32 slots (one
// pseudo-row per row: the row-by-row walk then does as well without the
// table).  The table is filled by flat_table.
constexpr int kForceWalkWidth = 4;  // set bits per step of the flattened force walk
constexpr int kForceLongWidth = 3;  // and where a wave's rows need more than one table
constexpr int kXsphWalkWidth = 4;   // and of the flattened XSPH walk
constexpr int kXsphRowWidth = 4;    // set bits per step of the row-by-row XSPH walk
template <int BS, int W, int WL, class Ld, class Fn>
__device__ __forceinline__ bool walk_flat(uint2 *__restrict__ tab, const RowSource &src, const uint32_t *b,
                                          const uint32_t *e, const RowMasks &mask, uint32_t nslots, uint32_t i,
                                          bool need_long, Ld &&ld, Fn &&fn) {
    const uint32_t t = threadIdx.x;
    bool batches = src.moved != nullptr;
    uint32_t cnt = 0u;
    if (__builtin_expect(!batches, 1)) {
        if (need_long) {
            bool lng = false;
#pragma unroll
            for (int r = 0; r < 9; ++r) lng = lng || e[r] - b[r] > 32u;
            if (!__ballot(lng)) return false;
        }
        // The nine masks' loads (row_mask64) are unconditional, so that all
        // are in flight together.
        uint64_t mw[9];
        bool fits = true;
#pragma unroll
        for (int r = 0; r < 9; ++r) {
            const uint32_t len = e[r] - b[r];
            mw[r] = row_mask64(mask, (size_t)r * nslots + i, len);
            fits = fits && len <= 64u;
        }
        // Entries at or past cnt are never stored and never used (the reads
        // in walk_table that may touch them are discarded).
        cnt = flat_table(mw, b, [&](uint32_t k, uint32_t m, uint32_t base) {
            tab[k * BS + t] = make_uint2(m, base);
        });
        batches = __ballot(!fits || cnt > (uint32_t)kFlatEntries) != 0ull;
    }
    if (__builtin_expect(!batches, 1)) {
        walk_table<BS, W>(tab, cnt, ld, fn);
        return true;
    }
    // Rows without a 64-bit mask, or more pseudo-rows than entries, in some
    // lane: the wave walks batch after batch of its pseudo-rows.  (WL set
    // bits per step: the force walk takes one fewer here, the fill's state
    // would otherwise cost every scene's force pass a wave per SIMD.)
    if constexpr (WL != 0) {
        uint32_t row = 0u, word = 0u;  // of the next pseudo-row (wave-uniform)
#pragma unroll 1
        while (row < 9u) {
            cnt = fill_long<BS>(tab, src, mask, nslots, i, row, word);
            walk_table<BS, WL>(tab, cnt, ld, fn);
        }
    }
    return WL != 0;
}

// Walk over the neighbour slots of lane i: with flat set and masks in use the
// flattened walk, unless it declines (walk_flat: a near-isolated wave whose
// rows need more than one table or whose particles moved far, or, in mode 2,
// a wave without rows of more than 32 slots); else walk_masks.  The
// choice is wave-uniform and does not change the result.  A callback is
// inlined into both walks (and every block size), and an implicit
// multiply-add contraction may differ between those copies: the callbacks
// write their multiply-adds as explicit fmaf, so every copy computes the
// same bits.
template <int BS, int W, int WL, int WR, bool PAIR = false, class Ld, class Fn>
__device__ __forceinline__ void walk_rows(uint2 *__restrict__ tab, const RowSource &src, const uint32_t *b,
                                          const uint32_t *e, const RowMasks &mask, bool use, int flat,
                                          uint32_t nslots, uint32_t i, Ld &&ld, Fn &&fn) {
    if (use && flat && walk_flat<BS, W, WL>(tab, src, b, e, mask, nslots, i, flat == 2, ld, fn)) return;
    walk_masks<WR, PAIR>(b, e, mask, use && !src.moved, nslots, i, ld, fn);
}

// The near-isolated particle's sum of t^3 over its pairs within h in FP64, in
// slot order (MS: its own masks, as just stored by this lane).
__device__ __forceinline__ double near_isolated_sum(const Consts &c, const uint32_t *b, const uint32_t *e,
                                                    const float4 *__restrict__ Ps, const RowMasks &MS,
                                                    uint32_t nslots, uint32_t i, float4 pi) {
    double Sd = 0.0;
    for (int r = 0; r < 9; ++r) {
        const uint32_t len = e[r] - b[r];
        const size_t at = (size_t)r * nslots + i;
        if (len <= 64u) {
            // the skin mask: a superset of the pairs within h
            uint64_t m = len <= 32u ? (uint64_t)MS.w32[at] : MS.w64[at];
            while (m) {
                const uint32_t j = b[r] + (uint32_t)__ffsll((unsigned long long)m) - 1u;
                m &= m - 1ull;
                const float4 q = at32(Ps, j);
                if (!(dist2(pi, q) <= c.h2)) continue;
                const double t = fmax(c.hh_d - dist2_d(pi, q), 0.0);
                Sd = __builtin_fma(t * t, t, Sd);
            }
        } else {
            for (uint32_t j = b[r]; j < e[r]; ++j) {
                const float4 q = at32(Ps, j);
                if (j == i || !(dist2(pi, q) <= c.h2)) continue;
                const double t = fmax(c.hh_d - dist2_d(pi, q), 0.0);
                Sd = __builtin_fma(t * t, t, Sd);
            }
        }
    }
    return Sd;
}

// What follows the density sum S (sum of m * poly6): the boundary term, the
// Tait EOS and the particle's packed neighbour data.
__device__ __forceinline__ void density_finish(const Consts &c, uint32_t i, float4 pi, float S,
                                               float4 *__restrict__ D, float4 *__restrict__ Q,
                                               float *__restrict__ Pr, uint32_t *__restrict__ flags,
                                               uint8_t *__restrict__ near) {
    // Boundary density term rho0 * (1 - boundaryDensity(d)) for d = |sdf| < h
    // (fluidphysics.cu:55-61, fluidkernel.cu:45-67), in FP64, written in t = d/h.
    const double dist = fabs(box_sdf(c, pi.x, pi.y, pi.z));
    float corrected = S;
    if (dist < c.h_d) {
        const double t = dist / c.h_d, t2 = t * t;
        const double q = 128.0 - 315.0 * t + t * t2 * (420.0 - 378.0 * t2 + t2 * t2 * (180.0 - 35.0 * t2));
        corrected = (float)((double)S + c.bd_rho0_d * q);
    }
    const float rho = (S == 0.0f) ? c.rho0 : corrected;
    const float ratio = corrected * c.inv_rho0;
    const float press = (corrected == 0.0f) ? 0.0f : c.eos_scale * (tait_pow(ratio, c.gamma, c.gamma_i) - 1.0f);
    const float cs_i = c.K * tait_pow(ratio, c.gamma_m1, c.gamma_m1_i);
    const float ir = 1.0f / rho;
    // Every pair the later passes treat as near-isolated (1/rho_j or 1/rho_i
    // above fragile_ir; rho_i + rho_j below fragile_sr, which needs one
    // density below fragile_sr / 2) has a particle that sets the flag here.
    if (ir > c.fragile_ir || rho < 0.5f * c.fragile_sr) {
        set_flag(flags, c.scene, kFragileByte, 1u);
        near[i / kNearBlock] = 1u;
    }
    D[i] = make_float4(rho, press, cs_i, ir);
    Q[i] = make_float4(pi.x, pi.y, pi.z, rho > c.eps ? ir : -1.0f);
    Pr[i] = press;
}

// 5. density + Tait EOS (computeDensity, fluidphysics.cu:8-84); also the
// neighbour masks of the substep and the packed neighbour data of the later
// passes: Q = (x, y, z, 1/density, or -1 when density <= FLT_MIN), Pr =
// pressure.  Clears the scene's far-move flag; sets its near-isolated flag
// when a particle's density is below rho0/64, so that the later passes take
// their FP64 pair-geometry walks for the scene.
template <int BS>
__global__ __launch_bounds__(BS) void k_density(const Consts *__restrict__ cs, const uint32_t *__restrict__ chunk,
                                                uint32_t nslots, const float4 *__restrict__ Ps,
                                                const float *__restrict__ soa, const uint32_t *__restrict__ start,
                                                float4 *__restrict__ D,
                                                float4 *__restrict__ Q, float *__restrict__ Pr,
                                                RowMasks MS, uint32_t *__restrict__ flags,
                                                const uint32_t *__restrict__ moves, uint8_t *__restrict__ near) {
    uint32_t slot0;
    const Consts *cp = block_scene<BS>(cs, chunk, slot0);
    if (!cp) return;
    const Consts &c = *cp;
    const float h2s = skin_h2s(c, skin_frac(scene_move_q(moves, c.scene)));
    const uint32_t i = slot0 + threadIdx.x;
    if (i == c.first) set_flag(flags, c.scene, kFarMoveByte, 0u);  // set by k_forces when the skin is exceeded
    if (i >= c.first + c.count) return;
    const uint32_t *st = start + c.cell_base;
    const uint32_t shift = c.first - st[0];
    if (i >= st[c.ncells] + shift) {  // out-of-grid bucket: never a neighbour, no masks
        D[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        return;
    }
    const float4 pi = Ps[i];
    uint32_t b[9], e[9];
    rows9(c, st, shift, pi, b, e);
    float S = 0.0f;
    // Branch-free candidate tests.  A candidate's r^2 is formed with the
    // skin radius folded in, rs = r^2 - h_s^2 (the multiply-add chain starts
    // from -h_s^2): its sign bit is the skin-mask bit, and its density term
    // is t^3 with t = (h^2 - r^2) / h^2 = c1 - rs / h^2, one multiply-add
    // whose result is clamped to [0, 1] by the instruction itself (t lies in
    // [0, 1] for every r).  A candidate outside h adds an exact zero to S;
    // the particle itself (centre row) and the slots of a partial group past
    // the end of the lane's row have their rs replaced by 1, which gives
    // t = 0 and a clear bit.
    // The first 64 slots of every lane's row are scanned four slots per step
    // (slots 0..31 into one mask word, 32..63 into another): the sorted
    // positions are also kept as x, y and z planes, so one 16-byte load per
    // plane brings four candidates.  The slot offset k is a scalar, so a
    // load's address is the lane's row offset plus a scalar (buffer
    // soffset).  Each mask word is built as m = 2m + bit (a funnel shift of
    // the sign bit in), which leaves slot k at bit n-1-k of the n slots
    // scanned into it; one bit reversal per row moves it to bit k.  A row's
    // slots past 64 follow below, 32 to a word.  Only the centre row
    // (r = 4: dz = dy = 0) holds the particle itself.
    const float nh2s = -h2s, ninv_h2 = -c.inv_h2;
    const float c1 = (c.h2 - h2s) * c.inv_h2;  // h2 - h2s is exact: h2 <= h2s <= 2 h2
    const __amdgpu_buffer_rsrc_t px = plane_buffer(soa, nslots), py = plane_buffer(soa + nslots, nslots),
                                 pz = plane_buffer(soa + 2 * (size_t)nslots, nslots);
#pragma unroll
    for (int r = 0; r < 9; ++r) {
        const uint32_t bb = b[r], len = e[r] - b[r];
        const uint32_t off = bb * (uint32_t)sizeof(float);
        const uint32_t kself = i - bb;  // < len only in the centre row
        // Slots scanned: the lane's row (at most 64 slots) rounded up to a
        // multiple of 4; slots past the row add nothing.
        // Slots with mask bits: [0, lm); whole groups of four: [0, nf).  The
        // group loop's bound is per lane (a lane leaves it when its row's
        // whole groups are done), so a group's four tests need no end-of-row
        // test; the last, partial group tests each slot against the row's
        // end.
        const uint32_t lm = len < 64u ? len : 64u, nf = lm & ~3u;
        uint32_t cur = 0u, s0 = 0u;  // the mask word being built; slots 0..31 once past them
        auto test = [&]<bool FULL>(uint32_t k, float qx, float qy, float qz) {
            const float dx = qx - pi.x, dy = qy - pi.y, dz = qz - pi.z;
            float rs = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, __builtin_fmaf(dx, dx, nh2s)));
            if (r == 4) rs = (k == kself) ? 1.0f : rs;
            if (!FULL) rs = (k < len) ? rs : 1.0f;  // past the row's end
            const float t = fminf(fmaxf(__builtin_fmaf(rs, ninv_h2, c1), 0.0f), 1.0f);
            S = __builtin_fmaf(t * t, t, S);
            cur = __builtin_amdgcn_alignbit(cur, __float_as_uint(rs), 31u);
        };
        auto group = [&]<bool FULL>(float4 X, float4 Y, float4 Z, uint32_t k0) {
            if (k0 == 32u) {  // the low word is complete
                s0 = cur;
                cur = 0u;
            }
            test.template operator()<FULL>(k0, X.x, Y.x, Z.x);
            test.template operator()<FULL>(k0 + 1u, X.y, Y.y, Z.y);
            test.template operator()<FULL>(k0 + 2u, X.z, Y.z, Z.z);
            test.template operator()<FULL>(k0 + 3u, X.w, Y.w, Z.w);
        };
        // Two whole groups per step, all six loads issued before the tests.
        uint32_t k = 0u;
        for (; k + 4u < nf; k += 8u) {
            const uint32_t so = k * (uint32_t)sizeof(float), so4 = so + 4u * (uint32_t)sizeof(float);
            const float4 AX = load4(px, off, so), AY = load4(py, off, so), AZ = load4(pz, off, so);
            const float4 BX = load4(px, off, so4), BY = load4(py, off, so4), BZ = load4(pz, off, so4);
            group.template operator()<true>(AX, AY, AZ, k);
            group.template operator()<true>(BX, BY, BZ, k + 4u);
        }
        // After the loop the slot offset differs between lanes: it goes into
        // the per-lane offset (a per-lane scalar offset would be issued once
        // per distinct value in the wave).
        if (k < nf) {
            const uint32_t vo = off + k * (uint32_t)sizeof(float);
            group.template operator()<true>(load4(px, vo, 0u), load4(py, vo, 0u), load4(pz, vo, 0u), k);
        }
        if (nf < lm) {  // the partial group
            const uint32_t vo = off + nf * (uint32_t)sizeof(float);
            group.template operator()<false>(load4(px, vo, 0u), load4(py, vo, 0u), load4(pz, vo, 0u), nf);
        }
        // The lane scanned lw = lm rounded up to 4 slots: n0 = min(lw, 32)
        // of them into the low word, lw - 32 into the high word.
        const uint32_t lw = (lm + 3u) & ~3u, n0 = lw < 32u ? lw : 32u;
        uint32_t s1 = 0u;
        if (lw > 32u)
            s1 = cur;
        else
            s0 = cur;
        const size_t at = (size_t)r * nslots + i;
        s0 = n0 ? __brev(s0) >> (32u - n0) : 0u;  // n0 == 0: nothing scanned
        if (len <= 32u)
            MS.w32[at] = s0;
        else
            MS.w64[at] = (uint64_t)(__brev(s1) >> (64u - lw)) << 32 | s0;  // lw > 32
        // A row's slots past 64, a mask word at a time (the first is kept).
        // (One group per step: two cost a wave per SIMD of every scene.)
        for (uint32_t k0 = 64u; k0 < len; k0 += 32u) {
            const uint32_t end = k0 + 32u < len ? k0 + 32u : len;
            cur = 0u;
            for (k = k0; k < end; k += 4u) {
                const uint32_t vo = off + k * (uint32_t)sizeof(float);
                group.template operator()<false>(load4(px, vo, 0u), load4(py, vo, 0u), load4(pz, vo, 0u), k);
            }
            if (k0 == 64u) MS.w32[at] = __brev(cur) >> (32u - (k - k0));
        }
    }
    if (S < c.fragile_S) {
        // Near-isolated: the same pairs again, in the same order, with the
        // pair geometry in FP64 (the FP32 h^2 - r^2 of a pair near r = h
        // carries a large relative error, and here few pairs make the sum).
        const double Sd = near_isolated_sum(c, b, e, Ps, MS, nslots, i, pi);
        S = (float)(Sd * c.mC6_d);
    } else {
        S *= c.mC6h6;  // sum of m * poly6
    }
    density_finish(c, i, pi, S, D, Q, Pr, flags, near);
}

// 6. surface normals (computeNormals, fluidphysics.cu:154-210):
// n_i = h * sum m gradPoly6(r) (x_i - x_j) / (rho_j r); r cancels against
// gradPoly6's factor r.  Neighbours with density <= FLT_MIN (Q.w < 0) or at
// r^2 <= FLT_MIN (or passed with ok = false) contribute zero.  Only the
// surface-tension force reads the normals: for a scene without it
// (lazy_normal) the pass runs only when the normals are read, over the last
// substep's data (all = 1), and gives the bits it would have given then.
// F: the scene has near-isolated particles; a pair with one takes h^2 - r^2
// in FP64.
template <bool F>
__device__ __forceinline__ float normal_weight(const Consts &c, float4 pi, float4 q, float rr, bool ok) {
    float t = fmaxf(c.h2 - rr, 0.0f);
    t = ok && rr > c.eps ? t : 0.0f;
    if constexpr (F) {
        if (t > 0.0f && q.w > c.fragile_ir)  // near-isolated neighbour: FP64 pair geometry
            t = (float)fmax(c.hh_d - dist2_d(pi, q), 0.0);
    }
    return t * t * fmaxf(q.w, 0.0f);
}

template <int BS>
__global__ __launch_bounds__(BS) void k_normals(const Consts *__restrict__ cs, const uint32_t *__restrict__ chunk,
                                                uint32_t nslots, const float4 *__restrict__ Q,
                                                const float *__restrict__ soa, const uint32_t *__restrict__ start,
                                                RowMasks M, int flat, int all, const uint32_t *__restrict__ flags,
                                                const uint32_t *__restrict__ moves,
                                                const uint8_t *__restrict__ near, float4 *__restrict__ N) {
    uint32_t slot0;
    const Consts *cp = block_scene<BS>(cs, chunk, slot0);
    if (!cp || (cp->lazy_normal && !all)) return;
    const Consts &c = *cp;
    const uint32_t i = slot0 + threadIdx.x;
    if (i >= c.first + c.count) return;
    const uint32_t *st = start + c.cell_base;
    const uint32_t shift = c.first - st[0];
    if (i >= st[c.ncells] + shift) {
        N[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        return;
    }
    const float4 pi = Q[i];
    uint32_t b[9], e[9];
    rows9(c, st, shift, pi, b, e);
    const RowSource rows{c, st, shift, Q, soa, moves, nullptr};
    float sx = 0.0f, sy = 0.0f, sz = 0.0f;
    __shared__ uint2 tab[kFlatEntries * BS];
    auto walk = [&]<bool F>() {
        walk_rows<BS, 2, F ? 0 : 2, 2>(
            tab, rows, b, e, M, c.use_masks, flat, nslots, i, [&](uint32_t j) { return at32(Q, j); },
            [&](const float4 &q, uint32_t, bool ok) {
                const float w = normal_weight<F>(c, pi, q, dist2(pi, q), ok);
                sx = __builtin_fmaf(w, pi.x - q.x, sx);
                sy = __builtin_fmaf(w, pi.y - q.y, sy);
                sz = __builtin_fmaf(w, pi.z - q.z, sz);
            });
    };
    if (__builtin_expect(flag_set(flag_word(flags, c.scene), kFragileByte), 0) && lanes(rows_near(near, b, e)))
        walk.template operator()<true>();
    else
        walk.template operator()<false>();
    N[i] = make_float4(c.hmCg6 * sx, c.hmCg6 * sy, c.hmCg6 * sz, 0.0f);
}

// ---------------------------------------------------------------------------
// 7. forces: one pair, the sums of a particle's pairs, what follows them.

struct PairSelf {
    float4 p, v, d, n;  // position, velocity, density record, normal
    float iri2;         // 1 / density^2
};

struct PairCand {
    float4 q;
    float p;
    float4 v, d, n;
};

// A candidate's loads for a walk of the scene's optional terms (V: velocity
// and density/sound speed; T: normal).  With viscosity the neighbour's
// pressure comes with its density record, D.y, instead of a load of its own.
template <bool V, bool T>
__device__ __forceinline__ PairCand pair_load(const float4 *__restrict__ Q, const float *__restrict__ Pr,
                                              const float4 *__restrict__ Vs, const float4 *__restrict__ D,
                                              const float4 *__restrict__ N, uint32_t j) {
    PairCand cd;
    cd.q = at32(Q, j);
    if constexpr (V) {
        cd.v = at32(Vs, j);
        cd.d = at32(D, j);
        cd.p = cd.d.y;
    } else {
        cd.p = at32(Pr, j);
    }
    if constexpr (T) cd.n = at32(N, j);
    return cd;
}

// One pair's contribution: coefficients of x_j - x_i = (rx, ry, rz) in the
// pressure sum (cpr; cprd in FP64 when frag) and the artificial-viscosity sum
// (cv), and the cohesion + curvature vector.
struct PairTerm {
    float rx, ry, rz, cpr, cv, tx, ty, tz;
    double cprd;
    bool frag;
};

// False (t unset) for a pair that adds nothing.
template <bool V, bool T, bool F>
__device__ __forceinline__ bool pair_term(const Consts &c, const PairSelf &me, const PairCand &cj, bool ok,
                                          PairTerm &t) {
    const float4 q = cj.q, pi = me.p;
    const float pj = cj.p;
    const float rr = dist2(pi, q);
    if (!(ok && rr <= c.h2 && rr > c.eps)) return false;
    if (!(q.w >= 0.0f)) return false;  // neighbour density <= FLT_MIN
    t.rx = q.x - pi.x;
    t.ry = q.y - pi.y;
    t.rz = q.z - pi.z;
    const float rho_i = me.d.x, p_i = me.d.y, cs_i = me.d.z, iri = me.d.w;
    const float inv_r = frsq(rr);
    const float r = rr * inv_r;
    const float irj = q.w;
    // h - r in one rounding with r's product, except in the near-isolated walk
    // (written out: left to the compiler, the choice changes with the code
    // around it).
    float hr;
    if constexpr (F) {
#pragma clang fp contract(off)
        const float d = c.h - r;
        hr = fmaxf(d, 0.0f);
    } else {
        hr = fmaxf(__builtin_fmaf(-rr, inv_r, c.h), 0.0f);
    }
    t.frag = false;
    double hrd = 0.0;
    if constexpr (F) {
        if (iri > c.fragile_ir || irj > c.fragile_ir) {
            // Near-isolated pair: h - r in FP64, r from the FP64 r^2 by one
            // Newton step from the FP32 r (relative error squared: ~1e-14).
            const double d2 = dist2_d(pi, q), r0 = (double)r;
            const double rd = __builtin_fma(__builtin_fma(-r0, r0, d2), (double)(0.5f * inv_r), r0);
            hrd = fmax(c.h_d - rd, 0.0);
            hr = (float)hrd;
            t.frag = true;
        }
    }
    const float cm = c.mCgs * hr * hr * inv_r;  // m gradSpiky(r) / r
    if (t.frag) {
        // and its pressure term in FP64: 1/rho^2 of a density near FLT_MIN
        // overflows FP32 (an infinite force).
        const double cmd = (double)c.mCgs * hrd * hrd * (double)inv_r;
        const double midd =
            __builtin_fma((double)pj, (double)iri * (double)iri, (double)p_i * ((double)irj * (double)irj));
        t.cprd = cmd * midd;
    } else {
        const float mid = __builtin_fmaf(pj, me.iri2, p_i * (irj * irj));
        t.cpr = cm * mid;
    }
    if constexpr (V) {
        // Approaching pairs only (ux < 0); the others add exact zeros.
        const float4 vi = me.v, vj = cj.v, dj = cj.d;
        const float ux =
            -__builtin_fmaf(vi.z - vj.z, t.rz, __builtin_fmaf(vi.y - vj.y, t.ry, (vi.x - vj.x) * t.rx));
        const float mu = c.h * ux * frcp(rr + c.visc_eps);
        const float Pi = -c.nu * (cs_i + dj.z) * mu * frcp(rho_i + dj.x);
        t.cv = keep(cm * Pi, lanes(ux < 0.0f));
    }
    if constexpr (T) {
        const float4 ni = me.n, nj = cj.n;
        const float hr3r3 = hr * hr * hr * r * r * r;
        const float coh = (r > c.halfh) ? hr3r3 : 2.0f * hr3r3 - c.coh_off;
        const float ch = -c.m2 * coh * inv_r;
        t.tx = __builtin_fmaf(ch, t.rx, -c.sigma_m * (ni.x - nj.x));
        t.ty = __builtin_fmaf(ch, t.ry, -c.sigma_m * (ni.y - nj.y));
        t.tz = __builtin_fmaf(ch, t.rz, -c.sigma_m * (ni.z - nj.z));
    }
    return true;
}

struct PairSums {
    float Px = 0.f, Py = 0.f, Pz = 0.f;      // pressure sum
    double Pdx = 0.0, Pdy = 0.0, Pdz = 0.0;  // its near-isolated pairs, in FP64
    float Qx = 0.f, Qy = 0.f, Qz = 0.f;      // artificial-viscosity part of the viscosity sum
    float Tx = 0.f, Ty = 0.f, Tz = 0.f;      // cohesion + curvature sum
    template <bool V, bool T, bool F>
    __device__ __forceinline__ void add(const PairTerm &t) {
        if (t.frag) {
            Pdx = __builtin_fma(t.cprd, (double)t.rx, Pdx);
            Pdy = __builtin_fma(t.cprd, (double)t.ry, Pdy);
            Pdz = __builtin_fma(t.cprd, (double)t.rz, Pdz);
        } else {
            Px = __builtin_fmaf(t.cpr, t.rx, Px);
            Py = __builtin_fmaf(t.cpr, t.ry, Py);
            Pz = __builtin_fmaf(t.cpr, t.rz, Pz);
        }
        if constexpr (V) {
            Qx = __builtin_fmaf(t.cv, t.rx, Qx);
            Qy = __builtin_fmaf(t.cv, t.ry, Qy);
            Qz = __builtin_fmaf(t.cv, t.rz, Qz);
        }
        if constexpr (T) {
            Tx += t.tx;
            Ty += t.ty;
            Tz += t.tz;
        }
    }
};

// A particle's summed forces; eP: pressure sum of near-isolated pairs (FP64).
struct Forces {
    float3 P = {0.f, 0.f, 0.f}, V = {0.f, 0.f, 0.f}, T = {0.f, 0.f, 0.f}, A = {0.f, 0.f, 0.f};
    double eP[3] = {0.0, 0.0, 0.0};
};

__device__ __forceinline__ void total_forces(const Consts &c, float4 pi, float4 di, const PairSums &s, Forces &f) {
    f.P = make_float3(s.Px, s.Py, s.Pz);
    f.eP[0] = s.Pdx;
    f.eP[1] = s.Pdy;
    f.eP[2] = s.Pdz;
    f.V = make_float3(c.nu * (s.Px + s.Qx), c.nu * (s.Py + s.Qy), c.nu * (s.Pz + s.Qz));
    // 2 rho0 / (rho_i + rho_i) applied once to the summed tension terms.
    const float ts = c.sigma * c.rho0 * di.w;
    f.T = make_float3(ts * s.Tx, ts * s.Ty, ts * s.Tz);
    if (c.has_adhesion) {
        // Adhesion toward the walls (fluidphysics.cu:330-350), FP64.
        const double z = -fmin(box_sdf(c, pi.x, pi.y, pi.z), 0.0) * c.quarter_inv_psize;
        if (z < 1.0) {
            double nbv[3];
            box_normal(c, pi.x, pi.y, pi.z, nbv);
            const double oz = 1.0 - z;
            const double k = c.alpha_inv_rho0 * (double)di.x / (oz * oz * oz);
            f.A = make_float3((float)(k * nbv[0]), (float)(k * nbv[1]), (float)(k * nbv[2]));
        }
    }
}

// Leapfrog integration and boundary clamp of the particle in slot i (src: its
// state slot), the outputs of the force pass and the far-move flag.
__device__ __forceinline__ void integrate(const Consts &c, uint32_t i, uint32_t src, float4 pi, float4 vi, float rho,
                                          const Forces &f, const float4 *__restrict__ A,
                                          const float4 *__restrict__ Lw, float4 *__restrict__ Pout,
                                          float4 *__restrict__ Vout, float4 *__restrict__ Aout,
                                          float4 *__restrict__ Lout, float4 *__restrict__ Fdbg,
                                          uint32_t *__restrict__ flags, uint32_t move_q) {
    // The viscosity force carries the pressure sum too (nu * (P + Pi)).
    const float3 fP = f.P, fV = f.V, fT = f.T, fA = f.A;
    const double *eP = f.eP;
    const double eV[3] = {(double)c.nu * eP[0], (double)c.nu * eP[1], (double)c.nu * eP[2]};
    if (Fdbg) {
        Fdbg[4 * (size_t)i + 0] = make_float4((float)((double)fP.x + eP[0]), (float)((double)fP.y + eP[1]),
                                              (float)((double)fP.z + eP[2]), 0.f);
        Fdbg[4 * (size_t)i + 1] = make_float4((float)((double)fV.x + eV[0]), (float)((double)fV.y + eV[1]),
                                              (float)((double)fV.z + eV[2]), 0.f);
        Fdbg[4 * (size_t)i + 2] = make_float4(fT.x, fT.y, fT.z, 0.f);
        Fdbg[4 * (size_t)i + 3] = make_float4(fA.x, fA.y, fA.z, 0.f);
    }
    // Leapfrog (fluidintegrator.cu:36-69), per particle in FP64 on the FP32
    // inputs: a' = F m + g (clamped to acc_limit); x += v dt + a dt^2/2 on the
    // double-float position; v += (a + a') dt/2 (clamped to vel_limit); then
    // the boundary projection and reflection.
    const double Fx = ((double)fP.x + eP[0]) + (double)fT.x + (double)fA.x + ((double)fV.x + eV[0]);
    const double Fy = ((double)fP.y + eP[1]) + (double)fT.y + (double)fA.y + ((double)fV.y + eV[1]);
    const double Fz = ((double)fP.z + eP[2]) + (double)fT.z + (double)fA.z + ((double)fV.z + eV[2]);
    double ax = Fx * c.m + c.g[0], ay = Fy * c.m + c.g[1], az = Fz * c.m + c.g[2];
    double s2 = ax * ax + ay * ay + az * az;
    if (s2 > c.alim2) {
        const double k = c.alim / sqrt(s2);
        ax *= k;
        ay *= k;
        az *= k;
    }
    const float4 ai = A[src], li = Lw[src];
    double x = ((double)pi.x + (double)li.x) + ((double)vi.x * c.dt + 0.5 * (double)ai.x * c.dtdt);
    double y = ((double)pi.y + (double)li.y) + ((double)vi.y * c.dt + 0.5 * (double)ai.y * c.dtdt);
    double z = ((double)pi.z + (double)li.z) + ((double)vi.z * c.dt + 0.5 * (double)ai.z * c.dtdt);
    double vx = (double)vi.x + 0.5 * ((double)ai.x + ax) * c.dt;
    double vy = (double)vi.y + 0.5 * ((double)ai.y + ay) * c.dt;
    double vz = (double)vi.z + 0.5 * ((double)ai.z + az) * c.dt;
    s2 = vx * vx + vy * vy + vz * vz;
    if (s2 > c.vlim2) {
        const double k = c.vlim / sqrt(s2);
        vx *= k;
        vy *= k;
        vz *= k;
    }
    // boundaryCheckSDF (fluidintegrator.cu:11-26).
    const double dd = box_sdf(c, x, y, z);
    if (dd > -c.psize) {
        double nbv[3];
        box_normal(c, x, y, z, nbv);
        const double push = dd + c.psize;
        const double vn = c.vdamp1 * (nbv[0] * vx + nbv[1] * vy + nbv[2] * vz);
        x -= push * nbv[0];
        y -= push * nbv[1];
        z -= push * nbv[2];
        vx -= vn * nbv[0];
        vy -= vn * nbv[1];
        vz -= vn * nbv[2];
    }
    const float hx = (float)x, hy = (float)y, hz = (float)z;
    Pout[i] = make_float4(hx, hy, hz, pi.w);
    Lout[i] = make_float4((float)(x - (double)hx), (float)(y - (double)hy), (float)(z - (double)hz), 0.0f);
    Vout[i] = make_float4((float)vx, (float)vy, (float)vz, rho);
    Aout[i] = make_float4((float)ax, (float)ay, (float)az, 0.0f);
    // Move of the FP32 positions the pair predicates see (the differences
    // are exact in FP64).  Every writer stores the same value; NaN counts
    // as too far.
    const double move_limit = skin_move_limit(c, skin_frac(move_q));
    const double ex = (double)hx - (double)pi.x, ey = (double)hy - (double)pi.y, ez = (double)hz - (double)pi.z;
    if (!(ex * ex + ey * ey + ez * ez <= move_limit * move_limit)) set_flag(flags, c.scene, kFarMoveByte, 1u);
}

// The force pass (computeAllForces, fluidphysics.cu:215-352) fused with the
// leapfrog integrator and boundary clamp (LeapfrogIntegratorOperator,
// fluidintegrator.cu:11-70).  Out-of-grid particles get zero forces and are
// still integrated.  Fdbg (may be null) receives the four force components.
// The pre-XSPH velocity carries the particle's density in w for the XSPH
// pass, which reads the integrated positions from Pout.  Sets the scene's
// far-move flag when a particle moved farther than the XSPH skin masks allow.
template <int BS>
__global__ __launch_bounds__(BS) void k_forces(const Consts *__restrict__ cs, const uint32_t *__restrict__ chunk,
                                               uint32_t nslots, const float4 *__restrict__ Ps,
                                               const float4 *__restrict__ Q, const float *__restrict__ Pr,
                                               const float4 *__restrict__ Vs, const float4 *__restrict__ A,
                                               const float4 *__restrict__ Lw, const uint32_t *__restrict__ order,
                                               const float4 *__restrict__ D,
                                               const float4 *__restrict__ N, const float *__restrict__ soa,
                                               const uint32_t *__restrict__ start,
                                               RowMasks M, int flat, float4 *__restrict__ Pout,
                                               float4 *__restrict__ Vout, float4 *__restrict__ Aout,
                                               float4 *__restrict__ Lout,
                                               float4 *__restrict__ Fdbg, uint32_t *__restrict__ flags,
                                               const uint32_t *__restrict__ moves, const uint8_t *__restrict__ near) {
    uint32_t slot0;
    const Consts *cp = block_scene<BS>(cs, chunk, slot0);
    if (!cp) return;
    const Consts &c = *cp;
    const uint32_t move_q = scene_move_q(moves, c.scene);
    const uint32_t i = slot0 + threadIdx.x;
    if (i >= c.first + c.count) return;
    const uint32_t *st = start + c.cell_base;
    const uint32_t shift = c.first - st[0];
    const uint32_t sw = flag_word(flags, c.scene);
    const uint32_t src = order[i];  // the particle's slot in the state arrays (A, Lw)
    const float4 pi = Ps[i], vi = Vs[i];
    const float4 di = D[i];
    Forces f;
    if (i < st[c.ncells] + shift) {
        const PairSelf me{pi, vi, di, c.has_tension ? N[i] : make_float4(0.f, 0.f, 0.f, 0.f), di.w * di.w};
        PairSums sum;
        uint32_t b[9], e[9];
        rows9(c, st, shift, pi, b, e);
        const RowSource rows{c, st, shift, Ps, soa, moves, nullptr};
        // One walk per combination of the scene's optional terms, so that a
        // candidate's loads (V: velocity and density/sound speed; T: normal)
        // are all issued with its position before any arithmetic.  F: the
        // scene has near-isolated particles, and a pair with one takes its
        // h - r in FP64 (a separate walk, so that the other scenes' walks
        // carry none of its registers' cost).
        __shared__ uint2 tab[kFlatEntries * BS];
        auto walk = [&]<bool V, bool T, bool F>() {
            // (with viscosity the neighbour's pressure comes with its
            // density record, D.y, instead of a load of its own)
            using Cand = PairCand;
            // (two set bits per step in the near-isolated walk: its FP64
            // terms would otherwise cost every scene's walk registers)
            walk_rows<BS, F ? 2 : kForceWalkWidth, F ? 0 : kForceLongWidth, 2>(
                tab, rows, b, e, M, c.use_masks, flat, nslots, i,
                [&](uint32_t j) { return pair_load<V, T>(Q, Pr, Vs, D, N, j); },
                [&](const Cand &cj, uint32_t, bool ok) {
                    PairTerm t;
                    if (!pair_term<V, T, F>(c, me, cj, ok, t)) return;
                    sum.template add<V, T, F>(t);
                });
        };
        const bool tension = c.has_tension != 0;
        auto terms = [&]<bool F>() {
            if (c.has_visc) {
                if (tension)
                    walk.template operator()<true, true, F>();
                else
                    walk.template operator()<true, false, F>();
            } else {
                if (tension)
                    walk.template operator()<false, true, F>();
                else
                    walk.template operator()<false, false, F>();
            }
        };
        if (flag_set(sw, kFragileByte) && lanes(rows_near(near, b, e)))
            terms.template operator()<true>();
        else
            terms.template operator()<false>();
        total_forces(c, pi, di, sum, f);
    }
    integrate(c, i, src, pi, vi, di.x, f, A, Lw, Pout, Vout, Aout, Lout, Fdbg, flags, move_q);
}

// A neighbour's integrated position and pre-XSPH velocity (density in w), and
// its XSPH weight.  A candidate outside h (or with rho_i + rho_j <= FLT_MIN,
// or passed with ok = false) weighs an exact zero, branch-free.
struct XsphCand {
    float4 x, v;
};
template <bool F>
__device__ __forceinline__ float xsph_weight(const Consts &c, float4 xi, float rho_i, const XsphCand &cj, uint64_t ok,
                                             const float4 *__restrict__ Lw, uint32_t i, uint32_t j) {
    const float4 q = cj.x;
    const float rr = dist2(xi, q);
    const float sr = rho_i + cj.v.w;
    const uint64_t in = lanes(rr <= c.h2) & lanes(sr > c.eps) & ok;
    float t = keep(c.h2 - rr, in);
    if constexpr (F) {
        if (sr < c.fragile_sr) {
            // Near-isolated pair: h^2 - r^2 in FP64 on the double-float
            // integrated positions (high word in X, low word in Lw).
            const float4 li = Lw[i], lj = at32(Lw, j);
            const double dx = ((double)q.x + (double)lj.x) - ((double)xi.x + (double)li.x);
            const double dy = ((double)q.y + (double)lj.y) - ((double)xi.y + (double)li.y);
            const double dz = ((double)q.z + (double)lj.z) - ((double)xi.z + (double)li.z);
            t = keep((float)fmax(c.hh_d - __builtin_fma(dz, dz, __builtin_fma(dy, dy, dx * dx)), 0.0), in);
        }
    }
    return keep(t * t * t * frcp(sr), in);
}

// 8. XSPH velocity smoothing (correctVelocityXSPH, fluidphysics.cu:355-409):
// the stencil of the pre-integration cell (Ps), integrated positions (Pn),
// and the pre-XSPH velocity of every neighbour, with its density in w (Vh;
// Jacobi update into Vout).  The skin
// masks hold every stencil slot within the skin radius h_s before the move;
// a pair within h after the move was within h + 2 max|dx| before it, so the
// masks are complete while no particle moved farther than move_limit
// (h + 2 move_limit <= h_s with FP32 margins); k_forces flags a farther move
// in the scene's far-move flag, and then every row's slots are tested again
// on the integrated positions (moved_word; the default driver's splash, 87
// against 106 us for 10,000 particles scanned).  Registers
// are capped for five waves per SIMD (four for 512-thread workgroups).
template <int BS>
__global__ __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(BS >= 512 ? 4 : 5))) void k_xsph(
                                             const Consts *__restrict__ cs, const uint32_t *__restrict__ chunk,
                                             uint32_t nslots, const float4 *__restrict__ Ps,
                                             const float4 *__restrict__ Pn, const float4 *__restrict__ Vh,
                                             const float4 *__restrict__ Lw, const float *__restrict__ soa,
                                             const uint32_t *__restrict__ start,
                                             RowMasks MS, int flat, const uint32_t *__restrict__ flags,
                                             const uint32_t *__restrict__ moves, const uint8_t *__restrict__ near,
                                             float4 *__restrict__ Vout) {
    uint32_t slot0;
    const Consts *cp = block_scene<BS>(cs, chunk, slot0);
    if (!cp) return;
    const Consts &c = *cp;
    const uint32_t i = slot0 + threadIdx.x;
    if (i >= c.first + c.count) return;
    const uint32_t *st = start + c.cell_base;
    const uint32_t shift = c.first - st[0];
    const float4 vi = Vh[i];
    if (i >= st[c.ncells] + shift) {
        Vout[i] = make_float4(vi.x, vi.y, vi.z, 0.0f);
        return;
    }
    const uint32_t fl = flag_word(flags, c.scene);
    const float4 xi = Pn[i];
    const float rho_i = vi.w;
    uint32_t b[9], e[9];
    // a particle moved farther than the masks allow: test the moved positions
    const RowSource rows{c, st, shift, Ps, soa, moves, flag_set(fl, kFarMoveByte) ? Pn : nullptr};
    rows9(c, st, shift, Ps[i], b, e);
    float sx = 0.f, sy = 0.f, sz = 0.f;
    // Both loads of a candidate are issued together.  F: the scene has
    // near-isolated particles (a separate walk, so that the other scenes'
    // walks carry none of its registers' cost).
    using Cand = XsphCand;
    __shared__ uint2 tab[kFlatEntries * BS];
    auto walk = [&]<bool F>() {
        walk_rows<BS, F ? 2 : kXsphWalkWidth, F ? 0 : kXsphWalkWidth, F ? 2 : kXsphRowWidth, !F>(
            tab, rows, b, e, MS, c.use_masks, flat, nslots, i,
            [&](uint32_t j) { return Cand{at32(Pn, j), at32(Vh, j)}; },
            [&](const Cand &cj, uint32_t j, auto ok) {
                const float4 vj = cj.v;
                const float w = xsph_weight<F>(c, xi, rho_i, cj, lane_mask(ok), Lw, i, j);
                sx = __builtin_fmaf(w, vj.x - vi.x, sx);
                sy = __builtin_fmaf(w, vj.y - vi.y, sy);
                sz = __builtin_fmaf(w, vj.z - vi.z, sz);
            });
    };
    if (__builtin_expect(flag_set(fl, kFragileByte), 0) && lanes(rows_near(near, b, e)))
        walk.template operator()<true>();
    else
        walk.template operator()<false>();
    Vout[i] = make_float4(vi.x + c.xsph_k * sx, vi.y + c.xsph_k * sy, vi.z + c.xsph_k * sz, 0.0f);
}

// ---------------------------------------------------------------------------
// Four lanes per particle.  Below about two waves per SIMD the neighbour
// passes are bound by each wave's serial chain (row after row, step after
// step), not by any pipe; there a particle's candidates are spread over four
// lanes (density / forces / XSPH of the 32,768-particle dam break in its
// splash: 20.2 / 19.2 / 15.7 us with one lane, 13.5 / 13.0 / 9.8 with four;
// density / normals / forces / XSPH of the driver's default scene: 28 / 41 /
// 72 / 90 and 14 / 15 / 25 / 30; quad_share says which launches).  Sums stay
// in slot order, so every bit is that of the one-lane kernels: each lane
// computes the terms of its candidates, then the quad's lanes take turns
// adding theirs to the running sums, the result of each turn broadcast to the
// quad (DPP).
constexpr int kQuadBlock = 256;                 // 64 particles per workgroup
constexpr uint32_t kQuadParts = kQuadBlock / 4;
constexpr uint32_t kQuadList = 128;             // neighbour slots of a particle listed at a time
constexpr uint32_t kQuadStride = kQuadList + 4;  // (lists of a wave's particles start in different banks)

template <int R>
__device__ __forceinline__ uint32_t quad_get(uint32_t v) {  // lane R's value
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, R * 0x55, 0xF, 0xF, true);
}
template <int R>
__device__ __forceinline__ float quad_get(float v) {
    return __uint_as_float(quad_get<R>(__float_as_uint(v)));
}
template <int R>
__device__ __forceinline__ double quad_get(double v) {
    const uint64_t u = (uint64_t)__double_as_longlong(v);
    return __longlong_as_double((long long)((uint64_t)quad_get<R>((uint32_t)(u >> 32)) << 32 |
                                            quad_get<R>((uint32_t)u)));
}
__device__ __forceinline__ uint32_t quad_or(uint32_t v) {
    v |= (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, true);  // lanes 1 0 3 2
    v |= (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, true);  // lanes 2 3 0 1
    return v;
}
// Orders a wave's LDS accesses of different lanes (a quad is inside one wave).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// First slots and lengths of the rows q, q + 4 and (lane 0) 8 of lane q.
struct QuadRows {
    uint32_t s[3], len[3];
};
__device__ __forceinline__ QuadRows quad_rows(const Consts &c, const uint32_t *__restrict__ start, uint32_t shift,
                                              float4 pc, uint32_t q) {
    QuadRows w;
#pragma unroll
    for (uint32_t k = 0; k < 3u; ++k) {
        const uint32_t r = q + 4u * k;
        const uint2 x = row_span(c, start, shift, pc, r < 9u ? r : 4u);
        w.s[k] = x.x;
        w.len[k] = r < 9u ? x.y - x.x : 0u;
    }
    return w;
}
__device__ __forceinline__ bool quad_near(const uint8_t *__restrict__ near, const QuadRows &w) {
    uint32_t any = 0u;
#pragma unroll
    for (int k = 0; k < 3; ++k)
        if (w.len[k])
            for (uint32_t a = w.s[k] / kNearBlock; a <= (w.s[k] + w.len[k] - 1u) / kNearBlock; ++a) any |= near[a];
    return any != 0u;
}

// Eight candidates [s, s + 8) of a lane (n of them in its row): those within
// the skin radius (slots' planes, as skin_word) or, with src.moved, within h
// of the integrated position pc (as moved_word); every one when !use.
__device__ __forceinline__ uint32_t skin_byte(const RowSource &src, uint32_t nslots, bool use, float4 pc, float h2s,
                                              uint32_t s, uint32_t n, uint32_t i) {
    uint32_t m = 0xFFu;
    if (use && src.moved) {
        float4 x[8];
#pragma unroll
        for (uint32_t k = 0; k < 8u; ++k) x[k] = at32(src.moved, k < n ? s + k : i);
        m = 0u;
#pragma unroll
        for (uint32_t k = 0; k < 8u; ++k) m |= dist2(pc, x[k]) <= src.c.h2 ? 1u << k : 0u;
    } else if (use) {
        const __amdgpu_buffer_rsrc_t px = plane_buffer(src.soa, nslots), py = plane_buffer(src.soa + nslots, nslots),
                                     pz = plane_buffer(src.soa + 2 * (size_t)nslots, nslots);
        const uint32_t vo = s * (uint32_t)sizeof(float);
        const float4 X[2] = {load4(px, vo, 0u), load4(px, vo, 16u)}, Y[2] = {load4(py, vo, 0u), load4(py, vo, 16u)},
                     Z[2] = {load4(pz, vo, 0u), load4(pz, vo, 16u)};
        m = 0u;
#pragma unroll
        for (uint32_t k = 0; k < 8u; ++k) {
            const float dx = (&X[k / 4].x)[k % 4] - pc.x, dy = (&Y[k / 4].x)[k % 4] - pc.y,
                        dz = (&Z[k / 4].x)[k % 4] - pc.z;
            const float rs = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, __builtin_fmaf(dx, dx, -h2s)));
            m |= (__float_as_uint(rs) >> 31) << k;
        }
    }
    if (n < 8u) m &= (1u << n) - 1u;
    if (i - s < 8u) m &= ~(1u << (i - s));  // the particle itself is no candidate
    return m;
}

// Lists the particle's candidates in slot order and walks the list sixteen at
// a time: lane q takes entries 4q .. 4q + 3.  Where the stored mask words are
// all a wave's particles have (rows of at most 96 slots), each lane lists the
// set bits of its own rows, in parts of kQuadList entries; else the quad goes
// through the rows together, eight slots of every mask word per lane (words
// not stored are tested, every slot taken when !use), and walks when another
// word may not fit.  term(candidate, slot, ok) gives a candidate's term (zero
// when !ok or it adds nothing), sums.add(term) adds it, sums.get<R>() is lane
// R's.
template <class Sums, class Ld, class Fn>
__device__ __forceinline__ void walk_quad(uint32_t *__restrict__ list, const RowSource &src, const QuadRows &w,
                                          const RowMasks &mask, bool use, uint32_t nslots, uint32_t i, uint32_t q,
                                          Sums &sums, Ld &&ld, Fn &&term) {
    uint64_t w01[3];
    uint32_t w2[3], at[3], total = 0u;
    bool tested = false;  // some word is not stored
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const uint32_t r = q + 4u * (uint32_t)k;
        const size_t m = (size_t)(r < 9u ? r : 4u) * nslots + i;
        w01[k] = w.len[k] ? row_mask64(mask, m, w.len[k]) : 0ull;
        w2[k] = w.len[k] > 64u ? mask.w32[m] : 0u;
        tested = tested || w.len[k] > 96u;
    }
    const bool words = __ballot(tested || src.moved || !use) == 0ull;
#pragma unroll
    for (int k = 0; k < 3; ++k) {  // each row's place in the list: rows 0..3 (one per lane), then 4..7, then 8
        const uint32_t cnt = (uint32_t)__popcll(w01[k]) + (uint32_t)__popc(w2[k]);
        const uint32_t c0 = quad_get<0>(cnt), c1 = quad_get<1>(cnt), c2 = quad_get<2>(cnt), c3 = quad_get<3>(cnt);
        at[k] = total + (q > 0u ? c0 : 0u) + (q > 1u ? c1 : 0u) + (q > 2u ? c2 : 0u);
        total += c0 + c1 + c2 + c3;
    }
    const auto put = [&](uint32_t &idx, uint32_t s, uint32_t m) {
        while (m) {
            if (idx < kQuadList) list[idx] = s + (uint32_t)__builtin_ctz(m);
            m &= m - 1u;
            ++idx;
        }
    };
    uint32_t base = 0u;             // words: entries walked so far
    uint32_t row = 0u, word = 0u;   // else the next word (wave-uniform)
    bool more = true;
#pragma unroll 1
    while (more) {
        uint32_t n = 0u;  // entries listed
        wave_lds_sync();  // the last part's entries have been read
        if (words) {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                uint32_t idx = at[k] - base;  // (entries of earlier parts wrap round past kQuadList)
                put(idx, w.s[k], (uint32_t)w01[k]);
                put(idx, w.s[k] + 32u, (uint32_t)(w01[k] >> 32));
                put(idx, w.s[k] + 64u, w2[k]);
            }
            n = base < total ? total - base : 0u;
            n = n < kQuadList ? n : kQuadList;
            base += kQuadList;
            more = __ballot(base < total) != 0ull;
        } else {
            const float4 pc = at32(src.pos, i);
            const float4 xt = src.moved ? at32(src.moved, i) : pc;
            const float h2s = skin_h2s(src.c, skin_frac(scene_move_q(src.moves, src.c.scene)));
            uint2 cur = row_span(src.c, src.st, src.shift, pc, row);
            bool full = false;
#pragma unroll 1
            while (row < 9u && !full) {
                const uint2 nxt = row_span(src.c, src.st, src.shift, pc, row < 8u ? row + 1u : 8u);
                const uint32_t len = cur.y - cur.x;
#pragma unroll 1
                for (; __ballot(32u * word < len); ++word) {
                    full = __ballot(n + 32u > kQuadList) != 0ull;
                    if (full) break;
                    const uint32_t o = 32u * word + 8u * q;
                    uint32_t m = 0u;
                    if (o < len) {
                        if (use && !src.moved && word < 3u) {
                            const size_t t = (size_t)row * nslots + i;
                            m = (word < 2u ? (uint32_t)(row_mask64(mask, t, len) >> (32u * word)) : mask.w32[t]) >>
                                    (8u * q) & 0xFFu;
                        } else {
                            m = skin_byte(src, nslots, use, xt, h2s, cur.x + o, len - o, i);
                        }
                    }
                    const uint32_t cnt = (uint32_t)__popc(m);
                    const uint32_t c0 = quad_get<0>(cnt), c1 = quad_get<1>(cnt), c2 = quad_get<2>(cnt),
                                   c3 = quad_get<3>(cnt);
                    uint32_t idx = n + (q > 0u ? c0 : 0u) + (q > 1u ? c1 : 0u) + (q > 2u ? c2 : 0u);
                    put(idx, cur.x + o, m);
                    n += c0 + c1 + c2 + c3;
                }
                if (!full) {
                    word = 0u;
                    ++row;
                    cur = nxt;
                }
            }
            more = row < 9u;
        }
        wave_lds_sync();
#pragma unroll 1
        for (uint32_t k0 = 0u; k0 < n; k0 += 16u) {
            const uint32_t mine = k0 + 4u * q;
            const uint4 e = *reinterpret_cast<const uint4 *>(list + mine);
            const uint32_t es[4] = {e.x, e.y, e.z, e.w};
            uint32_t j[4];
            bool ok[4];
            decltype(ld(0u)) a[4];
#pragma unroll
            for (uint32_t k = 0; k < 4u; ++k) {
                ok[k] = mine + k < n;
                j[k] = ok[k] ? es[k] : i;
                a[k] = ld(j[k]);
            }
            decltype(term(a[0], 0u, true)) t[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) t[k] = term(a[k], j[k], ok[k]);
            const auto turn = [&]<int R>() {
                Sums mine4 = sums;
#pragma unroll
                for (int k = 0; k < 4; ++k) mine4.add(t[k]);
                sums = mine4.template get<R>();
            };
            turn.template operator()<0>();
            turn.template operator()<1>();
            turn.template operator()<2>();
            turn.template operator()<3>();
        }
    }
}

// Scene, slot and lane of a four-lane kernel's thread; false: nothing to do.
__device__ __forceinline__ const Consts *quad_scene(const Consts *__restrict__ cs, const uint32_t *__restrict__ chunk,
                                                    uint32_t &i, uint32_t &q) {
    uint32_t slot0;
    const Consts *cp = block_scene<kQuadParts>(cs, chunk, slot0);
    i = slot0 + (threadIdx.x >> 2);
    q = threadIdx.x & 3u;
    return cp;
}

// k_density for few particles.  The quad scans a row sixteen slots at a time,
// four per lane, and the next row's first 32 slots are loaded before a row is
// tested.
__global__ __launch_bounds__(kQuadBlock) void k_density_quad(
    const Consts *__restrict__ cs, const uint32_t *__restrict__ chunk, uint32_t nslots, const float4 *__restrict__ Ps,
    const float *__restrict__ soa, const uint32_t *__restrict__ start, float4 *__restrict__ D, float4 *__restrict__ Q,
    float *__restrict__ Pr, RowMasks MS, uint32_t *__restrict__ flags, const uint32_t *__restrict__ moves,
    uint8_t *__restrict__ near) {
    uint32_t i, q;
    const Consts *cp = quad_scene(cs, chunk, i, q);
    if (!cp) return;
    const Consts &c = *cp;
    const float h2s = skin_h2s(c, skin_frac(scene_move_q(moves, c.scene)));
    if (i == c.first && q == 0u) set_flag(flags, c.scene, kFarMoveByte, 0u);
    if (i >= c.first + c.count) return;
    const uint32_t *st = start + c.cell_base;
    const uint32_t shift = c.first - st[0];
    if (i >= st[c.ncells] + shift) {
        if (q == 0u) D[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        return;
    }
    const float4 pi = Ps[i];
    uint32_t b[9], e[9];
    rows9(c, st, shift, pi, b, e);
    const float nh2s = -h2s, ninv_h2 = -c.inv_h2;
    const float c1 = (c.h2 - h2s) * c.inv_h2;
    const __amdgpu_buffer_rsrc_t px = plane_buffer(soa, nslots), py = plane_buffer(soa + nslots, nslots),
                                 pz = plane_buffer(soa + 2 * (size_t)nslots, nslots);
    struct Group {
        float4 X, Y, Z;
    };
    const auto load = [&](uint32_t s) {  // slots [s, s + 4) of the planes
        const uint32_t vo = s * (uint32_t)sizeof(float);
        return Group{load4(px, vo, 0u), load4(py, vo, 0u), load4(pz, vo, 0u)};
    };
    float S = 0.0f;
    // Slots [k0, k0 + 4) of row r, this lane's; returns the sixteen mask bits
    // of the quad's slots.
    const auto scan = [&](const Group &g, int r, uint32_t c0, uint32_t len, uint32_t kself) -> uint32_t {
        const float X[4] = {g.X.x, g.X.y, g.X.z, g.X.w}, Y[4] = {g.Y.x, g.Y.y, g.Y.z, g.Y.w},
                    Z[4] = {g.Z.x, g.Z.y, g.Z.z, g.Z.w};
        const uint32_t k0 = c0 + 4u * q;
        uint32_t bits = 0u;
        float t[4], tt[4];
#pragma unroll
        for (uint32_t k = 0; k < 4u; ++k) {
            const float dx = X[k] - pi.x, dy = Y[k] - pi.y, dz = Z[k] - pi.z;
            float rs = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, __builtin_fmaf(dx, dx, nh2s)));
            if (r == 4) rs = (k0 + k == kself) ? 1.0f : rs;
            rs = (k0 + k < len) ? rs : 1.0f;
            t[k] = fminf(fmaxf(__builtin_fmaf(rs, ninv_h2, c1), 0.0f), 1.0f);
            tt[k] = t[k] * t[k];
            bits |= (__float_as_uint(rs) >> 31) << k;
        }
        const auto turn = [&]<int R>() {
            float mine = S;
#pragma unroll
            for (int k = 0; k < 4; ++k) mine = __builtin_fmaf(tt[k], t[k], mine);
            S = quad_get<R>(mine);
        };
        turn.template operator()<0>();
        turn.template operator()<1>();
        turn.template operator()<2>();
        turn.template operator()<3>();
        return quad_or(bits << (4u * q));
    };
    Group g0 = load(b[0] + 4u * q), g1 = load(b[0] + 16u + 4u * q);
#pragma unroll
    for (int r = 0; r < 9; ++r) {
        const uint32_t len = e[r] - b[r], kself = i - b[r];
        const Group a0 = g0, a1 = g1;
        if (r < 8) {
            g0 = load(b[r + 1] + 4u * q);
            g1 = load(b[r + 1] + 16u + 4u * q);
        }
        uint32_t s0 = 0u, s1 = 0u, s2 = 0u;
        if (len > 0u) s0 = scan(a0, r, 0u, len, kself);
        if (len > 16u) s0 |= scan(a1, r, 16u, len, kself) << 16;
#pragma unroll 1
        for (uint32_t c0 = 32u; c0 < len; c0 += 16u) {
            const uint32_t m = scan(load(b[r] + c0 + 4u * q), r, c0, len, kself) << (c0 & 16u);
            if (c0 < 64u)
                s1 |= m;
            else if (c0 < 96u)
                s2 |= m;
        }
        if (q == 0u) {
            const size_t at = (size_t)r * nslots + i;
            if (len <= 32u)
                MS.w32[at] = s0;
            else
                MS.w64[at] = (uint64_t)s1 << 32 | s0;
            if (len > 64u) MS.w32[at] = s2;
        }
    }
    if (q != 0u) return;
    S = S < c.fragile_S ? (float)(near_isolated_sum(c, b, e, Ps, MS, nslots, i, pi) * c.mC6_d) : S * c.mC6h6;
    density_finish(c, i, pi, S, D, Q, Pr, flags, near);
}

struct Vec3Sum {
    float x = 0.f, y = 0.f, z = 0.f;
    __device__ __forceinline__ void add(float4 t) {  // t.w (t.x, t.y, t.z)
        x = __builtin_fmaf(t.w, t.x, x);
        y = __builtin_fmaf(t.w, t.y, y);
        z = __builtin_fmaf(t.w, t.z, z);
    }
    template <int R>
    __device__ __forceinline__ Vec3Sum get() const {
        Vec3Sum s;
        s.x = quad_get<R>(x);
        s.y = quad_get<R>(y);
        s.z = quad_get<R>(z);
        return s;
    }
};

__global__ __launch_bounds__(kQuadBlock) void k_normals_quad(
    const Consts *__restrict__ cs, const uint32_t *__restrict__ chunk, uint32_t nslots, const float4 *__restrict__ Q,
    const float *__restrict__ soa, const uint32_t *__restrict__ start, RowMasks M, int all,
    const uint32_t *__restrict__ flags, const uint32_t *__restrict__ moves, const uint8_t *__restrict__ near,
    float4 *__restrict__ N) {
    __shared__ __align__(16) uint32_t lists[kQuadParts * kQuadStride];
    uint32_t i, q;
    const Consts *cp = quad_scene(cs, chunk, i, q);
    if (!cp || (cp->lazy_normal && !all)) return;
    const Consts &c = *cp;
    if (i >= c.first + c.count) return;
    const uint32_t *st = start + c.cell_base;
    const uint32_t shift = c.first - st[0];
    if (i >= st[c.ncells] + shift) {
        if (q == 0u) N[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        return;
    }
    const float4 pi = Q[i];
    const QuadRows rows = quad_rows(c, st, shift, pi, q);
    const RowSource src{c, st, shift, Q, soa, moves, nullptr};
    Vec3Sum sum;
    auto walk = [&]<bool F>() {
        walk_quad(
            lists + (threadIdx.x >> 2) * kQuadStride, src, rows, M, c.use_masks != 0, nslots, i, q, sum,
            [&](uint32_t j) { return at32(Q, j); },
            [&](const float4 &cand, uint32_t, bool ok) {
                const float w = normal_weight<F>(c, pi, cand, dist2(pi, cand), ok);
                return make_float4(pi.x - cand.x, pi.y - cand.y, pi.z - cand.z, w);
            });
    };
    if (flag_set(flag_word(flags, c.scene), kFragileByte) && lanes(quad_near(near, rows)))
        walk.template operator()<true>();
    else
        walk.template operator()<false>();
    if (q == 0u) N[i] = make_float4(c.hmCg6 * sum.x, c.hmCg6 * sum.y, c.hmCg6 * sum.z, 0.0f);
}

template <bool V, bool T, bool F>
struct QuadPairSums : PairSums {
    __device__ __forceinline__ void add(const PairTerm &t) { PairSums::template add<V, T, F>(t); }
    template <int R>
    __device__ __forceinline__ QuadPairSums get() const {
        QuadPairSums s;
        s.Px = quad_get<R>(Px);
        s.Py = quad_get<R>(Py);
        s.Pz = quad_get<R>(Pz);
        if constexpr (F) {
            s.Pdx = quad_get<R>(Pdx);
            s.Pdy = quad_get<R>(Pdy);
            s.Pdz = quad_get<R>(Pdz);
        }
        if constexpr (V) {
            s.Qx = quad_get<R>(Qx);
            s.Qy = quad_get<R>(Qy);
            s.Qz = quad_get<R>(Qz);
        }
        if constexpr (T) {
            s.Tx = quad_get<R>(Tx);
            s.Ty = quad_get<R>(Ty);
            s.Tz = quad_get<R>(Tz);
        }
        return s;
    }
};

__global__ __launch_bounds__(kQuadBlock) void k_forces_quad(
    const Consts *__restrict__ cs, const uint32_t *__restrict__ chunk, uint32_t nslots, const float4 *__restrict__ Ps,
    const float4 *__restrict__ Q, const float *__restrict__ Pr, const float4 *__restrict__ Vs,
    const float4 *__restrict__ A, const float4 *__restrict__ Lw, const uint32_t *__restrict__ order,
    const float4 *__restrict__ D, const float4 *__restrict__ N, const float *__restrict__ soa,
    const uint32_t *__restrict__ start, RowMasks M, float4 *__restrict__ Pout, float4 *__restrict__ Vout,
    float4 *__restrict__ Aout, float4 *__restrict__ Lout, float4 *__restrict__ Fdbg, uint32_t *__restrict__ flags,
    const uint32_t *__restrict__ moves, const uint8_t *__restrict__ near) {
    __shared__ __align__(16) uint32_t lists[kQuadParts * kQuadStride];
    uint32_t i, q;
    const Consts *cp = quad_scene(cs, chunk, i, q);
    if (!cp) return;
    const Consts &c = *cp;
    const uint32_t move_q = scene_move_q(moves, c.scene);
    const uint32_t *st = start + c.cell_base;
    const uint32_t shift = c.first - st[0];
    const bool live = i < c.first + c.count, in_grid = live && i < st[c.ncells] + shift;
    const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
    const float4 pi = live ? Ps[i] : zero, vi = live ? Vs[i] : zero, di = live ? D[i] : zero;
    QuadRows rows = {};
    if (in_grid) rows = quad_rows(c, st, shift, pi, q);
    // The near-isolated walk rounds an ordinary pair's h - r differently
    // (pair_term), so it is chosen for the same 64 slots as in k_forces, the
    // workgroup's.
    bool fragile = false;
    if (flag_set(flag_word(flags, c.scene), kFragileByte)) fragile = __syncthreads_or(quad_near(near, rows)) != 0;
    if (!live) return;
    Forces f;
    if (in_grid) {
        const PairSelf me{pi, vi, di, c.has_tension ? N[i] : zero, di.w * di.w};
        const RowSource src{c, st, shift, Ps, soa, moves, nullptr};
        PairSums sum;
        auto walk = [&]<bool V, bool T, bool F>() {
            QuadPairSums<V, T, F> s;
            walk_quad(
                lists + (threadIdx.x >> 2) * kQuadStride, src, rows, M, c.use_masks != 0, nslots, i, q, s,
                [&](uint32_t j) { return pair_load<V, T>(Q, Pr, Vs, D, N, j); },
                [&](const PairCand &cj, uint32_t, bool ok) {
                    PairTerm t = {};
                    if (!pair_term<V, T, F>(c, me, cj, ok, t)) t = PairTerm{};
                    return t;
                });
            sum = s;
        };
        auto terms = [&]<bool F>() {
            if (c.has_visc) {
                if (c.has_tension)
                    walk.template operator()<true, true, F>();
                else
                    walk.template operator()<true, false, F>();
            } else {
                if (c.has_tension)
                    walk.template operator()<false, true, F>();
                else
                    walk.template operator()<false, false, F>();
            }
        };
        if (fragile)
            terms.template operator()<true>();
        else
            terms.template operator()<false>();
        total_forces(c, pi, di, sum, f);
    }
    if (q == 0u) integrate(c, i, order[i], pi, vi, di.x, f, A, Lw, Pout, Vout, Aout, Lout, Fdbg, flags, move_q);
}

__global__ __launch_bounds__(kQuadBlock) void k_xsph_quad(
    const Consts *__restrict__ cs, const uint32_t *__restrict__ chunk, uint32_t nslots, const float4 *__restrict__ Ps,
    const float4 *__restrict__ Pn, const float4 *__restrict__ Vh, const float4 *__restrict__ Lw,
    const float *__restrict__ soa, const uint32_t *__restrict__ start, RowMasks MS, const uint32_t *__restrict__ flags,
    const uint32_t *__restrict__ moves, const uint8_t *__restrict__ near, float4 *__restrict__ Vout) {
    __shared__ __align__(16) uint32_t lists[kQuadParts * kQuadStride];
    uint32_t i, q;
    const Consts *cp = quad_scene(cs, chunk, i, q);
    if (!cp) return;
    const Consts &c = *cp;
    if (i >= c.first + c.count) return;
    const uint32_t *st = start + c.cell_base;
    const uint32_t shift = c.first - st[0];
    const float4 vi = Vh[i];
    if (i >= st[c.ncells] + shift) {
        if (q == 0u) Vout[i] = make_float4(vi.x, vi.y, vi.z, 0.0f);
        return;
    }
    const uint32_t fl = flag_word(flags, c.scene);
    const float4 xi = Pn[i];
    const QuadRows rows = quad_rows(c, st, shift, Ps[i], q);
    const RowSource src{c, st, shift, Ps, soa, moves, flag_set(fl, kFarMoveByte) ? Pn : nullptr};
    Vec3Sum sum;
    auto walk = [&]<bool F>() {
        walk_quad(
            lists + (threadIdx.x >> 2) * kQuadStride, src, rows, MS, c.use_masks != 0, nslots, i, q, sum,
            [&](uint32_t j) { return XsphCand{at32(Pn, j), at32(Vh, j)}; },
            [&](const XsphCand &cj, uint32_t j, bool ok) {
                const float w = xsph_weight<F>(c, xi, vi.w, cj, lanes(ok), Lw, i, j);
                return make_float4(cj.v.x - vi.x, cj.v.y - vi.y, cj.v.z - vi.z, w);
            });
    };
    if (flag_set(fl, kFragileByte) && lanes(quad_near(near, rows)))
        walk.template operator()<true>();
    else
        walk.template operator()<false>();
    if (q == 0u)
        Vout[i] = make_float4(vi.x + c.xsph_k * sum.x, vi.y + c.xsph_k * sum.y, vi.z + c.xsph_k * sum.z, 0.0f);
}

// ---------------------------------------------------------------------------
// Per-scene data movement and inspection helpers (not on the stepping path).
// Slots [first, first + count) of one scene; ids are scene-local.

__global__ __launch_bounds__(kBlock) void k_upload(const float *__restrict__ stage, uint32_t first, uint32_t id0,
                                                   uint32_t count, float4 *__restrict__ P, float4 *__restrict__ V,
                                                   float4 *__restrict__ A, float4 *__restrict__ L) {
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= count) return;
    const float *s = stage + 9 * (size_t)k;
    const uint32_t id = id0 + k, slot = first + id;
    P[slot] = make_float4(s[0], s[1], s[2], __uint_as_float(id));
    V[slot] = make_float4(s[3], s[4], s[5], 0.0f);
    A[slot] = make_float4(s[6], s[7], s[8], 0.0f);
    L[slot] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}

// The same from one float3 array per quantity (vel and acc may be null: zero).
__global__ __launch_bounds__(kBlock) void k_upload_planes(const float *__restrict__ pos, const float *__restrict__ vel,
                                                          const float *__restrict__ acc, uint32_t first, uint32_t id0,
                                                          uint32_t count, float4 *__restrict__ P,
                                                          float4 *__restrict__ V, float4 *__restrict__ A,
                                                          float4 *__restrict__ L) {
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= count) return;
    const size_t o = 3 * (size_t)k;
    const uint32_t id = id0 + k, slot = first + id;
    P[slot] = make_float4(pos[o], pos[o + 1], pos[o + 2], __uint_as_float(id));
    V[slot] = vel ? make_float4(vel[o], vel[o + 1], vel[o + 2], 0.0f) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    A[slot] = acc ? make_float4(acc[o], acc[o + 1], acc[o + 2], 0.0f) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    L[slot] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}

__global__ __launch_bounds__(kBlock) void k_init_state(uint32_t first, uint32_t count, float4 *__restrict__ P,
                                                       float4 *__restrict__ V, float4 *__restrict__ A,
                                                       float4 *__restrict__ L, float4 *__restrict__ D) {
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= count) return;
    const uint32_t s = first + k;
    P[s] = make_float4(0.f, 0.f, 0.f, __uint_as_float(k));
    V[s] = make_float4(0.f, 0.f, 0.f, 0.f);
    A[s] = make_float4(0.f, 0.f, 0.f, 0.f);
    L[s] = make_float4(0.f, 0.f, 0.f, 0.f);
    D[s] = make_float4(0.f, 0.f, 0.f, 0.f);
}

// Moves slot s to slot first + id(s): the scene's state back to id order.
__global__ __launch_bounds__(kBlock) void k_to_id_order(uint32_t first, uint32_t count, const float4 *__restrict__ P,
                                                        const float4 *__restrict__ V, const float4 *__restrict__ A,
                                                        const float4 *__restrict__ L, const float4 *__restrict__ D,
                                                        float4 *__restrict__ P2, float4 *__restrict__ V2,
                                                        float4 *__restrict__ A2, float4 *__restrict__ L2,
                                                        float4 *__restrict__ D2) {
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= count) return;
    const uint32_t s = first + k;
    const float4 p = P[s];
    const uint32_t d = first + __float_as_uint(p.w);
    P2[d] = p;
    V2[d] = V[s];
    A2[d] = A[s];
    L2[d] = L[s];
    D2[d] = D[s];
}

// Copies `count` slots of five arrays from slot `from` of (P,V,A,L,D) to slot
// `to` of (P2,V2,A2,L2,D2): scene relocation and per-scene reordering.  The
// source and destination arrays are distinct.
__global__ __launch_bounds__(kBlock) void k_move(uint32_t from, uint32_t to, uint32_t count,
                                                 const float4 *__restrict__ P, const float4 *__restrict__ V,
                                                 const float4 *__restrict__ A, const float4 *__restrict__ L,
                                                 const float4 *__restrict__ D, float4 *__restrict__ P2,
                                                 float4 *__restrict__ V2, float4 *__restrict__ A2,
                                                 float4 *__restrict__ L2, float4 *__restrict__ D2) {
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= count) return;
    P2[to + k] = P[from + k];
    V2[to + k] = V[from + k];
    A2[to + k] = A[from + k];
    L2[to + k] = L[from + k];
    D2[to + k] = D[from + k];
}

// Copies `count` slots from `first` of (A, L) to (A2, L2): a paused scene's
// acceleration and low position words, carried to the buffers that become
// the state after a substep (the substep's kernels skip its slots).
__global__ __launch_bounds__(kBlock) void k_carry(uint32_t first, uint32_t count, const float4 *__restrict__ A,
                                                  const float4 *__restrict__ L, float4 *__restrict__ A2,
                                                  float4 *__restrict__ L2) {
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= count) return;
    A2[first + k] = A[first + k];
    L2[first + k] = L[first + k];
}

// AoS staging for downloads: 12 floats per particle (pos, colour, vel, acc).
__global__ __launch_bounds__(kBlock) void k_export(Consts c, const float4 *__restrict__ P,
                                                   const float4 *__restrict__ V, const float4 *__restrict__ A,
                                                   const float4 *__restrict__ D, int by_id, float *__restrict__ out,
                                                   uint32_t *__restrict__ ids) {
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= c.count) return;
    const uint32_t s = c.first + k;
    const float4 p = P[s], v = V[s], a = A[s];
    const uint32_t id = __float_as_uint(p.w);
    const uint32_t dst = by_id ? id : k;
    const float3 col = density_colour(c, D[s].x);
    float *o = out + 12 * (size_t)dst;
    o[0] = p.x; o[1] = p.y; o[2] = p.z;
    o[3] = col.x; o[4] = col.y; o[5] = col.z;
    o[6] = v.x; o[7] = v.y; o[8] = v.z;
    o[9] = a.x; o[10] = a.y; o[11] = a.z;
    ids[dst] = id;
}

// The same as one float3 array per quantity, those that are not null.
__global__ __launch_bounds__(kBlock) void k_export_planes(Consts c, const float4 *__restrict__ P,
                                                          const float4 *__restrict__ V, const float4 *__restrict__ A,
                                                          const float4 *__restrict__ D, int by_id,
                                                          float *__restrict__ pos, float *__restrict__ col,
                                                          float *__restrict__ vel, float *__restrict__ acc,
                                                          uint32_t *__restrict__ ids) {
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= c.count) return;
    const uint32_t s = c.first + k;
    const float4 p = P[s];
    const uint32_t id = __float_as_uint(p.w);
    const uint32_t dst = by_id ? id : k;
    const auto put = [&](float *out, float x, float y, float z) {
        float *o = out + 3 * (size_t)dst;
        o[0] = x;
        o[1] = y;
        o[2] = z;
    };
    if (pos) put(pos, p.x, p.y, p.z);
    if (col) {
        const float3 rgb = density_colour(c, D[s].x);
        put(col, rgb.x, rgb.y, rgb.z);
    }
    if (vel) {
        const float4 v = V[s];
        put(vel, v.x, v.y, v.z);
    }
    if (acc) {
        const float4 a = A[s];
        put(acc, a.x, a.y, a.z);
    }
    if (ids) ids[dst] = id;
}

// Copies up to kCopySpans spans (16-byte aligned, whole words) in one launch:
// between device memory and pinned host memory, where a few hundred kilobytes
// would spend longer in the set-up of one DMA per span.
__global__ __launch_bounds__(kBlock) void k_copy_spans(CopySpans c) {
    const uint32_t *__restrict__ src = static_cast<const uint32_t *>(c.src[blockIdx.y]);
    uint32_t *__restrict__ dst = static_cast<uint32_t *>(c.dst[blockIdx.y]);
    const size_t words = c.bytes[blockIdx.y] / 4u;
    const size_t k = 4u * ((size_t)blockIdx.x * kBlock + threadIdx.x);
    if (k + 4u <= words) {
        *reinterpret_cast<uint4 *>(dst + k) = *reinterpret_cast<const uint4 *>(src + k);
    } else {
        for (size_t q = k; q < words; ++q) dst[q] = src[q];
    }
}

// Exact state in particle-id order, 12 floats per particle: position high
// words, position low words, velocity, acceleration (checkpoints).
__global__ __launch_bounds__(kBlock) void k_state_out(Consts c, const float4 *__restrict__ P,
                                                      const float4 *__restrict__ L, const float4 *__restrict__ V,
                                                      const float4 *__restrict__ A, float *__restrict__ out) {
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= c.count) return;
    const uint32_t s = c.first + k;
    const float4 p = P[s], l = L[s], v = V[s], a = A[s];
    float *o = out + 12 * (size_t)__float_as_uint(p.w);
    o[0] = p.x; o[1] = p.y; o[2] = p.z;
    o[3] = l.x; o[4] = l.y; o[5] = l.z;
    o[6] = v.x; o[7] = v.y; o[8] = v.z;
    o[9] = a.x; o[10] = a.y; o[11] = a.z;
}

// Inverse of k_state_out into a scene in id order (slot first + id).
__global__ __launch_bounds__(kBlock) void k_state_in(uint32_t first, uint32_t count, const float *__restrict__ in,
                                                     float4 *__restrict__ P, float4 *__restrict__ L,
                                                     float4 *__restrict__ V, float4 *__restrict__ A) {
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= count) return;
    const float *i = in + 12 * (size_t)k;
    const uint32_t s = first + k;
    P[s] = make_float4(i[0], i[1], i[2], __uint_as_float(k));
    L[s] = make_float4(i[3], i[4], i[5], 0.0f);
    V[s] = make_float4(i[6], i[7], i[8], 0.0f);
    A[s] = make_float4(i[9], i[10], i[11], 0.0f);
}

// Device-side scene setup.  Both write positions (and clear the low words)
// of particle ids [id0, id0 + count) of a scene in id order; velocities and
// accelerations are left as they are, as the reference's createFluidBlock
// does (fluidsystem.cu:113-126).
//
// Lattice from per-axis coordinate lists (x outermost, z innermost): the
// lists are the FP32 running sums of createFluidBlock's loops.
__global__ __launch_bounds__(kBlock) void k_setup_axes(uint32_t first, uint32_t id0, uint32_t count, uint32_t ny,
                                                       uint32_t nz, const float *__restrict__ ax,
                                                       const float *__restrict__ ay, const float *__restrict__ az,
                                                       float4 *__restrict__ P, float4 *__restrict__ L) {
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= count) return;
    const uint32_t l = k % nz, j = (k / nz) % ny, i = k / (nz * ny);
    const uint32_t id = id0 + k;
    P[first + id] = make_float4(ax[i], ay[j], az[l], __uint_as_float(id));
    L[first + id] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}

// Jittered lattice, the same values as the host generator: the m-th
// SplitMix64 output (m = 3 point + axis + 1, counter-based) gives the
// jitter of one coordinate, evaluated in FP64 without contraction.
__device__ __forceinline__ uint64_t splitmix64_at(uint64_t seed, uint64_t m) {
    uint64_t z = seed + m * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

__global__ __launch_bounds__(kBlock) void k_setup_jitter(uint32_t first, uint32_t id0, uint32_t nx, uint32_t ny,
                                                         uint32_t nz, float dx, float ox, float oy, float oz,
                                                         float jitter, uint64_t seed, float4 *__restrict__ P,
                                                         float4 *__restrict__ L) {
#pragma clang fp contract(off)
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= nx * ny * nz) return;
    const uint32_t idx[3] = {k / (ny * nz), (k / nz) % ny, k % nz};
    const float org[3] = {ox, oy, oz};
    float v[3];
    for (int a = 0; a < 3; ++a) {
        const uint64_t z = splitmix64_at(seed, 3ull * k + (uint64_t)a + 1ull);
        const double u = 2.0 * ((double)(z >> 11) * (1.0 / 9007199254740992.0)) - 1.0;
        v[a] = (float)((double)org[a] + ((double)idx[a] + 0.5) * (double)dx + u * (double)jitter);
    }
    const uint32_t id = id0 + k;
    P[first + id] = make_float4(v[0], v[1], v[2], __uint_as_float(id));
    L[first + id] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}

// Neighbour sets of the density pass (debug): count, then fill; indexed by
// the scene-local slot.
__global__ __launch_bounds__(kBlock) void k_nb_count(Consts c, const float4 *__restrict__ Ps,
                                                     const uint32_t *__restrict__ start, uint32_t *__restrict__ cnt) {
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= c.count) return;
    const uint32_t i = c.first + k;
    const uint32_t *st = start + c.cell_base;
    const uint32_t shift = c.first - st[0];
    uint32_t num = 0;
    if (i < st[c.ncells] + shift) {
        const float4 pi = Ps[i];
        int cx, cy, cz;
        cell_xyz(c, pi, cx, cy, cz);
        for_stencil(c, st, shift, cx, cy, cz, [&](uint32_t j) {
            if (dist2(pi, Ps[j]) <= c.h2 && j != i) ++num;
        });
    }
    cnt[k] = num;
}

__global__ __launch_bounds__(kBlock) void k_nb_fill(Consts c, const float4 *__restrict__ Ps,
                                                    const uint32_t *__restrict__ start,
                                                    const uint64_t *__restrict__ off, uint32_t *__restrict__ list) {
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= c.count) return;
    const uint32_t i = c.first + k;
    const uint32_t *st = start + c.cell_base;
    const uint32_t shift = c.first - st[0];
    if (i >= st[c.ncells] + shift) return;
    const float4 pi = Ps[i];
    int cx, cy, cz;
    cell_xyz(c, pi, cx, cy, cz);
    uint64_t o = off[k];
    for_stencil(c, st, shift, cx, cy, cz, [&](uint32_t j) {
        const float4 q = Ps[j];
        if (dist2(pi, q) <= c.h2 && j != i) list[o++] = __float_as_uint(q.w);
    });
}

__global__ __launch_bounds__(kBlock) void k_copy(const float4 *__restrict__ src, float4 *__restrict__ dst,
                                                 size_t n4) {
    size_t k = (size_t)blockIdx.x * kBlock + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * kBlock;
    for (; k < n4; k += stride) dst[k] = src[k];
}

// ---------------------------------------------------------------------------
// Host launchers.  A timed launch goes through hipExtLaunchKernelGGL, so that
// its start/stop events are bound to the dispatch packet itself; an untimed
// one through hipLaunchKernelGGL (also under stream capture).

static inline unsigned blocks_for(size_t n, unsigned bs = kBlock) { return (unsigned)((n + bs - 1) / bs); }

#define LF_GO(L, kern, nblocks, bs, ev0, ev1, ...)                                                        \
    do {                                                                                                  \
        if ((ev0) || (ev1))                                                                               \
            hipExtLaunchKernelGGL(kern, dim3(nblocks), dim3(bs), 0, (L).st, (ev0), (ev1), 0, __VA_ARGS__); \
        else                                                                                              \
            hipLaunchKernelGGL(kern, dim3(nblocks), dim3(bs), 0, (L).st, __VA_ARGS__);                    \
    } while (0)

// Runs body.template operator()<BS>() for the block size bs (128, 256, 512).
template <class F>
static inline void with_bs(int bs, F &&body) {
    switch (bs) {
        case 128: body.template operator()<128>(); break;
        case 512: body.template operator()<512>(); break;
        default: body.template operator()<256>(); break;
    }
}

// Which launches take four lanes per particle in the neighbour passes: those
// whose active scenes hold so few slots that one lane each leaves the chip's
// 1,024 SIMDs with less than a wave or two.  A slot counts by what its pairs
// cost: kQuadSlots plain ones fill a launch, or kQuadSlotsFull of scenes with
// viscosity or tension, or kQuadSlotsLong of those whose stencil rows hold
// more than 32 slots at rest density.  A substep with one / four lanes, us:
//   plain, block 49,152 56.4 / 46.5, 61,440 57.3 / 55.8; spray 61,440 58.7 /
//   57.7; 16 scenes of 4,000 53.1 / 54.2; 65,000 in the splash 91 / 91
//   full, block 65,536 75.4 / 70.5, 81,920 84.9 / 85.6, 98,304 87.4 / 93.6;
//   spray (0.4 a cell) 65,536 69.2 / 67.2, 73,728 72.7 / 80.4; 17 scenes of
//   4,000 80.2 / 81.7, 24 of them 78.9 / 93.5
//   full with long rows, double dam 81,920 141 / 117 at rest and 377 / 305 in
//   the splash, 98,304 144 / 129 and 395 / 396; 131,000 521 / 519
//   mixed, 12 plain scenes of 4,000 and a full one of 500 68.5 / 59.2, 16 and
//   one 67.7 / 68.5, 16 and 8 of 4,000 78.4 / 92.7
// Slots of paused scenes only cost their empty workgroups: every other of 24
// plain scenes of 4,000 paused (98,304 launched) 77.1 / 75.2.  Longer
// launches take one lane.
constexpr double kQuadSlots = 61440, kQuadSlotsFull = 65536, kQuadSlotsLong = 98304;
constexpr uint32_t kQuadLaunch = 98304;
double quad_share(const lf_params &p, uint32_t slots) {
    if (p.viscosity == 0.0f && p.surface_tension == 0.0f) return slots / kQuadSlots;
    const double per_cell =
        (double)p.rest_density / ((double)p.mass * p.inv_cell[0] * p.inv_cell[1] * p.inv_cell[2]);
    return slots / (3.0 * per_cell > 32.0 ? kQuadSlotsLong : kQuadSlotsFull);
}
bool takes_quads(double share, uint32_t nlaunch) { return nlaunch <= kQuadLaunch && share <= 1.0 + 1e-9; }

bool valid_block_size(int bs) { return bs == 128 || bs == 256 || bs == 512; }

void launch_hash(const Launch &L, const PoolView &pv, const float4 *P, uint32_t *keys, uint32_t *ranks,
                 uint32_t *counts, uint32_t *flags, uint32_t *moves, uint32_t *nsegs) {
    LF_GO(L, k_hash, pv.nlaunch / (kBlock * kHashItems), kBlock, L.a, L.b, pv.cs, pv.chunk, P, keys, ranks, counts,
          flags, moves, nsegs);
}

uint32_t scan_tiles(uint32_t m) { return (m + kScanTile - 1) / kScanTile; }

// Whether launch_scan scans m buckets in one launch (and launch_scatter
// clears their counts).
static inline bool scan_in_one(uint32_t m) { return m <= kScanOneTiles * kScanOneTile; }

void launch_scan(const Launch &L, uint32_t *counts, uint32_t m, uint32_t *bsum, uint32_t *start) {
    if (scan_in_one(m)) {
        LF_GO(L, k_scan_one, (m + kScanOneTile - 1u) / kScanOneTile, kScanOneThreads, L.a, L.b,
              (const uint32_t *)counts, m, start);
        return;
    }
    const uint32_t nb = scan_tiles(m);
    const bool prefixed = nb > kScanDirectTiles;
    LF_GO(L, k_scan_sum, nb, kBlock, L.a, nullptr, (const uint32_t *)counts, m, bsum);
    if (prefixed) LF_GO(L, k_scan_tiles, 1, kBlock, nullptr, nullptr, bsum, nb);
    LF_GO(L, k_scan_down, nb, kBlock, nullptr, L.b, counts, m, (const uint32_t *)bsum, nb, prefixed ? 1 : 0, start);
}

void launch_scatter(const Launch &L, const PoolView &pv, const float4 *P, const uint32_t *keys, const uint32_t *ranks,
                    const uint32_t *start, uint32_t *slot_src, uint32_t *slot_id, uint4 *segs, uint32_t *nsegs,
                    uint2 *tmp, uint32_t *counts, uint32_t m) {
    LF_GO(L, k_scatter, pv.nlaunch / kBlock, kBlock, L.a, nullptr, pv.cs, pv.chunk, P, keys, ranks, start, slot_src,
          slot_id, segs, nsegs, counts, scan_in_one(m) ? m : 0u);
    LF_GO(L, k_sort_segments, kSegBlocks, kSegThreads, nullptr, L.b, (const uint4 *)segs, (const uint32_t *)nsegs,
          slot_id, slot_src, tmp);
}

void launch_gather(const Launch &L, const PoolView &pv, const uint32_t *slot_src, const uint32_t *slot_id,
                   const uint32_t *keys, const uint32_t *start, const float4 *P, const float4 *V, float4 *Ps,
                   float4 *Vs, uint32_t *order, float *soa, uint32_t *moves) {
    LF_GO(L, k_gather, pv.nlaunch / kBlock, kBlock, L.a, L.b, pv.cs, pv.chunk, slot_src, slot_id, keys, start, P, V,
          Ps, Vs, order, soa, pv.nslots, pv.near, moves);
}

void launch_density(const Launch &L, const PoolView &pv, int bs, const float4 *Ps, const float *soa,
                    const uint32_t *start, float4 *D, float4 *Q, float *Pr, RowMasks MS, uint32_t *flags,
                    const uint32_t *moves) {
    if (pv.quads) {
        LF_GO(L, k_density_quad, pv.nlaunch / kQuadParts, kQuadBlock, L.a, L.b, pv.cs, pv.chunk, pv.nslots, Ps, soa,
              start, D, Q, Pr, MS, flags, moves, pv.near);
        return;
    }
    with_bs(bs, [&]<int BS>() {
        LF_GO(L, k_density<BS>, pv.nlaunch / BS, BS, L.a, L.b, pv.cs, pv.chunk, pv.nslots, Ps, soa, start, D, Q, Pr,
              MS, flags, moves, pv.near);
    });
}

void launch_normals(const Launch &L, const PoolView &pv, int bs, int flat, bool all, const float4 *Q,
                    const float *soa, const uint32_t *start, RowMasks M, const uint32_t *flags, const uint32_t *moves,
                    float4 *N) {
    if (pv.quads) {
        LF_GO(L, k_normals_quad, pv.nlaunch / kQuadParts, kQuadBlock, L.a, L.b, pv.cs, pv.chunk, pv.nslots, Q, soa,
              start, M, all ? 1 : 0, flags, moves, pv.near, N);
        return;
    }
    with_bs(bs, [&]<int BS>() {
        LF_GO(L, k_normals<BS>, pv.nlaunch / BS, BS, L.a, L.b, pv.cs, pv.chunk, pv.nslots, Q, soa, start, M,
              flat, all ? 1 : 0, flags, moves, pv.near, N);
    });
}

void launch_forces(const Launch &L, const PoolView &pv, int bs, int flat, const float4 *Ps, const float4 *Q,
                   const float *Pr, const float4 *Vs, const float4 *A, const float4 *Lw, const uint32_t *order,
                   const float4 *D, const float4 *N, const float *soa, const uint32_t *start, RowMasks M,
                   float4 *Pout, float4 *Vout, float4 *Aout, float4 *Lout, float4 *Fdbg, uint32_t *flags,
                   const uint32_t *moves) {
    if (pv.quads) {
        LF_GO(L, k_forces_quad, pv.nlaunch / kQuadParts, kQuadBlock, L.a, L.b, pv.cs, pv.chunk, pv.nslots, Ps, Q, Pr,
              Vs, A, Lw, order, D, N, soa, start, M, Pout, Vout, Aout, Lout, Fdbg, flags, moves, pv.near);
        return;
    }
    with_bs(bs, [&]<int BS>() {
        LF_GO(L, k_forces<BS>, pv.nlaunch / BS, BS, L.a, L.b, pv.cs, pv.chunk, pv.nslots, Ps, Q, Pr, Vs, A, Lw, order,
              D, N, soa, start, M, flat, Pout, Vout, Aout, Lout, Fdbg, flags, moves, pv.near);
    });
}

void launch_xsph(const Launch &L, const PoolView &pv, int bs, int flat, const float4 *Ps, const float4 *Pn,
                 const float4 *Vh, const float4 *Lw, const float *soa, const uint32_t *start, RowMasks MS,
                 const uint32_t *flags, const uint32_t *moves, float4 *Vout) {
    if (pv.quads) {
        LF_GO(L, k_xsph_quad, pv.nlaunch / kQuadParts, kQuadBlock, L.a, L.b, pv.cs, pv.chunk, pv.nslots, Ps, Pn, Vh,
              Lw, soa, start, MS, flags, moves, pv.near, Vout);
        return;
    }
    with_bs(bs, [&]<int BS>() {
        LF_GO(L, k_xsph<BS>, pv.nlaunch / BS, BS, L.a, L.b, pv.cs, pv.chunk, pv.nslots, Ps, Pn, Vh, Lw, soa,
              start, MS, flat, flags, moves, pv.near, Vout);
    });
}

void launch_upload(hipStream_t st, const float *stage, uint32_t first, uint32_t id0, uint32_t count, float4 *P,
                   float4 *V, float4 *A, float4 *Lw) {
    if (count)
        hipLaunchKernelGGL(k_upload, dim3(blocks_for(count)), dim3(kBlock), 0, st, stage, first, id0, count, P, V, A,
                           Lw);
}

void launch_init_state(hipStream_t st, uint32_t first, uint32_t count, float4 *P, float4 *V, float4 *A, float4 *Lw,
                       float4 *D) {
    if (count)
        hipLaunchKernelGGL(k_init_state, dim3(blocks_for(count)), dim3(kBlock), 0, st, first, count, P, V, A, Lw, D);
}

void launch_to_id_order(hipStream_t st, uint32_t first, uint32_t count, const float4 *P, const float4 *V,
                        const float4 *A, const float4 *Lw, const float4 *D, float4 *P2, float4 *V2, float4 *A2,
                        float4 *L2, float4 *D2) {
    if (count)
        hipLaunchKernelGGL(k_to_id_order, dim3(blocks_for(count)), dim3(kBlock), 0, st, first, count, P, V, A, Lw, D,
                           P2, V2, A2, L2, D2);
}

void launch_move(hipStream_t st, uint32_t from, uint32_t to, uint32_t count, const float4 *P, const float4 *V,
                 const float4 *A, const float4 *Lw, const float4 *D, float4 *P2, float4 *V2, float4 *A2, float4 *L2,
                 float4 *D2) {
    if (count)
        hipLaunchKernelGGL(k_move, dim3(blocks_for(count)), dim3(kBlock), 0, st, from, to, count, P, V, A, Lw, D, P2,
                           V2, A2, L2, D2);
}

void launch_carry(hipStream_t st, uint32_t first, uint32_t count, const float4 *A, const float4 *Lw, float4 *A2,
                  float4 *L2) {
    if (count)
        hipLaunchKernelGGL(k_carry, dim3(blocks_for(count)), dim3(kBlock), 0, st, first, count, A, Lw, A2, L2);
}

void launch_export(hipStream_t st, const Consts &c, const float4 *P, const float4 *V, const float4 *A,
                   const float4 *D, bool by_id, float *out, uint32_t *ids) {  // ids may not be null
    if (c.count)
        hipLaunchKernelGGL(k_export, dim3(blocks_for(c.count)), dim3(kBlock), 0, st, c, P, V, A, D, by_id ? 1 : 0,
                           out, ids);
}

void launch_upload_planes(hipStream_t st, const float *pos, const float *vel, const float *acc, uint32_t first,
                          uint32_t id0, uint32_t count, float4 *P, float4 *V, float4 *A, float4 *Lw) {
    if (count)
        hipLaunchKernelGGL(k_upload_planes, dim3(blocks_for(count)), dim3(kBlock), 0, st, pos, vel, acc, first, id0,
                           count, P, V, A, Lw);
}

void launch_export_planes(hipStream_t st, const Consts &c, const float4 *P, const float4 *V, const float4 *A,
                          const float4 *D, bool by_id, float *pos, float *col, float *vel, float *acc,
                          uint32_t *ids) {
    if (c.count)
        hipLaunchKernelGGL(k_export_planes, dim3(blocks_for(c.count)), dim3(kBlock), 0, st, c, P, V, A, D,
                           by_id ? 1 : 0, pos, col, vel, acc, ids);
}

void launch_copy_spans(hipStream_t st, const CopySpans &c, uint32_t count) {
    size_t most = 0;
    for (uint32_t k = 0; k < count; ++k) most = std::max(most, c.bytes[k]);
    if (most)
        hipLaunchKernelGGL(k_copy_spans, dim3(blocks_for((most + 15) / 16), count), dim3(kBlock), 0, st, c);
}

void launch_state_out(hipStream_t st, const Consts &c, const float4 *P, const float4 *Lw, const float4 *V,
                      const float4 *A, float *out) {
    if (c.count)
        hipLaunchKernelGGL(k_state_out, dim3(blocks_for(c.count)), dim3(kBlock), 0, st, c, P, Lw, V, A, out);
}

void launch_state_in(hipStream_t st, uint32_t first, uint32_t count, const float *in, float4 *P, float4 *Lw,
                     float4 *V, float4 *A) {
    if (count)
        hipLaunchKernelGGL(k_state_in, dim3(blocks_for(count)), dim3(kBlock), 0, st, first, count, in, P, Lw, V, A);
}

void launch_setup_axes(hipStream_t st, uint32_t first, uint32_t id0, uint32_t count, uint32_t ny, uint32_t nz,
                       const float *ax, const float *ay, const float *az, float4 *P, float4 *Lw) {
    if (count)
        hipLaunchKernelGGL(k_setup_axes, dim3(blocks_for(count)), dim3(kBlock), 0, st, first, id0, count, ny, nz, ax,
                           ay, az, P, Lw);
}

void launch_setup_jitter(hipStream_t st, uint32_t first, uint32_t id0, uint32_t nx, uint32_t ny, uint32_t nz,
                         float dx, const float origin[3], float jitter, uint64_t seed, float4 *P, float4 *Lw) {
    const size_t n = (size_t)nx * ny * nz;
    if (n)
        hipLaunchKernelGGL(k_setup_jitter, dim3(blocks_for(n)), dim3(kBlock), 0, st, first, id0, nx, ny, nz, dx,
                           origin[0], origin[1], origin[2], jitter, seed, P, Lw);
}

void launch_nb_count(hipStream_t st, const Consts &c, const float4 *Ps, const uint32_t *start, uint32_t *cnt) {
    if (c.count) hipLaunchKernelGGL(k_nb_count, dim3(blocks_for(c.count)), dim3(kBlock), 0, st, c, Ps, start, cnt);
}

void launch_nb_fill(hipStream_t st, const Consts &c, const float4 *Ps, const uint32_t *start, const uint64_t *off,
                    uint32_t *list) {
    if (c.count)
        hipLaunchKernelGGL(k_nb_fill, dim3(blocks_for(c.count)), dim3(kBlock), 0, st, c, Ps, start, off, list);
}

void launch_copy(const Launch &L, const float4 *src, float4 *dst, size_t n4) {
    const unsigned nb = (unsigned)std::min<size_t>(std::max<size_t>(blocks_for(n4), 1), 65536);
    LF_GO(L, k_copy, nb, kBlock, L.a, L.b, src, dst, n4);
}

}  // namespace lf
