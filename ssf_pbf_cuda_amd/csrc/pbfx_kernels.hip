// pbfx_kernels.hip -- HIP kernels of the PBF solver step for gfx950 (CDNA4).
//
// One step = bookkeeping kernels (predict+hash+histogram, scan, scatter, stable
// reorder), then:
//   k_ns_groups, k_ns_big        neighbour lists (frozen, capped), eight lanes a particle
//   k_lambda                     lambda over the lists, 16, 4 or 1 lanes a particle (x I)
//   k_deltap                     delta-p + tensile correction + boundary response   (x I)
//   k_cur_*                      regrouping by final cell       (vort_on or xsph_on)
//   k_final_groups, k_final_big  in-range pairs around each final cell
//   k_ovf_part                   per-cell partial sums of particles in piles, before
//                                each of the next three
//   k_vort                       vorticity over the final lists             (vort_on)
//   k_confine                    vorticity confinement                      (vort_on)
//   k_xsph_out                   XSPH + AoS write-back                      (xsph_on)
//   k_out                        AoS write-back                             (otherwise)
// All kernels are integer or FP32 vector work; nothing is a contraction, so MFMA
// is not used.  Arithmetic follows the reference's
// operation order with IEEE division/sqrt and explicit fmaf (the library is
// compiled with -ffp-contract=off), so results are reproducible bit-for-bit
// on the host.
#include "pbfx_device.hpp"

#include <algorithm>
#include <climits>
#include <type_traits>

namespace pbfx {
namespace {

// ------------------------------------------------- K1: predict + hash + histogram
// pbf_predict.cu:15-45 (v* = fmaf(g,dt,v), x* = fmaf(v*,dt,x)), calcHashCUDA
// (pbf_neighbor_search_util.cu:20-37), checkDeleteParticleCUDA
// (pbf_delete.cu:9-28, sentinel key CT) and the histogram of insertAndCountCUDA
// (pbf_counting_sort.cu:21-32) with wave-aggregated atomics; each particle
// marks its 4096-cell scan tile as occupied (a plain store, no contention).
// Input i belongs to the scene whose input range holds it.  A batch takes
// its input count from the device (in_off[nscenes], at most n, the count the
// grid was sized for), so that a recorded graph of steps stays valid while
// deletion shrinks the scenes.  The first workgroup also clears the step's
// counters.
template <bool kB>
__global__ __launch_bounds__(256) void k_predict_hash(const float* __restrict__ x, const float* __restrict__ v,
                                                      uint32_t n, Bufs b, Scenes<kB> SC, uint32_t* __restrict__ key,
                                                      uint32_t* __restrict__ rank, uint32_t* __restrict__ count,
                                                      uint32_t* __restrict__ tflag, uint32_t lgT) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (blockIdx.x == 0u)
        for (uint32_t t = threadIdx.x; t < kCtrWords; t += blockDim.x) b.ctr[t] = 0;
    const bool active = i < (kB ? min(n, b.in_off[b.nscenes]) : n);
    uint32_t k = 0;
    const uint32_t si = active ? scene_index<kB>(b.in_off, b.nscenes, i) : 0u;
    by_scene<kB>(si, active, [&](uint32_t sc) {
        const Scene& S = SC[sc];
        const float dt = S.P.dt;
        float q[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            float vs = __builtin_fmaf(S.P.g[c], dt, v[3 * i + c]);
            q[c] = __builtin_fmaf(vs, dt, x[3 * i + c]);
        }
        const Grid G = S.G;
        int gp[3];
        grid_pos(mk3(q[0], q[1], q[2]), G.cw, gp);
        k = scene_key(gp[0], gp[1], gp[2], G);
        if (q[0] < S.lo[0] || S.hi[0] < q[0] || q[1] < S.lo[1] || S.hi[1] < q[1] || q[2] < S.lo[2] ||
            S.hi[2] < q[2])
            k = b.CT;
    });
    const uint32_t r = wave_rank(count, k, active, k);
    if (active) {
        mark_tile(tflag, k >> lgT);
        key[i] = k;
        rank[i] = r;
        if (kB) b.isid[i] = si;
    }
}

// Where the counter of key c is stored.  lgnc = 0: at c.  Otherwise keys are
// (run << lgnc | copy) and copy j of every run lives in region j of C >> lgnc
// words, so that the copies of one run sit on different cache lines: a run
// that gathers particles from the whole domain (a wall or corner pile) is
// counted through nc separate lines instead of one.
__device__ __forceinline__ uint32_t count_slot(uint32_t c, uint32_t C, uint32_t lgnc) {
    return (c & ((1u << lgnc) - 1u)) * (C >> lgnc) + (c >> lgnc);
}

// ------------------------------------------------- K2a: per-tile totals
// Totals of the cell counts of each occupied scan tile (unoccupied tiles are
// all zero); tile nT is the deleted bucket (cell C).  Left out up to kDirectTiles
// tiles, where k_scan_cells sums the counts before its tile itself.
// k_scan_cells has kScanBlock threads a workgroup; a tile of at most kScanTile
// cells gives each thread at most kScanPer of them.
constexpr uint32_t kScanBlock = 512;
constexpr uint32_t kScanPer = kScanTile / kScanBlock;
constexpr uint32_t kScanWaves = kScanBlock / 64;

__global__ __launch_bounds__(kBlock) void k_tile_reduce(const uint32_t* __restrict__ count,
                                                            const uint32_t* __restrict__ tflag, uint32_t* __restrict__ tsum,
                                                            uint32_t nT, uint32_t lgT, uint32_t C, uint32_t lgnc) {
    __shared__ uint32_t wsum[kWaves];
    const uint32_t t = blockIdx.x;
    if (t == nT) {
        if (threadIdx.x == 0) tsum[nT] = count[C];
        return;
    }
    if (tflag[t] == 0u) {
        if (threadIdx.x == 0) tsum[t] = 0u;
        return;
    }
    const uint32_t T = 1u << lgT, c0 = t << lgT;
    // all of a thread's loads are issued before the first add
    uint32_t v[kScanTile / kBlock];
#pragma unroll
    for (uint32_t k = 0; k < kScanTile / kBlock; ++k) {
        const uint32_t j = threadIdx.x + k * kBlock;
        v[k] = j < T ? count[count_slot(c0 + j, C, lgnc)] : 0u;
    }
    uint32_t s = 0;
#pragma unroll
    for (uint32_t k = 0; k < kScanTile / kBlock; ++k) s += v[k];
    uint32_t total;
    block_excl_scan(s, wsum, total);
    if (threadIdx.x == 0) tsum[t] = total;
}

// ------------------------------------------------- K2: scan of the tile totals
// One workgroup: exclusive scan of tsum[0..nT] (nT real tiles + the deleted
// bucket).  Left out up to kPrefixTiles tiles, where k_scan_cells sums the totals
// before its tile itself.
__global__ __launch_bounds__(1024) void k_scan_tiles(const uint32_t* __restrict__ tsum,
                                                     uint32_t* __restrict__ tprefix, uint32_t nT1) {
    __shared__ uint32_t wsum[16];
    const uint32_t per = (nT1 + blockDim.x - 1) / blockDim.x;
    const uint32_t b0 = threadIdx.x * per;
    uint32_t s = 0;
    for (uint32_t j = 0; j < per; ++j)
        if (b0 + j < nT1) s += tsum[b0 + j];
    const uint32_t lane = lane_id(), wid = threadIdx.x >> 6;
    uint32_t xs = s;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        uint32_t y = __shfl_up(xs, d, 64);
        if (lane >= (uint32_t)d) xs += y;
    }
    if (lane == 63) wsum[wid] = xs;
    __syncthreads();
    uint32_t off = 0;
    for (uint32_t w = 0; w < wid; ++w) off += wsum[w];
    uint32_t run = off + xs - s;
    for (uint32_t j = 0; j < per; ++j)
        if (b0 + j < nT1) {
            tprefix[b0 + j] = run;
            run += tsum[b0 + j];
        }
}

// ------------------------------------------------- K3: scan of the cell counts
// Workgroup t scans the counts of cell tile t (empty tiles only write their
// prefix), clears the counts it read and the tile's occupied flag; the last
// workgroup writes the deleted bucket: off[C] = live count, off[C+1] = n (also to
// live[0..1] when given).
// (CUB DeviceScan::ExclusiveSum in pbf_counting_sort.cu:62-71.)
//
// What the cells before the tile hold comes from tprefix (k_scan_tiles), from the
// tile totals (tprefix NULL) or from the counts themselves (tsum NULL: then
// another workgroup may still read a count, and the next kernel over them clears
// them).  A small step is a chain of short launches, about 2 us each and another
// between two of them; with totals and prefixes in launches of their own, its two
// scans were six of 35.
//
// With the offsets of its tile in LDS, the workgroup also lists the work
// items of the tile's runs (kEmit, no run straddles a tile) with one atomic
// on the item counter:
//   EMIT_SEARCH  each run of uw cells along x.  A run whose estimated 27-cell
//                neighbourhood (9 rows of W+2 cells at the run's mean density)
//                exceeds `budget` particles is split into narrower units, and a
//                unit with more than kChunk own particles into several items
//                that share its neighbourhood (item = (first cell, W | chunk
//                << 6)).  Also counts the occupied tiles (CTR_SCANTILES).
//   EMIT_FINAL   each run of uw final cells (1 << lgrun counters) holding
//                at least kSparse particles, one item per kChunk of them.
// Listed here, the counter takes one atomic per occupied tile (128 on the 1M
// dam).  Listed by the wave that meets a run's first particle, as the reorder
// and the regrouping's scatter did, it takes thousands, which one address
// serialises: k_reorder took 101 us on the 1M dam and 756 us on the 8M double
// dam at uw = 16, now 15 and 153; k_cur_scatter 24 and 329 us, now 14 and 138;
// k_scan_cells 18 and 122 us in its two launches, now 22 and 122, of which the sum
// before a tile replaces k_scan_tiles up to kPrefixTiles (7 us at 1M).
enum EmitMode : int { EMIT_NONE = 0, EMIT_SEARCH, EMIT_FINAL };
struct EmitArgs {
    uint32_t uw, lguw, lgrun, budget;  // lgrun: tile words per run
    uint2* units;
    uint32_t* nunits;
};

// Calls item(first cell, W | chunk << 6) for the items of the search run of uw
// cells starting at tile cell r0 (key kb); off(c) gives a tile cell's offset.
template <class OffF, class ItemF>
__device__ __forceinline__ void search_items(uint32_t r0, uint32_t kb, uint32_t uw, uint32_t budget, OffF&& off,
                                             ItemF&& item) {
    const uint32_t nseg = off(r0 + uw) - off(r0);
    if (nseg == 0u) return;
    uint32_t W = uw;
    while (W > 1u && 9ull * (W + 2u) * nseg > (unsigned long long)budget * uw) W >>= 1;
    for (uint32_t q0 = 0; q0 < uw; q0 += W) {
        const uint32_t nch = (off(r0 + q0 + W) - off(r0 + q0) + kChunk - 1u) / kChunk;
        for (uint32_t c = 0; c < nch; ++c) item(kb + q0, W | (c << 6));
    }
}

// Sum of v over the workgroup.
__device__ __forceinline__ uint32_t block_sum(uint32_t v, uint32_t* wsum) {
    uint32_t total;
    block_excl_scan(v, wsum, total);
    return total;
}

template <int kEmit>
__global__ __launch_bounds__(kScanBlock) void k_scan_cells(uint32_t* __restrict__ count, uint32_t* __restrict__ offset,
                                                           const uint32_t* __restrict__ tsum, uint32_t* __restrict__ tflag,
                                                           const uint32_t* __restrict__ tprefix, uint32_t nT,
                                                           uint32_t lgT, uint32_t C, uint32_t lgnc, EmitArgs E,
                                                           uint32_t* __restrict__ stat, uint32_t* __restrict__ live) {
    __shared__ uint32_t wsum[kScanWaves];
    const uint32_t t = blockIdx.x;
    const uint32_t T = 1u << lgT, c0 = t << lgT;
    // the tile's counts and what is summed before it are loaded together; an empty
    // tile's are not, where the totals tell (most tiles of a large grid)
    const bool own = t < nT && (!tsum || tsum[t] != 0u);
    uint32_t v[kScanPer];
#pragma unroll
    for (uint32_t k = 0; k < kScanPer; ++k) {
        const uint32_t j = threadIdx.x + k * kScanBlock;
        v[k] = own && j < T ? count[count_slot(c0 + j, C, lgnc)] : 0u;
    }
    uint32_t base;
    if (tprefix) {
        base = tprefix[t];
    } else {
        uint32_t s = 0;
        if (tsum) {
            for (uint32_t j = threadIdx.x; j < t; j += kScanBlock) s += tsum[j];
        } else if (T == kScanTile) {
            // a thread takes four words (of one copy's region) at a time of each tile before
            static_assert(kScanPer % 4u == 0u, "four words at a time");
            const uint32_t lgw = lgT - lgnc;
#pragma unroll
            for (uint32_t h = 0; h < kScanPer / 4u; ++h) {
                const uint32_t in = (threadIdx.x + h * kScanBlock) * 4u;
                const uint32_t* __restrict__ p = count + (in >> lgw) * (C >> lgnc) + (in & ((1u << lgw) - 1u));
#pragma unroll 8
                for (uint32_t k = 0; k < t; ++k) {
                    const uint4 c4 = *reinterpret_cast<const uint4*>(p + (k << lgw));
                    s += c4.x + c4.y + c4.z + c4.w;
                }
            }
        } else {
            const uint32_t lgw = lgT - lgnc;
            for (uint32_t j = threadIdx.x; j < c0; j += kScanBlock) {
                const uint32_t in = j & (T - 1u);
                s += count[(in >> lgw) * (C >> lgnc) + ((j >> lgT) << lgw) + (in & ((1u << lgw) - 1u))];
            }
        }
        base = block_sum(s, wsum);
    }
    if (t == nT) {
        if (threadIdx.x == 0) {
            const uint32_t end = base + (tsum ? tsum[nT] : count[C]);
            offset[C] = base;
            offset[C + 1] = end;
            if (live) {
                live[0] = base;
                live[1] = end;
            }
            if (tsum) {
                count[C] = 0;
                tflag[nT] = 0;
            }
        }
        return;
    }
    if ((tsum ? tsum[t] : tflag[t]) == 0u) {
        for (uint32_t i = threadIdx.x; i < T; i += blockDim.x) offset[c0 + i] = base;
        return;
    }
    if (kEmit == EMIT_SEARCH && threadIdx.x == 0) atomicAdd(&stat[CTR_NUM * (1u + (t & (kStatRep - 1u))) + CTR_SCANTILES], 1u);
    // The tile passes through LDS so that global reads and writes are
    // coalesced; thread t scans cells t*per .. t*per+per-1 there.  Word w is
    // kept at w + w/16, so the threads' strides hit distinct banks.
    __shared__ uint32_t cell[kScanTile + kScanTile / 16 + 1];
    auto at = [](uint32_t w) { return w + (w >> 4); };
#pragma unroll
    for (uint32_t k = 0; k < kScanPer; ++k) {
        const uint32_t j = threadIdx.x + k * kScanBlock;
        if (j < T) cell[at(j)] = v[k];
    }
    __syncthreads();
    const uint32_t per = (T + blockDim.x - 1) / blockDim.x;
    const uint32_t my0 = threadIdx.x * per;
    const uint32_t myn = (my0 < T) ? min(per, T - my0) : 0u;
    uint32_t s = 0;
    for (uint32_t j = 0; j < myn; ++j) s += cell[at(my0 + j)];
    uint32_t total;
    uint32_t run = base + block_excl_scan(s, wsum, total);
    for (uint32_t j = 0; j < myn; ++j) {
        const uint32_t c = cell[at(my0 + j)];
        cell[at(my0 + j)] = run;
        run += c;
    }
    if (kEmit != EMIT_NONE && threadIdx.x == 0) cell[at(T)] = base + total;
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < T; i += blockDim.x) {
        offset[c0 + i] = cell[at(i)];
        if (tsum) count[count_slot(c0 + i, C, lgnc)] = 0;
    }
    if (tsum && threadIdx.x == 0) tflag[t] = 0;
    if (kEmit == EMIT_NONE) return;
    // thread t takes consecutive runs, so that the items stay in key order
    __shared__ uint32_t ubase;
    auto off = [&](uint32_t c) { return cell[at(c)]; };
    const uint32_t lgrun = E.lgrun;
    const uint32_t nrun = T >> lgrun, rper = (nrun + blockDim.x - 1) / blockDim.x;
    const uint32_t r0 = threadIdx.x * rper, r1 = min(r0 + rper, nrun);
    auto items = [&](auto&& item) {
        for (uint32_t r = r0; r < r1; ++r) {
            if (kEmit == EMIT_SEARCH) {
                search_items(r << lgrun, c0 + (r << lgrun), E.uw, E.budget, off, item);
            } else {
                const uint32_t own = off((r + 1u) << lgrun) - off(r << lgrun);
                const uint32_t nch = own >= kSparse ? (own + kChunk - 1u) / kChunk : 0u;
                for (uint32_t c = 0; c < nch; ++c) item(((c0 >> lgrun) + r) << E.lguw, E.uw | (c << 6));
            }
        }
    };
    uint32_t mine = 0, all;
    items([&](uint32_t, uint32_t) { ++mine; });
    uint32_t u = block_excl_scan(mine, wsum, all);
    if (threadIdx.x == 0 && all) ubase = atomicAdd(E.nunits, all);
    __syncthreads();
    u += ubase;
    items([&](uint32_t k, uint32_t w) { E.units[u++] = make_uint2(k, w); });
}

// ------------------------------------------------- K4: scatter
// sortByCountingCUDA (pbf_counting_sort.cu:120-134): slot = off[key] + rank.
// The rank-0 particle of a cell above kSmallCell particles lists the cell
// for k_sort_cells.
// n_dev (a batch's device-resident input count, or NULL) bounds the inputs.
// clear: counts and tile flags the scan left (a scan without tile totals).
struct ClearArgs {
    uint32_t *count, *tflag;  // NULL: nothing to clear
    uint32_t nc, nt;
};
__device__ __forceinline__ void clear_counts(const ClearArgs& a) {
    if (!a.count) return;
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x, nt = gridDim.x * blockDim.x;
    for (uint32_t i = t; i < a.nc; i += nt) a.count[i] = 0;
    for (uint32_t i = t; i < a.nt; i += nt) a.tflag[i] = 0;
}

__global__ __launch_bounds__(256) void k_clear_counts(ClearArgs search, ClearArgs final) {
    clear_counts(search);
    clear_counts(final);
}

__global__ __launch_bounds__(256) void k_scatter(const uint32_t* __restrict__ key, const uint32_t* __restrict__ rank,
                                                 const uint32_t* __restrict__ offset, uint32_t* __restrict__ tmp,
                                                 uint32_t n, const uint32_t* __restrict__ n_dev,
                                                 uint32_t* __restrict__ big, uint32_t* __restrict__ nbig,
                                                 uint32_t cap, uint32_t* __restrict__ bslot, ClearArgs clear) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    clear_counts(clear);
    if (i >= (n_dev ? min(n, *n_dev) : n)) return;
    const uint32_t k = key[i], r = rank[i], o0 = offset[k];
    tmp[o0 + r] = i;
    if (r == 0u) list_big_cell(offset, k, o0, big, nbig, cap, bslot);
}

// ------------------------------------------------- K4b: large cells in stable order
// Ascending bitonic sort of src[0..len) (len <= kSortMax, distinct values)
// into dst[0..len), by the whole workgroup (dst may be src: all of src is read
// before the first write).  Exchanges over less than 64 places stay in a wave's
// registers; wider ones go through LDS, a barrier each (28 of the 91 rounds of
// 8,192 values; with all of them through LDS k_sort_cells took 162 us a launch over the
// first ten chained steps of the wild 1M dam and 15.7 over 40 of the 32k dam, now 75
// and 7.8).  Contains barriers: call uniformly.
__device__ void lds_sort_segment(const uint32_t* src, uint32_t* dst, uint32_t len, uint32_t* __restrict__ buf) {
    uint32_t P = 64u;
    while (P < len) P <<= 1;
    // the rounds of k over j = from, from / 2 .. 1 (from < 64) on the value at place i
    auto in_wave = [](uint32_t v, uint32_t i, uint32_t k, uint32_t from) {
        for (uint32_t j = from; j > 0u; j >>= 1) {
            const uint32_t o = (uint32_t)__shfl_xor((int)v, (int)j, 64);
            v = ((i & j) == 0u) == ((i & k) == 0u) ? min(v, o) : max(v, o);
        }
        return v;
    };
    for (uint32_t i = threadIdx.x; i < P; i += blockDim.x) {
        uint32_t v = i < len ? src[i] : 0xFFFFFFFFu;
        for (uint32_t k = 2u; k <= 64u; k <<= 1) v = in_wave(v, i, k, k >> 1);
        buf[i] = v;
    }
    __syncthreads();
    for (uint32_t k = 128u; k <= P; k <<= 1) {
        for (uint32_t j = k >> 1; j >= 64u; j >>= 1) {
            for (uint32_t t = threadIdx.x; t < P / 2u; t += blockDim.x) {
                const uint32_t i = ((t & ~(j - 1u)) << 1) | (t & (j - 1u));
                const uint32_t a = buf[i], b = buf[i + j];
                if ((a > b) == ((i & k) == 0u)) {
                    buf[i] = b;
                    buf[i + j] = a;
                }
            }
            __syncthreads();
        }
        for (uint32_t i = threadIdx.x; i < P; i += blockDim.x) buf[i] = in_wave(buf[i], i, k, 32u);
        __syncthreads();
    }
    for (uint32_t i = threadIdx.x; i < len; i += blockDim.x) dst[i] = buf[i];
    __syncthreads();
}

// The segment of each listed cell (all indices distinct) in ascending order,
// so that the stable in-cell order is the segment's own order.  Cells of at
// most kSortMax (cells[0 .. ncells[0])) are sorted in place by one workgroup
// each; the segment of a larger cell (cells[huge_base(cap) ..] + ncells[1])
// is cut into chunks of kSortMax, each sorted by one workgroup into the same
// range of `scratch`, for k_merge_huge.
__global__ __launch_bounds__(1024) void k_sort_cells(const uint32_t* __restrict__ offset,
                                                     const uint32_t* __restrict__ cells,
                                                     const uint32_t* __restrict__ ncells, uint32_t* __restrict__ vals,
                                                     uint32_t* __restrict__ scratch, uint32_t cap) {
    __shared__ uint32_t buf[kSortMax];
    const uint32_t nc = ncells[0];
    for (uint32_t w = blockIdx.x; w < nc; w += gridDim.x) {
        const uint32_t c = cells[w];
        const uint32_t o0 = offset[c];
        lds_sort_segment(vals + o0, vals + o0, offset[c + 1] - o0, buf);
    }
    const uint32_t nh = ncells[1];
    const uint32_t* __restrict__ huge = cells + huge_base(cap);
    uint32_t w = blockIdx.x;  // chunk index over all huge cells, in list order
    for (uint32_t h = 0; h < nh; ++h) {
        const uint32_t c = huge[h];
        const uint32_t o0 = offset[c], len = offset[c + 1] - o0;
        const uint32_t nch = (len + kSortMax - 1u) / kSortMax;
        for (; w < nch; w += gridDim.x) {
            const uint32_t q0 = w * kSortMax;
            lds_sort_segment(vals + o0 + q0, scratch + o0 + q0, min(kSortMax, len - q0), buf);
        }
        w -= nch;
    }
}

// Merges the sorted chunks of every huge cell: the element at position p of
// chunk q lands at p + (the number of smaller elements in every other
// chunk), found by binary search.  Reads scratch, writes vals.
__global__ __launch_bounds__(256) void k_merge_huge(const uint32_t* __restrict__ offset,
                                                    const uint32_t* __restrict__ cells,
                                                    const uint32_t* __restrict__ ncells, uint32_t* __restrict__ vals,
                                                    const uint32_t* __restrict__ scratch, uint32_t cap) {
    const uint32_t nh = ncells[1];
    const uint32_t* __restrict__ huge = cells + huge_base(cap);
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t h = 0; h < nh; ++h) {
        const uint32_t c = huge[h];
        const uint32_t o0 = offset[c], len = offset[c + 1] - o0;
        const uint32_t* __restrict__ seg = scratch + o0;
        const uint32_t nch = (len + kSortMax - 1u) / kSortMax;
        for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < len; p += stride) {
            const uint32_t x = seg[p], q = p / kSortMax;
            uint32_t r = p - q * kSortMax;
            for (uint32_t o = 0; o < nch; ++o) {
                if (o == q) continue;
                uint32_t lo = o * kSortMax, hi = min(lo + kSortMax, len);  // first element >= x
                while (lo < hi) {
                    const uint32_t mid = (lo + hi) >> 1;
                    if (seg[mid] < x) lo = mid + 1u;
                    else hi = mid;
                }
                r += lo - o * kSortMax;
            }
            vals[o0 + r] = x;
        }
    }
}

// ------------------------------------------------- K5: stable reorder
// Makes the in-cell order ascending by original index (the stable order of
// the reference's radix-sort paths, pbf_neighbor_search.cpp:112-131), gathers
// x* (as float4) and x (SoA) (reorderDataCUDA, pbf_neighbor_search_util.cu:143-154).
template <bool kB>
__global__ __launch_bounds__(256) void k_reorder(const float* __restrict__ x, const float* __restrict__ v, Bufs b, Scenes<kB> SC,
                                                 const uint32_t* __restrict__ key, const uint32_t* __restrict__ tmp,
                                                 uint32_t n) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    const bool active = s < (kB ? min(n, b.in_off[b.nscenes]) : n);
    const uint32_t i = active ? tmp[s] : 0u;
    const uint32_t si = (kB && active) ? b.isid[i] : 0u;
    by_scene<kB>(si, active, [&](uint32_t sc) {
        const uint32_t k = key[i];
        const uint32_t o0 = b.offset[k], o1 = b.offset[k + 1];
        uint32_t f = s;  // a sorted cell (k_sort_cells, k_merge_huge): the rank is the position
        if (!sorted_cell(o1 - o0)) {
            uint32_t r = 0;
            for (uint32_t t = o0; t < o1; ++t) r += (tmp[t] < i) ? 1u : 0u;
            f = o0 + r;
        }
        b.sidx[f] = i;
        b.rank[f] = 0u;  // the histogram ranks are dead: the slot's big-cell group mark (k_big_seg)
        if (kB) b.sid[f] = sc;
        const Phys& P = SC[sc].P;
        const float dt = P.dt;
        // one 12-byte load each for the gathered x and v
        const F3 xi = reinterpret_cast<const F3*>(x)[i], vi = reinterpret_cast<const F3*>(v)[i];
        const float xo[3] = {xi.x, xi.y, xi.z}, vv[3] = {vi.x, vi.y, vi.z};
        float q[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            float vs = __builtin_fmaf(P.g[c], dt, vv[c]);
            q[c] = __builtin_fmaf(vs, dt, xo[c]);
        }
        b.Pf[f] = make_float4(q[0], q[1], q[2], __uint_as_float(k));
        st3(b.X, b.cap, f, mk3(xo[0], xo[1], xo[2]));
    });
}

// ------------------------------------------------- K5b: groups of big cells
// Image of a position in the wrapped grid, as a group code:
// (ix+2) | (iy+2) << 2 | (iz+2) << 4 for the images ix = floor(cx / gx) of
// the unwrapped cell coordinate cx (the hash's, grid_pos) in [-2, 1] on each
// axis; kCodeOther for non-finite positions and farther images.  The code
// only groups particles; the boxes decide every skip.
__device__ __forceinline__ uint32_t image_code(F3 p, const Grid& G) {
    if (!(__builtin_isfinite(p.x) && __builtin_isfinite(p.y) && __builtin_isfinite(p.z))) return kCodeOther;
    int gp[3];
    grid_pos(p, G.cw, gp);
    const int ix = gp[0] >> (int)G.lgx, iy = gp[1] >> (int)G.lgy, iz = gp[2] >> (31 - __builtin_clz(G.gz));
    if (ix < -2 || ix > 1 || iy < -2 || iy > 1 || iz < -2 || iz > 1) return kCodeOther;
    return (uint32_t)(ix + 2) | ((uint32_t)(iy + 2) << 2) | ((uint32_t)(iz + 2) << 4);
}

// Running box of positions; `bad` once a non-finite one was seen (its group
// is then never skipped).
struct Box3 {
    F3 lo, hi;
    bool bad;
};
__device__ __forceinline__ Box3 box_empty() {
    const float inf = __builtin_huge_valf();
    return Box3{mk3(inf, inf, inf), mk3(-inf, -inf, -inf), false};
}
__device__ __forceinline__ void box_add(Box3& B, F3 p) {
    if (!(__builtin_isfinite(p.x) && __builtin_isfinite(p.y) && __builtin_isfinite(p.z))) B.bad = true;
    B.lo = mk3(fminf(B.lo.x, p.x), fminf(B.lo.y, p.y), fminf(B.lo.z, p.z));
    B.hi = mk3(fmaxf(B.hi.x, p.x), fmaxf(B.hi.y, p.y), fmaxf(B.hi.z, p.z));
}

// The box over the whole block (every thread calls it); valid in thread 0.
__device__ Box3 block_box(Box3 B, float (*red)[8]) {
    const uint32_t lane = lane_id(), wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        B.lo = mk3(fminf(B.lo.x, __shfl_xor(B.lo.x, d, 64)), fminf(B.lo.y, __shfl_xor(B.lo.y, d, 64)),
                   fminf(B.lo.z, __shfl_xor(B.lo.z, d, 64)));
        B.hi = mk3(fmaxf(B.hi.x, __shfl_xor(B.hi.x, d, 64)), fmaxf(B.hi.y, __shfl_xor(B.hi.y, d, 64)),
                   fmaxf(B.hi.z, __shfl_xor(B.hi.z, d, 64)));
    }
    B.bad = __any(B.bad);
    if (lane == 0) {
        red[wid][0] = B.lo.x;
        red[wid][1] = B.lo.y;
        red[wid][2] = B.lo.z;
        red[wid][3] = B.hi.x;
        red[wid][4] = B.hi.y;
        red[wid][5] = B.hi.z;
        red[wid][6] = B.bad ? 1.f : 0.f;
    }
    __syncthreads();
    if (threadIdx.x == 0)
        for (uint32_t w = 1; w < nw; ++w) {
            B.lo = mk3(fminf(B.lo.x, red[w][0]), fminf(B.lo.y, red[w][1]), fminf(B.lo.z, red[w][2]));
            B.hi = mk3(fmaxf(B.hi.x, red[w][3]), fmaxf(B.hi.y, red[w][4]), fmaxf(B.hi.z, red[w][5]));
            B.bad = B.bad || red[w][6] != 0.f;
        }
    __syncthreads();
    return B;
}

// The box as stored: a group with a non-finite member spans everything.
__device__ __forceinline__ void box_store(const Box3& B, float4& lo, float4& hi) {
    const float inf = __builtin_huge_valf();
    lo = B.bad ? make_float4(-inf, -inf, -inf, 0.f) : make_float4(B.lo.x, B.lo.y, B.lo.z, 0.f);
    hi = B.bad ? make_float4(inf, inf, inf, 0.f) : make_float4(B.hi.x, B.hi.y, B.hi.z, 0.f);
}

// Order-preserving key of a float (a < b  =>  fkey(a) <= fkey(b), -0 below
// +0), so that boxes gather with integer atomics; funkey inverts it.
__device__ __forceinline__ uint32_t fkey(float f) {
    const uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float funkey(uint32_t k) { return __uint_as_float((k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k); }

// Group mark of a big cell's member: descriptor d, group k (0 marks the
// slots of other cells).
__device__ __forceinline__ uint32_t big_mark(uint32_t d, uint32_t k) { return d * kMaxSeg + k + 1u; }

// Adds the final x* of the lanes' marked slots to their groups' final boxes.
// Lanes of one group merge over the wave first and one of them issues the
// atomics.  Called by every lane of the wave (bm = 0 where nothing is added).
__device__ void big_box_add(BigSeg* __restrict__ bseg, uint32_t bm, F3 p) {
    const uint32_t lane = lane_id();
    const bool bad = !(__builtin_isfinite(p.x) && __builtin_isfinite(p.y) && __builtin_isfinite(p.z));
    const uint32_t k[3] = {fkey(p.x), fkey(p.y), fkey(p.z)};
    uint64_t todo = __ballot(bm != 0u);
    while (todo) {
        const int l = __ffsll((unsigned long long)todo) - 1;
        const uint32_t key = (uint32_t)__shfl((int)bm, l, 64);
        const bool mine = bm == key;
        uint32_t lo[3], hi[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            lo[c] = mine ? k[c] : 0xFFFFFFFFu;
            hi[c] = mine ? k[c] : 0u;
        }
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                lo[c] = min(lo[c], (uint32_t)__shfl_xor((int)lo[c], d, 64));
                hi[c] = max(hi[c], (uint32_t)__shfl_xor((int)hi[c], d, 64));
            }
        const bool anybad = __any(mine && bad);
        if (lane == (uint32_t)l) {
            BigSeg& D = bseg[(key - 1u) / kMaxSeg];
            const uint32_t g = (key - 1u) % kMaxSeg;
            atomicMin(&D.fmin[g].x, lo[0]);
            atomicMin(&D.fmin[g].y, lo[1]);
            atomicMin(&D.fmin[g].z, lo[2]);
            atomicMax(&D.fmax[g].x, hi[0]);
            atomicMax(&D.fmax[g].y, hi[1]);
            atomicMax(&D.fmax[g].z, hi[2]);
            if (anybad) atomicOr(&D.fmin[g].w, 1u);
        }
        todo &= ~__ballot(mine);
    }
}

// Big cell of work item `it` (huge cells first: they take longest): its
// descriptor index d and key c.
__device__ __forceinline__ uint32_t big_item(const Bufs& b, uint32_t it, uint32_t nh, uint32_t& c) {
    const uint32_t d = it < nh ? huge_base(b.cap) + it : it - nh;
    c = b.big[d];
    return d;
}

// Groups the slots of every big cell by image code: a stable partition into
// aux (ascending slots inside each group, the groups in code order), the
// groups' ends and the boxes of their x* (after k_reorder, before the
// search).  One workgroup per cell; a cell of one group keeps aux unused.
template <bool kB>
__global__ __launch_bounds__(1024) void k_big_seg(Bufs b, Scenes<kB> SC) {
    __shared__ uint32_t cnt[kCodes];
    __shared__ uint32_t segof[kCodes];       // group of each code (kMaxSeg: none)
    __shared__ uint32_t sbeg[kMaxSeg + 1];   // first aux position of each group, then the cell's size
    __shared__ uint32_t put[kMaxSeg];        // where each group's next chunk goes
    __shared__ uint32_t wcnt[16][kMaxSeg];   // members of each group per wave in a chunk
    __shared__ uint32_t nseg_s;
    __shared__ float red[16][8];
    const uint32_t lane = lane_id(), wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const uint32_t nb0 = b.ctr[CTR_BIGCELLS], nh = b.ctr[CTR_HUGECELLS];
    uint32_t most = 0;
    for (uint32_t it = blockIdx.x; it < nh + nb0; it += gridDim.x) {
        uint32_t c;
        const uint32_t d = big_item(b, it, nh, c);
        const uint32_t o0 = b.offset[c], n = b.offset[c + 1] - o0;
        most = max(most, n);
        const Grid G = SC[scene_index<kB>(b.kbase, b.nscenes, c)].G;
        for (uint32_t k = threadIdx.x; k < kCodes; k += blockDim.x) cnt[k] = 0u;
        __syncthreads();
        for (uint32_t p = threadIdx.x; p < n; p += blockDim.x) atomicAdd(&cnt[image_code(f3of(b.Pf[o0 + p]), G)], 1u);
        __syncthreads();
        if (threadIdx.x == 0) {
            uint32_t ns = 0, run = 0;
            for (uint32_t k = 0; k < kCodes; ++k) {
                segof[k] = kMaxSeg;
                if (cnt[k]) {
                    if (ns < kMaxSeg) {
                        segof[k] = ns;
                        sbeg[ns] = run;
                        put[ns] = run;
                    }
                    ++ns;
                    run += cnt[k];
                }
            }
            nseg_s = ns <= kMaxSeg ? ns : 0u;
            if (ns <= kMaxSeg) sbeg[ns] = n;
        }
        __syncthreads();
        const uint32_t ns = nseg_s;
        if (ns >= 2u) {
            for (uint32_t q0 = 0; q0 < n; q0 += blockDim.x) {
                const uint32_t p = q0 + threadIdx.x;
                const uint32_t sg = p < n ? segof[image_code(f3of(b.Pf[o0 + p]), G)] : kMaxSeg;
                uint32_t lrank = 0;
                for (uint32_t k = 0; k < ns; ++k) {
                    const uint64_t m = __ballot(sg == k);
                    if (sg == k) lrank = (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
                    if (lane == 0) wcnt[wid][k] = (uint32_t)__popcll(m);
                }
                __syncthreads();
                if (sg < kMaxSeg) {
                    uint32_t o = put[sg] + lrank;
                    for (uint32_t w = 0; w < wid; ++w) o += wcnt[w][sg];
                    b.aux[o0 + o] = o0 + p;
                    b.rank[o0 + p] = big_mark(d, sg);
                }
                __syncthreads();
                if (threadIdx.x < ns) {
                    uint32_t t = 0;
                    for (uint32_t w = 0; w < nw; ++w) t += wcnt[w][threadIdx.x];
                    put[threadIdx.x] += t;
                }
                __syncthreads();
            }
        }
        BigSeg& D = b.bseg[d];
        if (ns == 1u)
            for (uint32_t p = threadIdx.x; p < n; p += blockDim.x) b.rank[o0 + p] = big_mark(d, 0u);
        for (uint32_t k = 0; k < ns; ++k) {
            const uint32_t p0 = sbeg[k], p1 = sbeg[k + 1];
            Box3 B = box_empty();
            for (uint32_t p = p0 + threadIdx.x; p < p1; p += blockDim.x)
                box_add(B, f3of(b.Pf[ns == 1u ? o0 + p : b.aux[o0 + p]]));
            B = block_box(B, red);
            if (threadIdx.x == 0) {
                box_store(B, D.slo[k], D.shi[k]);
                D.end[k] = p1;
                // the final box, gathered by k_cur_hash
                D.fmin[k] = make_uint4(0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu, 0u);
                D.fmax[k] = make_uint4(0u, 0u, 0u, 0u);
            }
        }
        if (threadIdx.x == 0) D.nseg = ns;
        __syncthreads();
    }
    if (threadIdx.x == 0 && most) atomicMax(&b.ctr[kCtrMostCell], most);
}

// What a scan of big cell D (n particles) for a particle at `self` must
// visit.  kFinal: the final positions, whose pair test passes
// !(glm_dot(d, d) > thr); otherwise the search's, which passes
// fmaf-dot(d, d) < thr.  Every component of a member's difference to self
// lies, in magnitude, between the rounded gap from self to the group's box
// and the rounded distance to the box's far side (rounding is monotone), and
// both dot products are monotone in the components' magnitudes: a group
// whose gap fails the test holds no pair, and one whose far corner passes it
// holds only pairs.  A non-finite self skips nothing.
struct BigPart {
    uint32_t how;     // 0: no member passes; 1: visit the whole cell; 2: visit aux positions [p0, p1) only
    uint32_t p0, p1;  // the one group that may pass (how 2, or how 1 with a single group: the whole cell)
    bool all_in;      // every member of that group passes
    uint32_t inside;  // members of the cell's groups whose every member passes
};
__device__ __forceinline__ float box_gap(float x, float lo, float hi) {
    return (x < lo) ? (lo - x) : ((x > hi) ? (x - hi) : 0.f);
}
__device__ __forceinline__ float box_far(float x, float lo, float hi) { return fmaxf(x - lo, hi - x); }
template <bool kFinal>
__device__ __forceinline__ bool pair_test(F3 d, float thr) {
    return kFinal ? !(glm_dot(d, d) > thr) : (__builtin_fmaf(d.z, d.z, __builtin_fmaf(d.y, d.y, d.x * d.x)) < thr);
}
template <bool kFinal>
__device__ __forceinline__ BigPart big_part(const BigSeg* __restrict__ D, F3 self, float thr, uint32_t n) {
    BigPart r{1u, 0u, n, false, 0u};
    const uint32_t ns = D->nseg;
    if (ns == 0u) return r;
    uint32_t hits = 0, beg = 0, p0 = 0, p1 = 0;
    bool in0 = false;
    for (uint32_t k = 0; k < ns; ++k) {
        const uint32_t end = D->end[k];
        float4 lo, hi;
        if (kFinal) {
            const uint4 a = D->fmin[k], z = D->fmax[k];
            const float inf = __builtin_huge_valf();
            lo = a.w ? make_float4(-inf, -inf, -inf, 0.f) : make_float4(funkey(a.x), funkey(a.y), funkey(a.z), 0.f);
            hi = a.w ? make_float4(inf, inf, inf, 0.f) : make_float4(funkey(z.x), funkey(z.y), funkey(z.z), 0.f);
        } else {
            lo = D->slo[k];
            hi = D->shi[k];
        }
        const F3 g = mk3(box_gap(self.x, lo.x, hi.x), box_gap(self.y, lo.y, hi.y), box_gap(self.z, lo.z, hi.z));
        const F3 f = mk3(box_far(self.x, lo.x, hi.x), box_far(self.y, lo.y, hi.y), box_far(self.z, lo.z, hi.z));
        const bool in = pair_test<kFinal>(f, thr);
        if (pair_test<kFinal>(g, thr)) {
            if (hits == 0u) {
                p0 = beg;
                p1 = end;
                in0 = in;
            }
            ++hits;
        }
        if (in) r.inside += end - beg;
        beg = end;
    }
    if (hits == 0u) {
        r.how = 0u;
    } else if (hits == 1u) {
        r.how = ns == 1u ? 1u : 2u;
        r.p0 = p0;
        r.p1 = p1;
        r.all_in = in0;
    }
    return r;
}

// What the global-memory scans read of a step's cells: the cell offsets and
// the big cells' descriptors (passed by value, so that no kernel argument
// block is copied to scratch memory for its address).
struct CellView {
    const uint32_t* __restrict__ offset;
    const uint32_t* __restrict__ bslot;
    const uint32_t* __restrict__ aux;
    const BigSeg* __restrict__ bseg;
};
__device__ __forceinline__ CellView cell_view(const Bufs& b) { return CellView{b.offset, b.bslot, b.aux, b.bseg}; }

// Whether this step has cells of more than kSmallCell particles (a
// grid-uniform value: the scans without them keep their plain loops).
__device__ __forceinline__ bool big_cells(const Bufs& b) { return (b.ctr[CTR_BIGCELLS] | b.ctr[CTR_HUGECELLS]) != 0u; }

// Whether visiting one group through aux beats scanning the whole cell (the
// indirection costs a load per candidate): when it skips a quarter or more.
__device__ __forceinline__ bool aux_pays(const BigPart& bp, uint32_t n) {
    return bp.how == 2u && 4u * (bp.p1 - bp.p0) <= 3u * n;
}


// Per-thread event tallies, summed per wave and added once at kernel end.
struct Tally {
    uint32_t trunc = 0, slowpart = 0, slowunits = 0, maxtile = 0, sweepcap = 0, maxsweep = 0,
             nan = 0, listovf = 0;
};

__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
    return v;
}
__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v = max(v, (uint32_t)__shfl_xor(v, d, 64));
    return v;
}

// Called by every thread of the block at kernel end.
// Statistics go to one of kStatRep copies of the counters (by workgroup), so
// that waves of a large grid do not all update the same words; the host
// reduces the copies.
__device__ void flush_tally(uint32_t* __restrict__ ctr_base, const Tally& t) {
    uint32_t* ctr = ctr_base + CTR_NUM * (1u + (blockIdx.x & (kStatRep - 1u)));
    const uint32_t tr = wave_sum(t.trunc), sp = wave_sum(t.slowpart), su = wave_sum(t.slowunits),
                   mt = wave_max(t.maxtile), sc = wave_sum(t.sweepcap),
                   ms = wave_max(t.maxsweep), nn = wave_sum(t.nan), lo = wave_sum(t.listovf);
    if (lane_id() == 0) {
        if (tr) atomicAdd(&ctr[CTR_TRUNC], tr);
        if (sp) atomicAdd(&ctr[CTR_SLOWPART], sp);
        if (su) atomicAdd(&ctr[CTR_SLOWUNITS], su);
        if (mt && mt > ctr[CTR_MAXTILE]) atomicMax(&ctr[CTR_MAXTILE], mt);  // a stale read only costs an atomic
        if (sc) atomicAdd(&ctr[CTR_SWEEPCAP], sc);
        if (ms && ms > ctr[CTR_MAXSWEEP]) atomicMax(&ctr[CTR_MAXSWEEP], ms);
        if (nn) atomicAdd(&ctr[CTR_XSPHNAN], nn);
        if (lo) atomicAdd(&ctr[CTR_LISTOVF], lo);
    }
}

constexpr uint32_t kDeferred = 0xFFFFFFFFu;  // a group's count when it left its list to a wave

// ------------------------------------------------- lists by groups of eight
// Key of cell c (0..26, in z,y,x order) of the 27 around the cell of key `key`.
__device__ __forceinline__ uint32_t key27(uint32_t key, uint32_t c, const Grid& G) {
    const uint32_t k = key - G.base, dz = c / 9u, q = c % 9u;
    const uint32_t x = (k + q % 3u - 1u) & (G.gx - 1u), y = ((k >> G.lgx) + q / 3u - 1u) & (G.gy - 1u),
                   z = ((k >> (G.lgx + G.lgy)) + dz - 1u) & (G.gz - 1u);
    return G.base + (((z << G.lgy) + y) << G.lgx) + x;
}

constexpr uint32_t kGroup = 8;
constexpr uint32_t kGroups = kBlock / kGroup;  // groups of a workgroup
constexpr uint32_t kMaxPair = 64;              // the largest max_pair accepted
constexpr uint32_t kGroupList = 96;            // entries held on chip: the longest list kept, and a row's hits past it
static_assert(kGroupList >= kFinalK + 4u * kGroup && kGroupList >= kMaxPair - 1u + 4u * kGroup,
              "room for the hits past a full list");
// A group's cells (first slot and particles of each of the 27) and its list.
struct GroupShared {
    uint2 cell[kGroups][27];
    uint4 list[kGroups][kGroupList / 4];
};

// The list of one particle (slot `slot`, in the cell of key `key`), at list
// position i, built by a group of eight lanes from global memory: the 27 cells
// around its cell in z,y,x order, slots ascending, eight candidates x*_j = Pf[j]
// at a time (a cell of the lattice is one step).  A ballot ranks a step's hits,
// which go to the list on chip; the list is written out whole at the end, 16
// bytes a lane.  A row's three cells are tested together, and the next row's
// candidates are loaded before their hits are ranked.
//   search (kFinal false): pairs by pair_test<false>, the first lim kept; the
//     return value exceeds lim when there are more.
//   final (kFinal true): pairs by pair_test<true>, the first pair of each cell
//     marked by bit 31; past lim pairs the list overflows (returns more than
//     lim) and is not written.
// kBig (the step has cells of more than kSmallCell particles): in a big cell
// groups out of range are skipped, a group wholly in range is listed without
// tests (the final lists stop at once when such groups alone take them past
// lim), and a single group left is scanned through aux when that skips a
// quarter of the cell or more.  Returns kDeferred, leaving the list unfinished,
// before a range that would take the candidates tested past `budget` (only a
// neighbourhood holding a big cell can: 27 * kSmallCell is less).
// kWide: more than 2^28 slots, whose records' byte offsets pass 32 bits.
// Called by all eight lanes; every value but the candidates is the same on them.
//
// Bound by VALU issue at large sizes (0.95 of one wave64 instruction per SIMD
// every 4 cycles, about 95 instructions a particle; 177 us for the search and
// 184 us for the final lists of the 1M dam) and by the latency of nine dependent
// rows at small ones (4 us).  A thread per particle walks a serial chain of 54
// groups of four candidates instead, whose latency set the time: from tiles of
// cells staged in LDS 202 and 340 us on the 1M dam, 27 and 33 us for 960
// particles, and 576 us a launch for the final lists beside the piles of the
// chained 32k dam (now 40).  Taking a row's 24 particles as one range (fewer
// partial steps in the lattice) measured slower wherever cells hold more than
// eight or a row wraps: 521 against 247 us at 16 particles a cell (1M).
template <bool kFinal, bool kBig, bool kWide>
__device__ __forceinline__ uint32_t group_list(GroupShared& S, const Grid& G, CellView b,
                                               const float4* __restrict__ Pf, F3 self, uint32_t key, float thr,
                                               uint32_t lim, uint32_t* __restrict__ lst, uint32_t cap, uint32_t i,
                                               uint32_t slot, uint32_t budget) {
    const uint32_t lane = lane_id(), l = lane & (kGroup - 1u), sh = lane & 56u;
    uint2* __restrict__ cells = S.cell[threadIdx.x / kGroup];
    uint32_t* __restrict__ keep = reinterpret_cast<uint32_t*>(S.list[threadIdx.x / kGroup]);
    {
        // lane l finds the cells of row l (dz outer, dy inner), and lane 0 those of row 8
        const uint32_t k0 = key - G.base;
        const uint32_t x = k0 & (G.gx - 1u), y = (k0 >> G.lgx) & (G.gy - 1u), z = k0 >> (G.lgx + G.lgy);
        auto find_row = [&](uint32_t r) {
            const uint32_t dz = r / 3u, dy = r - 3u * dz;
            const uint32_t row = G.base + (((((z + dz - 1u) & (G.gz - 1u)) << G.lgy) + ((y + dy - 1u) & (G.gy - 1u))) << G.lgx);
#pragma unroll
            for (uint32_t dx = 0; dx < 3u; ++dx) {
                const uint32_t k = row + ((x + dx - 1u) & (G.gx - 1u));
                const uint32_t o = b.offset[k];
                cells[3u * r + dx] = make_uint2(o, b.offset[k + 1] - o);
            }
        };
        find_row(l);
        if (l == 0u) find_row(8u);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the group's own lanes wrote what it reads
    // A lane past its row's end loads some other record, which is not looked at.
    const Gather16 buf(Pf, cap);
    auto load = [&](uint32_t j) { return f3of(kWide ? Pf[min(j, cap - 1u)] : buf(j)); };
    auto test = [&](F3 pj) { return pair_test<kFinal>(kFinal ? pj - self : self - pj, thr); };
    uint32_t n = 0;
    const uint32_t under = (1u << l) - 1u;
    // a step's hits, this group's byte of the wave's
    auto byte_of = [&](bool in, bool ok) {
        return (uint32_t)((__builtin_amdgcn_ballot_w64(in) & __builtin_amdgcn_ballot_w64(ok)) >> sh) & 0xFFu;
    };
    // Appends a step's hits in lane order; first: none of this cell's came before.
    auto append = [&](uint32_t bits, bool hit, uint32_t j, bool first) {
        if (hit) {
            const uint32_t k = (uint32_t)__builtin_popcount(bits & under);
            // k - 1 has bit 31 set when no lane below hits
            (keep + n)[k] = (kFinal && first) ? (((k - 1u) & 0x80000000u) | j) : j;
        }
        n += (uint32_t)__builtin_popcount(bits);
    };
    uint2 c[3];
    F3 p[3], q[3];  // the cells' first and second steps
    bool two;       // some group's row has a cell of more than one step
    auto fetch = [&](uint32_t r) {
#pragma unroll
        for (uint32_t d = 0; d < 3u; ++d) c[d] = cells[3u * r + d];
#pragma unroll
        for (uint32_t d = 0; d < 3u; ++d) p[d] = load(c[d].x + l);
        two = __builtin_amdgcn_ballot_w64(max(max(c[0].y, c[1].y), c[2].y) > kGroup) != 0ull;
        if (two) {
#pragma unroll
            for (uint32_t d = 0; d < 3u; ++d) q[d] = load(c[d].x + l + kGroup);
        }
    };
    q[0] = q[1] = q[2] = self;
    fetch(0u);
    for (uint32_t r = 0; r < 9u; ++r) {
        const uint2 C[3] = {c[0], c[1], c[2]};
        const uint32_t most = max(max(C[0].y, C[1].y), C[2].y);
        uint32_t m[3], m2[3] = {0u, 0u, 0u};
        bool h[3], h2[3] = {false, false, false};
#pragma unroll
        for (uint32_t d = 0; d < 3u; ++d) {
            const bool in = l < C[d].y, ok = test(p[d]);
            m[d] = byte_of(in, ok);
            h[d] = in && ok;
        }
        const bool second = two;
        if (second) {
#pragma unroll
            for (uint32_t d = 0; d < 3u; ++d) {
                const bool in = l + kGroup < C[d].y, ok = test(q[d]);
                m2[d] = byte_of(in, ok);
                h2[d] = in && ok;
            }
        }
        if (r < 8u) fetch(r + 1u);
        if (!second) {  // every cell of every group's row is one step
            if (kBig) {
                const uint32_t all = C[0].y + C[1].y + C[2].y;
                if (all > budget) return kDeferred;
                budget -= all;
            }
#pragma unroll
            for (uint32_t d = 0; d < 3u; ++d) append(m[d], h[d], C[d].x + l, true);
        } else if (!kBig || most <= kSmallCell) {
            if (kBig) {
                const uint32_t all = C[0].y + C[1].y + C[2].y;
                if (all > budget) return kDeferred;
                budget -= all;
            }
#pragma unroll
            for (uint32_t d = 0; d < 3u; ++d) {
                const uint32_t n0 = n;
                append(m[d], h[d], C[d].x + l, true);
                if (n <= lim) append(m2[d], h2[d], C[d].x + l + kGroup, n == n0);
                for (uint32_t t = 2u * kGroup; t < C[d].y && n <= lim; t += kGroup) {
                    const bool in = t + l < C[d].y, ok = test(load(C[d].x + t + l));
                    const uint32_t bits = byte_of(in, ok);
                    append(bits, in && ok, C[d].x + t + l, n == n0);
                }
            }
        } else {
#pragma unroll 1
            for (uint32_t d = 0; d < 3u; ++d) {
                const uint32_t o0 = d == 0u ? C[0].x : (d == 1u ? C[1].x : C[2].x);
                const uint32_t ncell = d == 0u ? C[0].y : (d == 1u ? C[1].y : C[2].y);
                uint32_t p0 = 0, p1 = ncell;
                bool via = false;
                if (ncell > kSmallCell) {
                    const BigPart bp = big_part<kFinal>(b.bseg + b.bslot[o0], self, thr, ncell);
                    if (bp.how == 0u) continue;
                    if (kFinal && n + bp.inside > lim) return lim + 1u;
                    if (bp.all_in) {  // every member of the group is a pair: its first slots, ascending
                        const uint32_t size = bp.p1 - bp.p0;
                        for (uint32_t t = l; t < size && n + t < lim; t += kGroup) {
                            const uint32_t j = bp.how == 2u ? b.aux[o0 + bp.p0 + t] : o0 + bp.p0 + t;
                            keep[n + t] = (kFinal && t == 0u) ? (j | 0x80000000u) : j;
                        }
                        n += size;
                        if (n > lim) break;
                        continue;
                    }
                    if (aux_pays(bp, ncell)) {
                        p0 = bp.p0;
                        p1 = bp.p1;
                        via = true;
                    }
                }
                if (p1 - p0 > budget) return kDeferred;
                budget -= p1 - p0;
                const uint32_t n0 = n;
                // 32 candidates' records loaded together
                for (uint32_t t0 = p0; t0 < p1 && n <= lim; t0 += 4u * kGroup) {
                    uint32_t j[4];
                    F3 pj[4];
#pragma unroll
                    for (uint32_t u = 0; u < 4u; ++u) {
                        const uint32_t t = t0 + l + u * kGroup;
                        j[u] = via ? b.aux[o0 + min(t, p1 - 1u)] : o0 + t;
                    }
#pragma unroll
                    for (uint32_t u = 0; u < 4u; ++u) pj[u] = load(j[u]);
#pragma unroll
                    for (uint32_t u = 0; u < 4u; ++u) {
                        const bool in = t0 + l + u * kGroup < p1, ok = test(pj[u]);
                        // few candidates beside a pile are pairs: no ranking where none of the wave's is
                        if ((__builtin_amdgcn_ballot_w64(in) & __builtin_amdgcn_ballot_w64(ok)) == 0ull) continue;
                        append(byte_of(in, ok), in && ok, j[u], n == n0);
                    }
                }
                if (n > lim) break;
            }
        }
        if (n > lim) break;
    }
    if (kFinal && n > lim) return n;
    // The rest of the last word, whose records the walks load and do not use: the
    // own one for the search, where the slots of a wave are neighbours; for the final
    // lists, whose positions' slots are scattered, slot 0, one line for all lanes (with
    // the own record there the three passes took 44 / 53 / 59 us on the 1M dam, with
    // this 39 / 43 / 53, and 655 / 858 / 869 us on the 8M double dam, now 606 / 788 / 809).
    if (l < 3u) keep[min(n, lim) + l] = kFinal ? 0u : slot;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const uint32_t nw = (min(n, lim) + 3u) / 4u;
    for (uint32_t w = l; w < nw; w += kGroup)
        reinterpret_cast<uint4*>(lst)[(size_t)w * cap + i] = S.list[threadIdx.x / kGroup][w];
    return n;
}

// The search list of slot g by its group, and its count; true when the list
// is left to a whole wave instead (kDeferred).
template <bool kBig, bool kWide>
__device__ __forceinline__ bool group_search(GroupShared& S, const Bufs& b, const Scene& sc, uint32_t g, Tally& tl) {
    const Grid G = sc.G;
    const uint32_t ncap = (uint32_t)sc.P.cap;
    const float4 pk = b.Pf[g];
    const uint32_t n = group_list<false, kBig, kWide>(S, G, cell_view(b), b.Pf, f3of(pk), __float_as_uint(pk.w),
                                                      sc.P.h2, ncap, b.nlist, b.cap, g, g, kHeavySearch);
    if (kBig && n == kDeferred) return true;
    if ((lane_id() & (kGroup - 1u)) == 0u) {
        b.ncnt[g] = min(n, ncap);
        tl.trunc += n > ncap ? 1u : 0u;
    }
    return false;
}

// Statistics of the work items, one thread each (thread t of nt): the largest
// neighbourhood, and the items whose neighbourhood passes tile_cap particles;
// big(item) for each of those.
template <bool kB, class BigF>
__device__ __forceinline__ void item_stats(const Bufs& b, const Scenes<kB>& SC, const uint2* __restrict__ units,
                                           uint32_t nU, uint32_t tile_cap, uint32_t t, uint32_t nt, Tally& tl,
                                           BigF&& big) {
    for (uint32_t u = t; u < nU; u += nt) {
        const uint2 unit = units[u];
        const Grid G = SC[scene_index<kB>(b.kbase, b.nscenes, unit.x)].G;
        const uint32_t kb = unit.x - G.base;
        const uint32_t x = (kb - 1u) & (G.gx - 1u), y = (kb >> G.lgx) & (G.gy - 1u), z = kb >> (G.lgx + G.lgy);
        uint32_t total = 0;
        for (uint32_t r = 0; r < 9u; ++r) {
            const uint32_t cy = (y + r % 3u - 1u) & (G.gy - 1u), cz = (z + r / 3u - 1u) & (G.gz - 1u);
            const uint32_t row = G.base + (((cz << G.lgy) + cy) << G.lgx);
            // W + 2 cells from x on, wrapping
            uint32_t left = (unit.y & 63u) + 2u, at = x;
            while (left) {
                const uint32_t k = min(left, G.gx - at);
                total += b.offset[row + at + k] - b.offset[row + at];
                left -= k;
                at = 0;
            }
        }
        tl.maxtile = max(tl.maxtile, total);
        if (total > tile_cap) {
            tl.slowunits++;
            big(unit);
        }
    }
}

// The search list of slot g (x* = self), built by a whole wave:
// the 27 cells around its cell in z,y,x order with the same ranges and group
// skips as group_list, 64 candidates at a time, lane l testing the
// l-th, the hits appended in slot order through a ballot; the first ncap
// are kept and trunc is set when there are more.  Called by all lanes of the
// wave; every value it depends on is the same on every lane.
template <bool kBig>
__device__ uint32_t ns_heavy_list(const Grid& G, CellView b, const float4* __restrict__ Pf, F3 self, float h2,
                                  uint32_t ncap, uint32_t* __restrict__ nl, uint32_t cap, uint32_t g, bool& trunc) {
    const uint32_t lane = lane_id();
    const uint64_t below = (1ull << lane) - 1ull;
    int gp[3];
    grid_pos(self, G.cw, gp);
    uint32_t n = 0;
    for (int c = 0; c < 27; ++c) {
        const int r = c / 3, dx = c % 3;
        const uint32_t key = scene_key(gp[0] + dx - 1, gp[1] + (r % 3) - 1, gp[2] + (r / 3) - 1, G);
        const uint32_t o0 = b.offset[key], ncell = b.offset[key + 1] - o0;
        uint32_t p0 = 0, p1 = ncell;
        bool via = false;
        if (kBig && ncell > kSmallCell) {
            const BigPart bp = big_part<false>(b.bseg + b.bslot[o0], self, h2, ncell);
            if (bp.how == 0u) continue;
            if (bp.all_in) {  // every member is a pair: the first ones, ascending
                const uint32_t size = bp.p1 - bp.p0, take = min(ncap - n, size);
                for (uint32_t t = lane; t < take; t += 64u)
                    nl[list_at(cap, g, n + t)] = bp.how == 2u ? b.aux[o0 + bp.p0 + t] : o0 + bp.p0 + t;
                n += take;
                if (size > take) {
                    trunc = true;
                    return n;
                }
                continue;
            }
            if (aux_pays(bp, ncell)) {
                p0 = bp.p0;
                p1 = bp.p1;
                via = true;
            }
        }
        for (uint32_t p = p0; p < p1; p += 256u) {
            uint32_t j[4];
            F3 pj[4];
#pragma unroll
            for (uint32_t u = 0; u < 4u; ++u) {
                const uint32_t t = min(p + u * 64u + lane, p1 - 1u);
                j[u] = via ? b.aux[o0 + t] : o0 + t;
            }
#pragma unroll
            for (uint32_t u = 0; u < 4u; ++u) pj[u] = f3of(Pf[j[u]]);
#pragma unroll
            for (uint32_t u = 0; u < 4u; ++u) {
                const bool hit = p + u * 64u + lane < p1 && pair_test<false>(self - pj[u], h2);
                const uint64_t m = __ballot(hit);
                if (m == 0ull) continue;
                const uint32_t k = n + (uint32_t)__popcll(m & below);
                if (hit && k < ncap) nl[list_at(cap, g, k)] = j[u];
                n += (uint32_t)__popcll(m);
                if (n > ncap) {
                    trunc = true;
                    return ncap;
                }
            }
        }
    }
    return n;
}

// The search lists of a step with big cells (a step without them has its lists
// from k_ns_groups): 32 slots a workgroup at a time by groups of eight lanes;
// a list of more than kHeavySearch candidates is then built by its group's whole
// wave.
template <bool kB, bool kWide>
__device__ __forceinline__ void ns_big(GroupShared& GS, const Bufs& b, const Scenes<kB>& SC, uint32_t block,
                                       uint32_t nblock, Tally& tl) {
    const uint32_t nl = b.offset[b.CT], nblk = (nl + kGroups - 1u) / kGroups;
    for (uint32_t c = block; c < nblk; c += nblock) {
        const uint32_t g = c * kGroups + threadIdx.x / kGroup;
        const bool active = g < nl;
        bool left = false;
        by_scene<kB>((kB && active) ? b.sid[g] : 0u, active,
                     [&](uint32_t sc) { left = group_search<true, kWide>(GS, b, SC[sc], g, tl); });
        uint64_t todo = __ballot(left && (lane_id() & (kGroup - 1u)) == 0u);
        if (todo && lane_id() == 0u) atomicAdd(&b.ctr[CTR_NSHEAVY], (uint32_t)__popcll(todo));
        while (todo) {
            const int src = __ffsll((unsigned long long)todo) - 1;
            todo &= todo - 1ull;
            const uint32_t gw = (uint32_t)__builtin_amdgcn_readlane((int)g, src);
            const uint32_t sc = kB ? __builtin_amdgcn_readfirstlane(b.sid[gw]) : 0u;
            const Grid G = SC[sc].G;
            const uint32_t ncap = (uint32_t)SC[sc].P.cap;
            bool trunc = false;
            const uint32_t n = ns_heavy_list<true>(G, cell_view(b), b.Pf, f3of(b.Pf[gw]), SC[sc].P.h2, ncap, b.nlist,
                                                   b.cap, gw, trunc);
            if (lane_id() == 0u) {
                b.ncnt[gw] = n;
                tl.trunc += trunc ? 1u : 0u;
            }
        }
    }
}

// ------------------------------------------------- K6: neighbour lists
// detectNeighborsCUDA (pbf_neighbor_search_util.cu:361-482): per particle the
// 27 cells in z,y,x order, slots ascending, keep r2 < h^2 while fewer than
// cap are kept; the list is frozen for all Jacobi iterations.  Stored as
// sorted slots in groups of four (list_at), with the count in
// ncnt[slot].  Every slot by a group of eight lanes (the first ngroup
// workgroups, unless the step has big cells: ns_big, in the same launch when kBig,
// else in k_ns_big's); the rest of the grid walks the work items for their
// statistics.
template <bool kB, bool kWide, bool kBig>
__global__ __launch_bounds__(kBlock) void k_ns_groups(Bufs b, Scenes<kB> SC, uint32_t tile_cap, uint32_t ngroup) {
    __shared__ GroupShared GS;
    Tally tl;
    if (blockIdx.x < ngroup) {
        if (big_cells(b)) {
            if (!kBig) return;
            ns_big<kB, kWide>(GS, b, SC, blockIdx.x, ngroup, tl);
            flush_tally(b.ctr, tl);
            return;
        }
        const uint32_t g = xcd_block(blockIdx.x, ngroup) * kGroups + threadIdx.x / kGroup;
        const bool active = g < b.offset[b.CT];
        by_scene<kB>((kB && active) ? b.sid[g] : 0u, active,
                     [&](uint32_t sc) { group_search<false, kWide>(GS, b, SC[sc], in_scene<kB>(g), tl); });
    } else {
        item_stats<kB>(b, SC, b.units, b.ctr[CTR_UNITS], tile_cap, (blockIdx.x - ngroup) * kBlock + threadIdx.x,
                       (gridDim.x - ngroup) * kBlock, tl, [](uint2) {});
    }
    flush_tally(b.ctr, tl);
}

template <bool kB, bool kWide>
__global__ __launch_bounds__(kBlock) void k_ns_big(Bufs b, Scenes<kB> SC) {
    if (!big_cells(b)) return;  // uniform over the grid
    __shared__ GroupShared GS;
    Tally tl;
    ns_big<kB, kWide>(GS, b, SC, blockIdx.x, gridDim.x, tl);
    flush_tally(b.ctr, tl);
}

// ------------------------------------------------- K7: lambda
// calcScalingFactorCUDA, memo form (pbf_constraint.cu:168-209): over the
// frozen list, s = C / (m^2 inv_rho0^2 G + eps) with the reference's fma
// order; writes (x*, s).  L lanes per slot (sum_pairs).
template <bool kB, int L>
__global__ __launch_bounds__(256) void k_lambda(Bufs b, Scenes<kB> SC) {
    const uint32_t t = xcd_block() * blockDim.x + threadIdx.x;
    const uint32_t slot = t / L, l = t % L;
    const bool active = slot < b.offset[b.CT];
    by_scene<kB>((kB && active) ? b.sid[slot] : 0u, active, [&](uint32_t sc) {
        const uint32_t i = in_scene<kB>(slot);
        const Phys P = SC[sc].P;
        const F3 self = f3of(b.Pf[i]);
        float a[5] = {0.f, 0.f, 0.f, 0.f, 0.f};  // sum W, sum kg, sum |kg|^2
        sum_pairs<L>(b.nlist, b.cap, i, l, b.ncnt[i], self, b.Pf, P, a, [&](float W, F3 kg, float4, float(&c)[5]) {
            c[0] = W;
            c[1] = kg.x;
            c[2] = kg.y;
            c[3] = kg.z;
            c[4] = fdot(kg, kg);
        });
        const float Cc = __builtin_fmaf(a[0] * P.m, P.inv_rho0, -1.f);
        const float Gs = __builtin_fmaf(a[1], a[1], __builtin_fmaf(a[3], a[3], __builtin_fmaf(a[2], a[2], a[4])));
        if (l == 0u) b.Q[i] = make_float4(self.x, self.y, self.z, Cc / __builtin_fmaf(P.m2r2, Gs, P.relax));
    });
}

// ------------------------------------------------- K8: delta-p + collision + apply
// calcPositionUpdateCUDA (memo form, pbf_position_update.cu:131-188),
// responseCollisionCUDA (pbf_response_collision.cu:12-66) and
// updateInterimPositionCUDA (pbf_constraint.cu:335-345).  Reads (x*, s),
// writes the new x*.  L lanes per slot (sum_pairs).  A scene whose s_corr
// exponent is 4 takes a copy of the sum in which powi is two squarings, chosen by
// the scene (a wave works on one at a time): with the general loop there, a batch
// of 256 scenes took 925 us a launch, with the copy 750.
template <bool kB, int L>
__global__ __launch_bounds__(256) void k_deltap(Bufs b, Scenes<kB> SC) {
    const uint32_t t = xcd_block() * blockDim.x + threadIdx.x;
    const uint32_t slot = t / L, l = t % L;
    const bool active = slot < b.offset[b.CT];
    Tally tl;
    by_scene<kB>((kB && active) ? b.sid[slot] : 0u, active, [&](uint32_t sc) {
        const uint32_t i = in_scene<kB>(slot);
        const Phys P = SC[sc].P;
        const Boundary B = SC[sc].B;
        const float4 se = b.Q[i];
        const F3 self = f3of(se);
        const float si = se.w;
        const float self_cl = (si < 0.f) ? -si : 0.f;
        float sum[3] = {0.f, 0.f, 0.f};
        auto pairs = [&](auto pow4) {
            sum_pairs<L>(b.nlist, b.cap, i, l, b.ncnt[i], self, b.Q, P, sum, [&](float W, F3 kg, float4 pe, float(&c)[3]) {
                const float sj = pe.w;
                float corr;
                if (!pow4() && P.mode == 0) {
                    const float kr2 = W * W;
                    const float kr4 = kr2 * kr2;
                    const float tc = 10.f * kr4 * P.inv_k;
                    const float sup = (sj < 0.f) ? -sj : 0.f;
                    const float cl = self_cl + sup;
                    corr = cl * tc;
                } else {
                    corr = P.sk * powi(W * P.inv_wdq, pow4() ? 4 : P.sn);
                }
                const F3 ak = mulsv(-(si + sj + corr), kg);
                c[0] = ak.x;
                c[1] = ak.y;
                c[2] = ak.z;
            });
        };
        if (P.mode != 0 && P.sn == 4) pairs(std::true_type{});
        else pairs(std::false_type{});
        F3 dp = mk3(sum[0] * P.m * P.inv_rho0, sum[1] * P.m * P.inv_rho0, sum[2] * P.m * P.inv_rho0);
        bool capped = false;
        const int sw = (B.n_planes == 6 && B.n_inner == 0 && B.n_outer == 0)
                           ? collide_planes<6>(P, B, dp, self, capped)
                           : collide(P, B, dp, self, capped);
        const F3 np = self + dp;
        if (l == 0u) {
            b.Pf[i] = make_float4(np.x, np.y, np.z, 0.f);
            tl.sweepcap = capped ? 1u : 0u;
            tl.maxsweep = (uint32_t)sw;
        }
    });
    flush_tally(b.ctr, tl);
}

// ------------------------------------------------- final-cell regrouping
// The vorticity, confinement and XSPH sums visit the 27 cells around each
// particle's FINAL position, bucketed by the search's cell ranges
// (pbf/interaction/cuda/detail/pbf_contribution.inl:7-57).  Particles are
// regrouped by run of at most eight final cells along x (the order inside a run
// does not change a result, every sum is per particle): a counting sort.  Each
// run has four counters, one per group of workgroups (b mod 4), each on its own
// cache line (count_slot), so that a run that collects particles from all over
// the domain -- a corner pile of 7,000 particles on the 1M dam -- is not counted
// through one contended line; key = run * 4 + copy.  Narrower runs keep
// neighbours together in the lists and gathers of the final passes, fewer
// counters are contended: cells per run / counters 16/8, 8/4, 4/4, 1/1 take 1023,
// 1030, 1041, 1102 us for a step of the 1M dam, 8.91, 8.84, 8.79, 9.17 ms of the
// 8M double dam, 36.3, 35.9, 35.6, 35.7 ms for ten steps of the wild 1M flow and
// 15.2, 15.0, 14.9, 14.8 ms for a batch of 256 scenes.  Particles sorted by cell inside
// a run would make the three passes 2.09 ms at 8M instead of 2.20, and 0.14 in a sort of
// its own for that takes it away again.  The same
// pass packs each slot's record R = (x*, 0), (v, 0) with
// v = inv_dt*(x* - x_sorted) (updateVelocityCUDA, pbf_update.cu:25-39), so
// that a particle visited in run order costs one cache line.  Final cells
// need not follow slot order (a violent step scatters them), so equal keys
// are merged over the whole wave, not only over neighbouring lanes.
template <bool kB>
__global__ __launch_bounds__(256) void k_cur_hash(Bufs b, Scenes<kB> SC, uint32_t lguw, uint32_t lgnc, uint32_t lgT,
                                                  uint32_t CR) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    const bool active = s < b.offset[b.CT];
    uint32_t k = 0;
    by_scene<kB>((kB && active) ? b.sid[s] : 0u, active, [&](uint32_t sc) {
        const Scene& S = SC[sc];
        const F3 p = f3of(b.Pf[s]);
        const F3 vv = mulsv(S.P.inv_dt, p - ld3(b.X, b.cap, s));
        const Grid G = S.G;
        int gp[3];
        grid_pos(p, G.cw, gp);
        k = scene_key(gp[0], gp[1], gp[2], G);
        b.R[2 * s] = make_float4(p.x, p.y, p.z, __uint_as_float(k));
        b.R[2 * s + 1] = make_float4(vv.x, vv.y, vv.z, 0.f);
        k = ((k >> lguw) << lgnc) | (blockIdx.x & ((1u << lgnc) - 1u));
    });
    // the final boxes of the big cells' groups (the marks k_big_seg left)
    const uint32_t bm = active ? b.rank[s] : 0u;
    if (__any(bm != 0u)) big_box_add(b.bseg, bm, active ? f3of(b.Pf[s]) : mk3(0.f, 0.f, 0.f));
    const uint32_t r = wave_rank_any(b.ccount, k, active, count_slot(k, CR, lgnc));
    if (active) {
        mark_tile(b.ctflag, k >> lgT);
        b.ckey[s] = k;
        b.crank[s] = r;
    }
}

// Places each particle at its run's position; clears the overflow slots of
// the final-order blocks of 64.
__global__ __launch_bounds__(256) void k_cur_scatter(const uint32_t* __restrict__ offset, uint32_t CT,
                                                     const uint32_t* __restrict__ ckey,
                                                     const uint32_t* __restrict__ crank,
                                                     const uint32_t* __restrict__ coffset,
                                                     uint32_t* __restrict__ cperm, uint32_t* __restrict__ oslot,
                                                     ClearArgs clear) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    clear_counts(clear);
    const uint32_t nl = offset[CT];
    if (s >= nl) return;
    if (s <= (nl - 1u) / 64u) oslot[s] = kNoSlot;  // the final passes' blocks of 64 positions
    cperm[coffset[ckey[s]] + crank[s]] = s;
}

// The 27-cell neighbourhood of a particle's final cell, restated from
// calcContribution (pbf/interaction/cuda/detail/pbf_contribution.inl:7-57):
// cells in z,y,x order, slots ascending in each, per-cell partial sums added
// in that order.  Pairs with dot(d, d) > cut2 lie outside the kernel support
// and add exactly +-0 for finite states; they are skipped.
//
// The final passes run in two stages.  k_final_groups and k_final_big filter
// each particle's candidates once and store its in-range pairs (bit 31 marks
// the first pair of each cell); the vorticity, confinement and XSPH passes then
// walk those lists with every lane busy.  Adding only the cells that have pairs
// gives the same sums: the skipped cells add +0.

// A candidate's records for a pass's term: p = (x*_j, pass-specific w),
// q = the second record the pass needs (the velocity, or unused).  Loaded
// together by the sums, so no load waits on another.
struct El2 {
    float4 p, q;
};

// Partial sum of one cell (key) in slot order: the per-cell sum of
// calcContribution; elem(j) builds the pass's element of slot j.  A big
// cell's groups out of range (final boxes) add nothing and are skipped; a
// single group left is summed through aux, in slot order.
template <bool kBig, class ElemF, class TermF>
__device__ __forceinline__ F3 sum_cell(CellView b, uint32_t key, F3 self, float cut2, ElemF&& elem,
                                       TermF&& term) {
    const uint32_t st = b.offset[key], n = b.offset[key + 1] - st;
    F3 cs = mk3(0.f, 0.f, 0.f);
    if (!kBig) {
        // four candidates' records loaded together, then added in order
        for (uint32_t j = st; j < st + n; j += 4u) {
            El2 el[4];
#pragma unroll
            for (uint32_t i = 0; i < 4u; ++i) el[i] = elem(min(j + i, st + n - 1u));
#pragma unroll
            for (uint32_t i = 0; i < 4u; ++i) {
                const F3 d = f3of(el[i].p) - self;
                if (j + i < st + n && !(glm_dot(d, d) > cut2)) acc(cs, term(el[i]));
            }
        }
        return cs;
    }
    uint32_t p0 = 0, p1 = n;
    bool via = false;
    if (n > kSmallCell) {
        const BigPart bp = big_part<true>(b.bseg + b.bslot[st], self, cut2, n);
        if (bp.how == 0u) return cs;
        if (aux_pays(bp, n)) {
            p0 = bp.p0;
            p1 = bp.p1;
            via = true;
        }
    }
    if (p1 == p0) return cs;
    const uint32_t* __restrict__ ax = b.aux + st;
    uint32_t jn[4];
#pragma unroll
    for (uint32_t i = 0; i < 4u; ++i) jn[i] = via ? ax[min(p0 + i, p1 - 1u)] : st + min(p0 + i, p1 - 1u);
    // four candidates' records loaded together, then added in order
    for (uint32_t p = p0; p < p1; p += 4u) {
        El2 el[4];
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i) el[i] = elem(jn[i]);
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i) jn[i] = via ? ax[min(p + 4u + i, p1 - 1u)] : st + min(p + 4u + i, p1 - 1u);
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i) {
            const F3 d = f3of(el[i].p) - self;
            if (p + i < p1 && !(glm_dot(d, d) > cut2)) acc(cs, term(el[i]));
        }
    }
    return cs;
}

// Whether the final-cell run of slot g is too sparse for a unit (fewer than
// kSparse particles).
__device__ __forceinline__ bool sparse_run(const Bufs& b, uint32_t lgrun, uint32_t g) {
    const uint32_t run = b.ckey[g] >> lgrun;
    return b.coffset[(run + 1u) << lgrun] - b.coffset[run << lgrun] < kSparse;
}

// Own particles of a final-run work item: positions coffset[run] + chunk*kChunk .. of the run order.
struct OwnCur {
    uint32_t c0, n;
};
__device__ __forceinline__ OwnCur own_cur(const Bufs& b, uint2 unit, uint32_t lguw, uint32_t lgrun) {
    OwnCur o;
    const uint32_t run = unit.x >> lguw, skip = (unit.y >> 6) * kChunk;
    o.c0 = b.coffset[run << lgrun] + skip;
    o.n = min(kChunk, b.coffset[(run + 1u) << lgrun] - o.c0);
    return o;
}

// ------------------------------------------------- overflow slots
// A final-order position whose list overflowed keeps the count kFinalK + 1;
// the first such position of each block of 64 takes the block's overflow
// slot (oslot, one atomic per block; ovf lists the slots' blocks), so that
// the passes add its per-cell partials, computed for all 27 cells at once by
// k_ovf_part, instead of summing the cells one after another (which they do
// when no slot was left).  Called by the lanes whose list overflowed (any
// subset of the wave); a wave's positions are consecutive, so its lanes of
// one block are contiguous and only the first of them competes for the slot.
__device__ __forceinline__ uint32_t ovf_mark(const Bufs& b, uint32_t q) {
    const uint64_t m = __ballot(true);
    const uint32_t lane = lane_id(), blk = q >> 6;
    const uint64_t prev = m & ((1ull << lane) - 1ull);
    const uint32_t pb = prev ? (uint32_t)__shfl((int)blk, 63 - __builtin_clzll(prev), 64) : kNoSlot;
    if (pb != blk && atomicCAS(&b.oslot[blk], kNoSlot, kPendingSlot) == kNoSlot) {
        const uint32_t k = atomicAdd(&b.ctr[CTR_OVF], 1u);
        if (k < b.ovf_max) b.ovf[k] = blk;
        b.oslot[blk] = k < b.ovf_max ? k : kFullSlot;
    }
    return kFinalK + 1u;
}

// ------------------------------------------------- K9: final pair lists
// For each particle (by position q of the final-cell order) the slots of its
// in-range pairs in groups of four (list_at(cap, q, k), k < kFinalK); fcnt[q] =
// their count, or kFinalK + 1 when there are more (the passes then fall back
// to the direct sum, so the filter stops at the (kFinalK+1)-th pair: a
// particle in a pile of thousands does not scan its whole neighbourhood).
__device__ __forceinline__ float final_cut2(const Phys& P) { return fmaxf(P.cut2_w, P.cut2_wd); }

// The final list of position q (slot g) by its group of eight lanes, and its
// count or overflow entry; true when the list is left to a whole wave instead.
template <bool kBig, bool kWide>
__device__ __forceinline__ bool group_final(GroupShared& S, const Bufs& b, const Scene& sc, uint32_t q, uint32_t g,
                                            Tally& tl) {
    const Grid G = sc.G;
    const float4 pk = b.R[2 * g];
    const uint32_t n = group_list<true, kBig, kWide>(S, G, cell_view(b), b.Pf, f3of(pk), __float_as_uint(pk.w),
                                                     final_cut2(sc.P), kFinalK, b.flist, b.cap, q, g, kHeavyFinal);
    if (kBig && n == kDeferred) return true;
    if ((lane_id() & (kGroup - 1u)) == 0u) {
        b.fcnt[q] = n > kFinalK ? ovf_mark(b, q) : n;
        tl.listovf += n > kFinalK ? 1u : 0u;
    }
    return false;
}

// The final list of one particle (x* = self, final-order position q),
// built by a whole wave: each cell's candidates (the same ranges and group
// skips as group_list) 64 at a time, lane l testing the l-th; the hits are
// appended in slot order through a ballot.  Returns the pair count, or lim
// once it reaches lim = kFinalK + 1 (the list then overflows and is not
// read).  Called by all lanes of the wave; every value it depends on is the
// same on every lane.
template <bool kBig>
__device__ uint32_t heavy_list(const Grid& G, CellView b, const float4* __restrict__ Pf, F3 self, float cut2,
                               uint32_t* __restrict__ fl, uint32_t cap, uint32_t q) {
    const uint32_t lim = kFinalK + 1u;
    const uint32_t lane = lane_id();
    const uint64_t below = (1ull << lane) - 1ull;
    int gp[3];
    grid_pos(self, G.cw, gp);
    uint32_t n = 0;
    for (int c = 0; c < 27; ++c) {
        const int r = c / 3, dx = c % 3;
        const uint32_t key = scene_key(gp[0] + dx - 1, gp[1] + (r % 3) - 1, gp[2] + (r / 3) - 1, G);
        const uint32_t o0 = b.offset[key], ncell = b.offset[key + 1] - o0;
        uint32_t p0 = 0, p1 = ncell;
        bool via = false;
        if (kBig && ncell > kSmallCell) {
            const BigPart bp = big_part<true>(b.bseg + b.bslot[o0], self, cut2, ncell);
            if (bp.how == 0u) continue;
            if (n + bp.inside >= lim) return lim;
            if (bp.all_in) {  // fewer than lim - n members, all pairs, ascending
                const uint32_t size = bp.p1 - bp.p0;
                for (uint32_t t = lane; t < size; t += 64u) {
                    const uint32_t j = bp.how == 2u ? b.aux[o0 + bp.p0 + t] : o0 + bp.p0 + t;
                    if (n + t < kFinalK) fl[list_at(cap, q, n + t)] = j | (t == 0u ? 0x80000000u : 0u);
                }
                n += size;
                continue;
            }
            if (aux_pays(bp, ncell)) {
                p0 = bp.p0;
                p1 = bp.p1;
                via = true;
            }
        }
        bool any = false;  // a pair of this cell was appended
        for (uint32_t p = p0; p < p1; p += 256u) {
            uint32_t j[4];
            F3 pj[4];
#pragma unroll
            for (uint32_t u = 0; u < 4u; ++u) {
                const uint32_t t = min(p + u * 64u + lane, p1 - 1u);
                j[u] = via ? b.aux[o0 + t] : o0 + t;
            }
#pragma unroll
            for (uint32_t u = 0; u < 4u; ++u) pj[u] = f3of(Pf[j[u]]);
#pragma unroll
            for (uint32_t u = 0; u < 4u; ++u) {
                const bool hit = p + u * 64u + lane < p1 && pair_test<true>(pj[u] - self, cut2);
                const uint64_t m = __ballot(hit);
                if (m == 0ull) continue;
                const uint32_t k = n + (uint32_t)__popcll(m & below);
                if (hit && k < kFinalK)
                    fl[list_at(cap, q, k)] = j[u] | ((!any && (m & below) == 0ull) ? 0x80000000u : 0u);
                n += (uint32_t)__popcll(m);
                any = true;
                if (n >= lim) return lim;
            }
        }
    }
    return n;
}

// The final lists of a step with big cells, as ns_big builds the search's.
template <bool kB, bool kWide>
__device__ __forceinline__ void final_big(GroupShared& GS, const Bufs& b, const Scenes<kB>& SC, uint32_t block,
                                          uint32_t nblock, Tally& tl) {
    const uint32_t nl = b.offset[b.CT], nblk = (nl + kGroups - 1u) / kGroups;
    for (uint32_t c = block; c < nblk; c += nblock) {
        const uint32_t q = c * kGroups + threadIdx.x / kGroup;
        const bool active = q < nl;
        const uint32_t g = active ? b.cperm[q] : 0u;
        bool left = false;
        by_scene<kB>((kB && active) ? b.sid[g] : 0u, active,
                     [&](uint32_t sc) { left = group_final<true, kWide>(GS, b, SC[sc], q, g, tl); });
        uint64_t todo = __ballot(left && (lane_id() & (kGroup - 1u)) == 0u);
        if (todo && lane_id() == 0u) atomicAdd(&b.ctr[CTR_HEAVY], (uint32_t)__popcll(todo));
        while (todo) {
            const int src = __ffsll((unsigned long long)todo) - 1;
            todo &= todo - 1ull;
            const uint32_t qw = (uint32_t)__builtin_amdgcn_readlane((int)q, src);
            const uint32_t gw = (uint32_t)__builtin_amdgcn_readlane((int)g, src);
            const uint32_t sc = kB ? __builtin_amdgcn_readfirstlane(b.sid[gw]) : 0u;
            const Grid G = SC[sc].G;
            const uint32_t n = heavy_list<true>(G, cell_view(b), b.Pf, f3of(b.Pf[gw]), final_cut2(SC[sc].P), b.flist,
                                                b.cap, qw);
            if (lane_id() == 0u) {
                b.fcnt[qw] = n > kFinalK ? ovf_mark(b, qw) : n;
                tl.listovf += n > kFinalK ? 1u : 0u;
            }
        }
    }
}

// Every position by a group of eight lanes (the first ngroup workgroups, unless
// the step has big cells: final_big, in the same launch when kBig); the rest of the grid walks the work
// items for their statistics.
template <bool kB, bool kWide, bool kBig>
__global__ __launch_bounds__(kBlock) void k_final_groups(Bufs b, Scenes<kB> SC, uint32_t tile_cap, uint32_t lguw,
                                                         uint32_t lgrun, uint32_t ngroup) {
    __shared__ GroupShared GS;
    Tally tl;
    if (blockIdx.x < ngroup) {
        const bool any_big = big_cells(b);
        if (kBig && any_big) final_big<kB, kWide>(GS, b, SC, blockIdx.x, ngroup, tl);
        const uint32_t q = xcd_block(blockIdx.x, ngroup) * kGroups + threadIdx.x / kGroup;
        const bool active = q < b.offset[b.CT];
        const uint32_t g = active ? b.cperm[q] : 0u;
        if (active && (threadIdx.x & (kGroup - 1u)) == 0u && sparse_run(b, lgrun, g)) tl.slowpart++;
        by_scene<kB>((kB && active) ? b.sid[g] : 0u, active && !any_big,
                     [&](uint32_t sc) { group_final<false, kWide>(GS, b, SC[sc], in_scene<kB>(q), in_scene<kB>(g), tl); });
    } else {
        item_stats<kB>(b, SC, b.cunits, b.ctr[CTR_CUNITS], tile_cap, (blockIdx.x - ngroup) * kBlock + threadIdx.x,
                       (gridDim.x - ngroup) * kBlock, tl,
                       [&](uint2 unit) { tl.slowpart += own_cur(b, unit, lguw, lgrun).n; });
    }
    flush_tally(b.ctr, tl);
}

template <bool kB, bool kWide>
__global__ __launch_bounds__(kBlock) void k_final_big(Bufs b, Scenes<kB> SC) {
    if (!big_cells(b)) return;  // uniform over the grid
    __shared__ GroupShared GS;
    Tally tl;
    final_big<kB, kWide>(GS, b, SC, blockIdx.x, gridDim.x, tl);
    flush_tally(b.ctr, tl);
}

// Sum over a particle's stored pair list, per-cell partial sums in order;
// elem(j) builds the pass's element of slot j.
template <class ElemF, class TermF>
__device__ __forceinline__ F3 sum_list(const uint32_t* __restrict__ fl, uint32_t cap, uint32_t q, uint32_t n,
                                       ElemF&& elem, TermF&& term) {
    F3 sum = mk3(0.f, 0.f, 0.f), cs = mk3(0.f, 0.f, 0.f);
    uint4 w = n ? list_word(fl, cap, q, 0u) : make_uint4(0u, 0u, 0u, 0u);
    for (uint32_t k = 0; k < n; k += 4u) {
        uint32_t e[4];
        El2 el[4];
        list_group(w, k, n, e);
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i) el[i] = elem(e[i] & 0x7FFFFFFFu);
        w = list_word(fl, cap, q, min(k + 4u, (n - 1u) & ~3u));  // next group, in flight during this one
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i)
            if (k + i < n) {
                if (e[i] >> 31) {
                    acc(sum, cs);
                    cs = mk3(0.f, 0.f, 0.f);
                }
                acc(cs, term(el[i]));
            }
    }
    acc(sum, cs);
    return sum;
}

// sum_list for an elem that takes any index: the entries past n in the last
// word are loaded as they are and not summed.
template <class ElemF, class TermF>
__device__ __forceinline__ F3 sum_list_any(const uint32_t* __restrict__ fl, uint32_t cap, uint32_t q, uint32_t n,
                                           ElemF&& elem, TermF&& term) {
    F3 sum = mk3(0.f, 0.f, 0.f), cs = mk3(0.f, 0.f, 0.f);
    uint4 w = n ? list_word(fl, cap, q, 0u) : make_uint4(0u, 0u, 0u, 0u);
    for (uint32_t k = 0; k < n; k += 4u) {
        const uint32_t e[4] = {w.x, w.y, w.z, w.w};
        El2 el[4];
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i) el[i] = elem(e[i] & 0x7FFFFFFFu);
        w = list_word(fl, cap, q, min(k + 4u, (n - 1u) & ~3u));  // next group, in flight during this one
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i)
            if (k + i < n) {
                if (e[i] >> 31) {
                    acc(sum, cs);
                    cs = mk3(0.f, 0.f, 0.f);
                }
                acc(cs, term(el[i]));
            }
    }
    acc(sum, cs);
    return sum;
}

// sum_list by a group of L lanes (l: this lane), one entry each of every L: the
// entries' terms and first-of-cell marks are then taken in list order by every
// lane, which forms the same partial sums bit for bit (an entry past n adds a
// zero term).
template <int L, int m = 0>
__device__ __forceinline__ void add_cell_lanes(F3& sum, F3& cs, float first, F3 t) {
    if constexpr (m < L) {
        if (lane_of<L, m>(first) != 0.f) {
            acc(sum, cs);
            cs = mk3(0.f, 0.f, 0.f);
        }
        acc(cs, mk3(lane_of<L, m>(t.x), lane_of<L, m>(t.y), lane_of<L, m>(t.z)));
        add_cell_lanes<L, m + 1>(sum, cs, first, t);
    }
}
template <int L, class ElemF, class TermF>
__device__ __forceinline__ F3 sum_list_lanes(const uint32_t* __restrict__ fl, uint32_t cap, uint32_t q, uint32_t l,
                                             uint32_t n, ElemF&& elem, TermF&& term) {
    F3 sum = mk3(0.f, 0.f, 0.f), cs = mk3(0.f, 0.f, 0.f);
    uint32_t e = l < n ? fl[list_at(cap, q, l)] : 0u;
    for (uint32_t k = l; k - l < n; k += (uint32_t)L) {
        const El2 el = elem(e & 0x7FFFFFFFu);
        const float first = (e >> 31) ? 1.f : 0.f;
        const bool on = k < n;
        e = k + (uint32_t)L < n ? fl[list_at(cap, q, k + (uint32_t)L)] : 0u;
        const F3 t = term(el);
        add_cell_lanes<L>(sum, cs, first, on ? t : mk3(0.f, 0.f, 0.f));
    }
    acc(sum, cs);
    return sum;
}

// Visits position q of the final-cell order, L lanes each (l: this lane):
// body(q, slot, stored pair count, scene, l), grouped by scene (no operations
// across groups inside).
template <bool kB, int L, class F>
__device__ __forceinline__ void for_final(const Bufs& b, F&& body) {
    const uint32_t t = xcd_block() * blockDim.x + threadIdx.x;
    const uint32_t q = t / L, l = t % L;
    const bool active = q < b.offset[b.CT];
    const uint32_t g = active ? b.cperm[q] : 0u;
    by_scene<kB>((kB && active) ? b.sid[g] : 0u, active, [&](uint32_t sc) {
        const uint32_t qs = in_scene<kB>(q), gs = in_scene<kB>(g);
        body(qs, gs, b.fcnt[qs], sc, l);
    });
}

// The pair terms of the final passes.  Each takes its root (and the three
// divisions by it) from sqrt_inv_normal and div3_inv in a wave whose active
// lanes all qualify (the IEEE sequences otherwise): over the piles of the first
// ten chained steps of the 1M dam k_ovf_part went from 1.72 to 1.41 ms a launch
// (vorticity) and from 1.58 to 1.33 ms (confinement).  kPlain false: the IEEE
// sequences only, the same values.

// vorticity pair term (pbf_vorticity_confinement.cu:15-31)
template <bool kPlain>
__device__ __forceinline__ F3 vort_pair(F3 self, F3 selfv, F3 pj, F3 vj, float warg) {
    const F3 pd = pj - self;
    const F3 vd = vj - selfv;
    const float r2 = glm_dot(pd, pd);
    F3 w = mk3(0.f, 0.f, 0.f);
    if (kPlain && __builtin_expect(wave_plain_div(pd, r2), 1)) {
        const RootInv q = sqrt_inv_normal(r2);
        if (r2 != 0.f) w = mulvs(glm_cross(vd, div3_inv(pd, q.s, q.inv)), wspiky_deriv(q.s, warg));
        return w;
    }
    const float r = glm_length(pd);
    if (r > 0.f) w = mulvs(glm_cross(vd, divvs(pd, r)), wspiky_deriv(r, warg));
    return w;
}

// confinement location-vector pair term (pbf_vorticity_confinement.cu:121-138)
template <bool kPlain>
__device__ __forceinline__ F3 loc_pair(F3 self, F3 pj, float wj, float warg) {
    const F3 pd = pj - self;
    const float r2 = glm_dot(pd, pd);
    F3 l = mk3(0.f, 0.f, 0.f);
    if (kPlain && __builtin_expect(wave_plain_div(pd, r2), 1)) {
        const RootInv q = sqrt_inv_normal(r2);
        if (r2 != 0.f) l = mulvs(mulsv(wj, div3_inv(pd, q.s, q.inv)), wspiky_deriv(q.s, warg));
        return l;
    }
    const float r = glm_length(pd);
    if (r > 0.f) l = mulvs(mulsv(wj, divvs(pd, r)), wspiky_deriv(r, warg));
    return l;
}

// XSPH pair term (pbf_xsph.cu:15-29)
template <bool kPlain>
__device__ __forceinline__ F3 xsph_pair(F3 self, F3 selfv, F3 pj, F3 vj, float inv_h) {
    const F3 pd = pj - self;
    const F3 vd = vj - selfv;
    const float r2 = glm_dot(pd, pd);
    if (kPlain && __builtin_expect(wave_plain_r2(r2), 1))
        return mulvs(vd, wpoly6(r2 != 0.f ? sqrt_inv_normal(r2).s : 0.f, inv_h));
    return mulvs(vd, wpoly6(glm_length(pd), inv_h));
}

// The three final passes as (elements, pair term, support) for the particle
// at slot g: the list walk, the direct sum, the per-cell partials and their
// combination all evaluate a pass through these.
enum FinalPass : int { PASS_VORT = 0, PASS_CONF = 1, PASS_XSPH = 2 };

template <int kPass>
struct PassTerms {
    const float4* __restrict__ R;
    const float4* __restrict__ OM4;
    F3 self, selfv;
    uint32_t key;  // of the final cell
    float arg, cut2;
    __device__ __forceinline__ PassTerms(const Bufs& b, const Phys& P, uint32_t g)
        : PassTerms(b, P, g, b.R[2 * g]) {}
    __device__ __forceinline__ PassTerms(const Bufs& b, const Phys& P, uint32_t g, float4 r0)
        : R(b.R), OM4(b.OM4), self(f3of(r0)),
          selfv(kPass == PASS_CONF ? mk3(0.f, 0.f, 0.f) : f3of(b.R[2 * g + 1])), key(__float_as_uint(r0.w)),
          arg(kPass == PASS_XSPH ? P.inv_h : P.warg), cut2(kPass == PASS_XSPH ? P.cut2_w : P.cut2_wd) {}
    __device__ __forceinline__ El2 elem(uint32_t j) const {
        if (kPass == PASS_CONF) {
            const float4 r = R[2 * j];
            return El2{make_float4(r.x, r.y, r.z, OM4[j].w), make_float4(0.f, 0.f, 0.f, 0.f)};
        }
        return El2{R[2 * j], R[2 * j + 1]};
    }
    // the same through buffer resources (records of slot j at byte 32j of R, 16j of OM4)
    __device__ __forceinline__ El2 elem_buf(const Gather16& gr, const Gather16& go, uint32_t j) const {
        if (kPass == PASS_CONF) {
            const float4 r = gr(2u * j);
            return El2{make_float4(r.x, r.y, r.z, go(j).w), make_float4(0.f, 0.f, 0.f, 0.f)};
        }
        return El2{gr(2u * j), gr(2u * j + 1u)};
    }
    template <bool kPlain = true>
    __device__ __forceinline__ F3 term(const El2& e) const {
        if (kPass == PASS_VORT) return vort_pair<kPlain>(self, selfv, f3of(e.p), f3of(e.q), arg);
        if (kPass == PASS_CONF) return loc_pair<kPlain>(self, f3of(e.p), e.p.w, arg);
        return xsph_pair<kPlain>(self, selfv, f3of(e.p), f3of(e.q), arg);
    }
};

// Partial sum of cell c (0..26) of the 27 around the pass particle's final
// cell, by a group of L lanes (l: this lane): L candidates at a time, a lane
// each, and the terms of those in range added in slot order by every lane (the
// others add +0), as sum_cell adds them; the next candidates are loaded while one
// step is added.  Called by all lanes of the group.
template <bool kBig, int L, class Pass>
__device__ __forceinline__ F3 sum_cell_lanes(CellView b, const Grid& G, const Pass& ps, uint32_t c, uint32_t l) {
    const uint32_t key = key27(ps.key, c, G);
    const uint32_t st = b.offset[key], n = b.offset[key + 1] - st;
    float cs[3] = {0.f, 0.f, 0.f};
    uint32_t p0 = 0, p1 = n;
    bool via = false;
    if (kBig && n > kSmallCell) {
        const BigPart bp = big_part<true>(b.bseg + b.bslot[st], ps.self, ps.cut2, n);
        if (bp.how == 0u) p1 = 0u;
        if (aux_pays(bp, n)) {
            p0 = bp.p0;
            p1 = bp.p1;
            via = true;
        }
    }
    if (p0 < p1) {
        auto slot = [&](uint32_t t) {
            const uint32_t u = min(t, p1 - 1u);
            return kBig && via ? b.aux[st + u] : st + u;
        };
        El2 el = ps.elem(slot(p0 + l));
        uint32_t jn = slot(p0 + (uint32_t)L + l);
        for (uint32_t p = p0; p < p1; p += (uint32_t)L) {
            const El2 nx = ps.elem(jn);
            jn = slot(p + 2u * (uint32_t)L + l);
            const F3 d = f3of(el.p) - ps.self;
            const bool in = p + l < p1 && !(glm_dot(d, d) > ps.cut2);
            if (__builtin_amdgcn_ballot_w64(in)) {
                F3 t = mk3(0.f, 0.f, 0.f);
                if (in) t = ps.term(el);
                const float v[3] = {t.x, t.y, t.z};
                add_lanes<L>(cs, v);
            }
            el = nx;
        }
    }
    return mk3(cs[0], cs[1], cs[2]);
}

// Direct sum over the 27 cells, for an overflowing position whose block has no
// overflow slot (only in the allocation-free step, which has 64): the cells' partial
// sums added in z,y,x order, each by the pass's own L lanes.  With every lane adding
// the whole sum a static step of 12,000 particles in 3x3x3 cells took 6.2 ms (12,000
// and 30,000 of about 30 a cell 0.65 and 0.68), now 1.6 (0.28 and 0.40).
template <bool kBig, int L, class Pass>
__device__ __forceinline__ F3 sum27(const Bufs& b, const Grid& G, const Pass& ps, uint32_t l) {
    F3 sum = mk3(0.f, 0.f, 0.f);
    for (uint32_t c = 0; c < 27u; ++c) {
        if constexpr (L > 1)
            acc(sum, sum_cell_lanes<kBig, L>(cell_view(b), G, ps, c, l));
        else
            acc(sum, sum_cell<kBig>(cell_view(b), key27(ps.key, c, G), ps.self, ps.cut2,
                                    [&](uint32_t j) { return ps.elem(j); }, [&](const El2& e) { return ps.term(e); }));
    }
    return sum;
}

// The pass's sum for final-order position q with stored count n: the list
// (n <= kFinalK), or, for n = kFinalK + 1, the 27 per-cell partials that
// k_ovf_part left in its block's overflow slot, added in the same z,y,x order
// as the direct 27-cell sum adds its cells (which it does when the block has
// no slot).
template <int L, class Pass>
__device__ __forceinline__ F3 pass_sum(const Bufs& b, const Grid& G, const Pass& ps, uint32_t q, uint32_t n,
                                       uint32_t l) {
    auto elem = [&](uint32_t j) { return ps.elem(j); };
    auto term = [&](const El2& e) { return ps.term(e); };
    if (n <= kFinalK) {
        if constexpr (L > 1) return sum_list_lanes<L>(b.flist, b.cap, q, l, n, elem, term);
        if (b.cap < kGatherMaxSlots / 2u) {
            const Gather16 gr(b.R, 2u * b.cap), go(b.OM4, b.cap);
            return sum_list_any(b.flist, b.cap, q, n, [&](uint32_t j) { return ps.elem_buf(gr, go, j); }, term);
        }
        return sum_list(b.flist, b.cap, q, n, elem, term);
    }
    const uint32_t k = b.oslot[q >> 6];
    if (k >= b.ovf_max)
        return big_cells(b) ? sum27<true, L>(b, G, ps, l) : sum27<false, L>(b, G, ps, l);
    const float4* __restrict__ pk = b.part + (size_t)k * 27u * 64u + (q & 63u);
    F3 sum = mk3(0.f, 0.f, 0.f);
    for (uint32_t c = 0; c < 27u; ++c) acc(sum, f3of(pk[c * 64u]));
    return sum;
}


// Per-cell partials of pass kPass for the overflow slots, in one of two forms.
//
// By rows: a wave task is (slot k, cell c, four consecutive positions of the slot's
// block), row r summing cell c of the 27 around final-order position
// 64 * ovf[k] + 4 * sub + r, when that position overflowed, in slot order
// (sum_cell_lanes) into part[(k * 27 + c) * 64 + 4 * sub + r].  Consecutive tasks
// share a cell index, so a workgroup's rows mostly scan the same cell, and the
// pass reads each row of 64 whole.
//
// By threads: a wave task is (slot k, cell c), lane l summing the cell for position
// 64 * ovf[k] + l.  Few candidates of large piles are pairs, so the terms take the
// IEEE root without asking whether the wave's pairs allow the short one (143 against
// 153 ms for the three sums of a step of the 8M double dam, steps 30 to 35).
//
// A cell of a pile is one serial sum of thousands of terms, which sets the time of the
// threads until there are sums enough to hide it; by rows it is 16 times shorter, but
// adding the terms on every lane doubles the work.  So the threads take over when the
// overflowing particles are more than kOvfCell times the largest cell, or more than
// kOvfFull times where their blocks are seven eighths full (in others the lanes of
// the threads idle), or more than kOvfRows.  Measured, time of the rows over time of the
// threads:
//   fluid of 20 to 1,000 particles a cell throughout, by overflowing particles over
//   the largest cell (64 at least): 0.8 at 25, 1.0 at 50, 1.15 at 100, 1.4 at 200, 2 at 2,000;
//   full cells of 700 to 15,000 particles in a cube: 1.0 at 8, 1.1 to 1.4 from 24 to 60;
//   a dam of 200,000 particles with a weak tensile term, falling together: 1.0 at 200, 1.2
//   at 300; with a strong one (blocks half full): 0.45 at 25, 0.6 at 40;
//   chained 1M to 8M dams (cells of 12,000 to 300,000: at most 41; blocks seven eighths
//   full: 1.0 to 1.3 at 35), by overflowing particles: 0.3 up to 50,000, 0.45 up to
//   200,000, 0.67 up to 350,000, 0.87 up to 600,000, 0.98 up to 700,000, 1.17 up to
//   800,000, 1.3 up to 2,000,000, 1.7 above.
//
// The tasks differ by a thousand times, so the launch has many times the workgroups
// that fit the chip (ovf_blocks), which the hardware hands out as others end.  With the
// 2,048 that fit, each wave going round the tasks in a fixed order, the three sums of a
// step took 652 ms on the 8M double dam, steps 20 to 25, and 14.5 ms on the 1M dam, steps
// 80 to 100; with 32,768 and 8,192 workgroups 419 and 12.0.
constexpr uint32_t kOvfRows = 655360, kOvfCell = 64, kOvfFull = 24;

// Whether the ns slots' cells are summed by threads.  The overflowing positions come
// from the statistics the list builds left.
__device__ __forceinline__ bool ovf_by_threads(const uint32_t* __restrict__ ctr, uint32_t ns) {
    static_assert(kStatRep == 64, "a lane reads a copy");
    const uint64_t cell = max(kSmallCell, ctr[kCtrMostCell]);
    if (64ull * ns <= min((uint64_t)kOvfRows, kOvfFull * cell)) return false;
    uint32_t v = ctr[CTR_NUM * (1u + lane_id()) + CTR_LISTOVF];
    for (int d = 32; d > 0; d >>= 1) v += (uint32_t)__shfl_xor((int)v, d, 64);
    return v > kOvfRows || v > kOvfCell * cell || (v > kOvfFull * cell && v > 56ull * ns);
}

template <bool kB, int kPass>
__global__ __launch_bounds__(256) void k_ovf_part(Bufs b, Scenes<kB> SC) {
    const uint32_t ns = min(b.ctr[CTR_OVF], b.ovf_max);
    if (ns == 0u) return;  // uniform over the grid
    const uint32_t nl = b.offset[b.CT], lane = lane_id();
    const bool any_big = big_cells(b);
    const uint32_t w0 = __builtin_amdgcn_readfirstlane((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
    const uint32_t nw = (gridDim.x * blockDim.x) >> 6;
    if (!ovf_by_threads(b.ctr, ns)) {
        const uint32_t ntask = ns * (27u * 16u), l = lane & 15u;
        for (uint32_t t = w0; t < ntask; t += nw) {
            const uint32_t kc = t >> 4, k = kc / 27u, c = kc - k * 27u;
            const uint32_t at = (t & 15u) * 4u + (lane >> 4);  // position in the block
            const uint32_t q = b.ovf[k] * 64u + at;
            const bool active = q < nl && b.fcnt[q] == kFinalK + 1u;
            if (!__any(active)) continue;
            const uint32_t g = active ? b.cperm[q] : 0u;
            by_scene<kB>((kB && active) ? b.sid[g] : 0u, active, [&](uint32_t sc) {
                const PassTerms<kPass> ps(b, SC[sc].P, g);
                const F3 cs = any_big ? sum_cell_lanes<true, 16>(cell_view(b), SC[sc].G, ps, c, l)
                                      : sum_cell_lanes<false, 16>(cell_view(b), SC[sc].G, ps, c, l);
                if (l == 0u) b.part[((size_t)k * 27u + c) * 64u + at] = make_float4(cs.x, cs.y, cs.z, 0.f);
            });
        }
        return;
    }
    const uint32_t ntask = ns * 27u;
    for (uint32_t t = w0; t < ntask; t += nw) {
        const uint32_t k = t / 27u, c = t - k * 27u;
        const uint32_t q = b.ovf[k] * 64u + lane;
        const bool active = q < nl && b.fcnt[q] == kFinalK + 1u;
        const uint32_t g = active ? b.cperm[q] : 0u;
        by_scene<kB>((kB && active) ? b.sid[g] : 0u, active, [&](uint32_t sc) {
            const Grid G = SC[sc].G;
            const PassTerms<kPass> ps(b, SC[sc].P, g);
            auto elem = [&](uint32_t j) { return ps.elem(j); };
            auto term = [&](const El2& e) { return ps.template term<false>(e); };
            const uint32_t key = key27(ps.key, c, G);
            const F3 cs = any_big ? sum_cell<true>(cell_view(b), key, ps.self, ps.cut2, elem, term)
                                  : sum_cell<false>(cell_view(b), key, ps.self, ps.cut2, elem, term);
            b.part[((size_t)k * 27u + c) * 64u + lane] = make_float4(cs.x, cs.y, cs.z, 0.f);
        });
    }
}

// ------------------------------------------------- K10: vorticity
// calcVorticityCUDA (pbf_vorticity_confinement.cu:87-115) with inv_h in the
// spiky derivative (or h, when reproducing the reference's argument);
// writes (omega, |omega|).  Elements: (x*_j, slot j).
template <bool kB, int L>
__global__ __launch_bounds__(kBlock) void k_vort(Bufs b, Scenes<kB> SC) {
    for_final<kB, L>(b, [&](uint32_t q, uint32_t g, uint32_t n, uint32_t sc, uint32_t l) {
        const Phys P = SC[sc].P;
        if (!P.vort_on) {
            if (l == 0u) b.OM4[g] = make_float4(0.f, 0.f, 0.f, 0.f);
            return;
        }
        const float mr = P.m * P.inv_rho0;
        const F3 w = pass_sum<L>(b, SC[sc].G, PassTerms<PASS_VORT>(b, P, g), q, n, l);
        const F3 om = mulsv(mr, w);
        if (l == 0u) b.OM4[g] = make_float4(om.x, om.y, om.z, glm_length(om));
    });
}

// ------------------------------------------------- K11: vorticity confinement
// addVorticityConfinementCUDA (pbf_vorticity_confinement.cu:192-222), in place
// on the record's velocity.  Elements: (x*_j, |omega_j|).
template <bool kB, int L>
__global__ __launch_bounds__(kBlock) void k_confine(Bufs b, Scenes<kB> SC) {
    float4* __restrict__ R = b.R;
    const float4* __restrict__ OM4 = b.OM4;
    for_final<kB, L>(b, [&](uint32_t q, uint32_t g, uint32_t n, uint32_t sc, uint32_t l) {
        const Phys P = SC[sc].P;
        if (!P.vort_on) return;
        F3 N = pass_sum<L>(b, SC[sc].G, PassTerms<PASS_CONF>(b, P, g), q, n, l);
        if (l == 0u && glm_length(N) > 0.f) {
            N = mulvs(mulvs(N, P.m), P.inv_rho0);
            N = divvs(N, glm_length(N));
            const F3 add = mulvs(divvs(mulsv(P.vc, glm_cross(N, f3of(OM4[g]))), P.inv_rho0), P.dtc);
            const F3 nv = f3of(R[2 * g + 1]) + add;
            R[2 * g + 1] = make_float4(nv.x, nv.y, nv.z, 0.f);
        }
    });
}

// ------------------------------------------------- K12: XSPH + write-back
// calcXSPHCUDA (pbf_xsph.cu:84-113) and updatePosition (pbf_update.cu:16-23):
// x_out = x*, v_out = v + c*m*inv_rho0*sum unless the sum is NaN, with v the
// record's velocity (after confinement when that ran).
template <bool kB, int L>
__global__ __launch_bounds__(kBlock) void k_xsph_out(Bufs b, Scenes<kB> SC, float* __restrict__ xo, float* __restrict__ vo) {
    const float4* __restrict__ R = b.R;
    Tally tl;
    for_final<kB, L>(b, [&](uint32_t q, uint32_t g, uint32_t n, uint32_t sc, uint32_t l) {
        const Phys P = SC[sc].P;
        const F3 self = f3of(R[2 * g]);
        const F3 selfv = f3of(R[2 * g + 1]);
        if (!P.xsph_on) {
            if (l == 0u) {
                reinterpret_cast<F3*>(xo)[g] = self;
                reinterpret_cast<F3*>(vo)[g] = selfv;
            }
            return;
        }
        const F3 a = pass_sum<L>(b, SC[sc].G, PassTerms<PASS_XSPH>(b, P, g), q, n, l);
        if (l != 0u) return;
        F3 out;
        if (isnan(a.x) || isnan(a.y) || isnan(a.z)) {
            out = selfv;
            ++tl.nan;
        } else {
            out = selfv + mulsv(P.xsph_c * P.m * P.inv_rho0, a);
        }
        reinterpret_cast<F3*>(xo)[g] = self;  // 12-byte stores
        reinterpret_cast<F3*>(vo)[g] = out;
    });
    flush_tally(b.ctr, tl);
}

// ------------------------------------------------- K13: write-back without XSPH
// pbf_solve.cpp:125-145 as shipped: v = inv_dt*(x* - x_sorted), x = x*; with
// R (vorticity ran without XSPH) the record's position and confined velocity.
template <bool kB>
__global__ __launch_bounds__(256) void k_out(Bufs b, Scenes<kB> SC, const float4* __restrict__ R, float* __restrict__ xo,
                                             float* __restrict__ vo) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t nl = b.offset[b.CT];
    if (s >= nl) return;
    const uint32_t cap = b.cap;
    F3 p, vv;
    if (R) {
        p = f3of(R[2 * s]);
        vv = f3of(R[2 * s + 1]);
    } else {
        p = f3of(b.Pf[s]);
        vv = mulsv(SC[kB ? b.sid[s] : 0u].P.inv_dt, p - ld3(b.X, cap, s));
    }
    reinterpret_cast<F3*>(xo)[s] = p;  // 12-byte stores
    reinterpret_cast<F3*>(vo)[s] = vv;
}

// ------------------------------------------------- views
__global__ __launch_bounds__(256) void k_neighbors_view(Bufs b, uint32_t* __restrict__ out,
                                                        uint32_t* __restrict__ counts, uint32_t max_pair) {
    const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= b.offset[b.CT]) return;
    const uint32_t cnt = b.ncnt[g];
    counts[g] = cnt;
    for (uint32_t c = 0; c < max_pair; ++c)
        out[(size_t)g * max_pair + c] = c < cnt ? b.nlist[list_at(b.cap, g, c)] : 0xFFFFFFFFu;
}

__global__ void k_cell_ranges(const uint32_t* __restrict__ offset, uint32_t C, uint32_t* __restrict__ start,
                              uint32_t* __restrict__ end) {
    const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= C) return;
    const uint32_t a = offset[c], z = offset[c + 1];
    start[c] = (z > a) ? a : 0xFFFFFFFFu;
    end[c] = (z > a) ? z : 0u;
}

__global__ void k_copy_lambda(const uint32_t* __restrict__ offset, uint32_t C, const float4* __restrict__ Q,
                              float* __restrict__ out) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= offset[C]) return;
    out[s] = Q[s].w;
}

// calcDensityCUDA (pbf/solver/cuda/pbf_density.cu:11-71) over the last
// step's frozen lists: rho_i = sum_j m * W(|x_i - x_j|), W with inv_h (the
// reference passes h as the kernel's inv_h argument, pbf_density.cu:22).
// x: AoS float3 in the step's sorted order.
// Eight entries' positions in flight and the root from one v_rsq_f32 where the wave's
// pairs allow it (entry by entry with the IEEE root, the chain of list and gather
// loads took 31 us for 290,000 particles, now 17).
template <bool kB>
__global__ __launch_bounds__(256) void k_density(Bufs b, Scenes<kB> SC, const float* __restrict__ x, float* __restrict__ rho) {
    const F3* __restrict__ pos = reinterpret_cast<const F3*>(x);
    const uint32_t slot = xcd_block() * blockDim.x + threadIdx.x;
    const bool active = slot < b.offset[b.CT];
    by_scene<kB>((kB && active) ? b.sid[slot] : 0u, active, [&](uint32_t sc) {
        const uint32_t i = in_scene<kB>(slot);
        const Phys P = SC[sc].P;
        const F3 self = pos[i];
        float sum = 0.f;
        for_list8(
            b.nlist, b.cap, i, b.ncnt[i],
            [&](uint32_t j) {
                const F3 p = pos[j];
                return make_float4(p.x, p.y, p.z, 0.f);
            },
            [&](uint32_t, float4 el) {
                const F3 d = self - f3of(el);
                const float r2 = glm_dot(d, d);
                float r;
                if (__builtin_expect(wave_plain_r2(r2), 1)) r = r2 != 0.f ? sqrt_inv_normal(r2).s : 0.f;
                else r = glm_length(d);
                sum += wpoly6(r, P.inv_h) * P.m;
            });
        rho[i] = sum;
    });
}

// restoreOrderCUDA (pbf/interaction/cuda/pbf_neighbor_search_util.cu:156-170):
// out[sorted_index[s]] = sorted[s] for the live slots of the last step.
__global__ void k_restore(Bufs b, const float* __restrict__ xs, const float* __restrict__ vs,
                          float* __restrict__ xo, float* __restrict__ vo) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= b.offset[b.CT]) return;
    const uint32_t o = b.sidx[s];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        xo[3 * o + c] = xs[3 * s + c];
        vo[3 * o + c] = vs[3 * s + c];
    }
}

// First sorted slot of each scene after the step (the particles of scene s
// are slots [out[s], out[s+1]) of the output), out[nscenes] = live total.
__global__ void k_scene_offsets(Bufs b, uint32_t* __restrict__ out) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s <= b.nscenes) out[s] = b.offset[b.kbase[s]];
}

// x / y, sqrt(x), fma(x, y, x) and floor(x / y) of each pair, as the device computes them.
__global__ void k_selftest(const float* __restrict__ a, const float* __restrict__ bb, float* __restrict__ out,
                           uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float x = a[i], y = bb[i];
    out[4 * i + 0] = x / y;
    out[4 * i + 1] = __builtin_sqrtf(x);
    out[4 * i + 2] = __builtin_fmaf(x, y, x);
    out[4 * i + 3] = floorf(x / y);
}

// sqrt_inv against sqrtf and 1.f / sqrtf on every bit pattern in [lo, hi]
// (grid-stride): counts the mismatches and records the first one's input bits (any one, if
// several race).
__global__ __launch_bounds__(256) void k_selftest_inv_sqrt(uint32_t lo, uint32_t hi,
                                                           unsigned long long* __restrict__ mismatches,
                                                           uint32_t* __restrict__ first) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    uint32_t bad = 0, which = 0;
    for (uint64_t u = (uint64_t)lo + blockIdx.x * blockDim.x + threadIdx.x; u <= hi; u += stride) {
        const float r2 = __uint_as_float((uint32_t)u);
        const RootInv q = sqrt_inv(r2);
        const float s = __builtin_sqrtf(r2);
        if (__float_as_uint(q.s) != __float_as_uint(s) || __float_as_uint(q.inv) != __float_as_uint(1.f / s)) {
            if (!bad) which = (uint32_t)u;
            ++bad;
        }
    }
    if (bad) {
        atomicAdd(mismatches, (unsigned long long)bad);
        atomicExch(first, which);
    }
}


inline uint32_t ceil_div(uint32_t a, uint32_t b) { return (a + b - 1) / b; }

}  // namespace

const char* kernel_name(int id) {
    static const char* names[K_NUM] = {"k_predict_hash", "k_scan_tiles", "k_scan_cells", "k_scatter",
                                       "k_reorder",      "k_ns",         "k_lambda",     "k_deltap",
                                       "k_vort",         "k_confine",    "k_xsph_out",   "k_out",
                                       "k_cur_sort",     "k_final_list",  "k_big_seg"};
    return (id >= 0 && id < K_NUM) ? names[id] : "?";
}

namespace {
struct Mark {
    Timer* t;
    hipStream_t s;
    int slot;
    Mark(Timer* tm, hipStream_t st, int id) : t(tm), s(st), slot(-1) {
        if (t && t->n < kTimerSlots) {
            slot = t->n++;
            t->id[slot] = id;
            (void)hipEventRecord(t->ev[2 * slot], s);
        }
    }
    ~Mark() {
        if (slot >= 0) (void)hipEventRecord(t->ev[2 * slot + 1], s);
    }
};
}  // namespace

namespace {
// Lanes per particle of the passes that walk a list per particle: as many as
// leave the chip (65,536 lanes at one wave a SIMD) about full.  Measured, k_deltap
// with 16 / 4 / 1 lanes: 8.2 / 10.4 / 12.1 us for 960 particles, 8.3 / 10.3 / 12.6
// for 8,000, 12.2 / 10.4 / 12.7 for 32,768, 18.4 / 12.5 / 13.3 for 65,600 and
// 28.8 / 17.7 / 14.2 for 130,000; k_lambda and the final passes cross at the same
// sizes.
constexpr uint32_t kRowMax = 16384, kQuadMax = 81920;
template <class F>
void by_lanes(uint32_t n, F&& f) {
    if (n <= kRowMax) f(std::integral_constant<int, 16>{});
    else if (n <= kQuadMax) f(std::integral_constant<int, 4>{});
    else f(std::integral_constant<int, 1>{});
}
// Whether a record's byte offset passes 32 bits.
template <class F>
void by_width(uint32_t cap, F&& f) {
    if (cap < kGatherMaxSlots) f(std::false_type{});
    else f(std::true_type{});
}
// workgroups that walk the work items for statistics, one item a thread or more
uint32_t stat_blocks(uint32_t n) { return std::min(64u, 1u + ceil_div(n, 4096u)); }
// workgroups of the big-cell list builds (a loop over 32 particles each)
dim3 big_grid(uint32_t n) { return dim3(std::min(4096u, ceil_div(n, kGroups))); }
// Workgroups of k_ovf_part: at least what fills the chip, and one for every two
// blocks of positions up to 32,768 (where no position overflows, a launch takes 4.6 us
// with 2,048 or 8,192 workgroups and 8.3 with 32,768).
uint32_t ovf_blocks(uint32_t n) { return std::min(32768u, std::max(2048u, n / 128u)); }
// Tiles up to which a scan needs no launch for the tile totals (the last workgroup
// then reads 8 x 4096 counts; a step of 10,000 particles over 8 tiles 97 us, with
// the launch 101, of 960 over 4 tiles 150 and 155; the same at 16 tiles), and up to
// which it needs none for their prefixes (at most 16 KiB read by each workgroup;
// above, the reads grow with the square of the tiles).
constexpr uint32_t kDirectTiles = 8, kPrefixTiles = 4096;
// Particles up to which the lists of a step with big cells are built in the launch
// of the others, which then has registers for five waves a SIMD instead of eight:
// 40 chained steps of the wild 32,768-particle dam 18.8 ms, with launches of their
// own 19.4; ten differentiable steps of 65,536 particles 29.0 and 29.2; 24 scenes of
// 150,000 particles in all 287 us and 285.
constexpr uint32_t kOneListMax = 81920;
const uint32_t* totals_of(const uint32_t* tsum, bool direct) { return direct ? nullptr : tsum; }
const uint32_t* prefix_of(const uint32_t* tprefix, uint32_t nT) { return nT <= kPrefixTiles ? nullptr : tprefix; }
// The launches before k_scan_cells: the tile totals, and their prefixes.
void scan_totals(uint32_t* count, uint32_t* tsum, uint32_t* tflag, uint32_t* tprefix, uint32_t nT, uint32_t lgT,
                 uint32_t C, uint32_t lgnc, bool direct, hipStream_t s, Timer* tm) {
    Mark m(tm, s, K_SCAN_TILES);
    if (!direct)
        hipLaunchKernelGGL(k_tile_reduce, dim3(nT + 1), dim3(kBlock), 0, s, count, tflag, tsum, nT, lgT, C, lgnc);
    if (nT > kPrefixTiles) hipLaunchKernelGGL(k_scan_tiles, dim3(1), dim3(1024), 0, s, tsum, tprefix, nT + 1);
}
dim3 lane_grid(uint32_t n, int lanes) { return dim3(ceil_div(n > 0 ? n : 1u, 256u / (uint32_t)lanes)); }

template <bool kB>
hipError_t step_seq(const Bufs& b, const Scenes<kB>& SC, const Tuning& T, float* x, float* v, uint32_t n, int iters,
                    int any_xsph, int any_vort, uint32_t uw, hipStream_t s, Timer* tm, float4* qtape) {
    const uint32_t nb = ceil_div(n > 0 ? n : 1, 256);
    const uint32_t CT = b.CT;
    const uint32_t budget = (T.tile_cap * 3u) / 4u > 0 ? (T.tile_cap * 3u) / 4u : 1u;
    uint32_t lguw = 0;
    while ((1u << lguw) < uw) ++lguw;
    {
        Mark m(tm, s, K_PREDICT_HASH);
        hipLaunchKernelGGL(k_predict_hash<kB>, dim3(nb), dim3(256), 0, s, x, v, n, b, SC, b.key, b.rank, b.count, b.tflag,
                           b.lgT);
    }
    const bool direct = b.nT <= kDirectTiles;
    scan_totals(b.count, b.tsum, b.tflag, b.tprefix, b.nT, b.lgT, CT, 0u, direct, s, tm);
    {
        Mark m(tm, s, K_SCAN_CELLS);
        const EmitArgs E{uw, lguw, lguw, budget, b.units, &b.ctr[CTR_UNITS]};
        hipLaunchKernelGGL(k_scan_cells<EMIT_SEARCH>, dim3(b.nT + 1), dim3(kScanBlock), 0, s, b.count, b.offset,
                           totals_of(b.tsum, direct), b.tflag, prefix_of(b.tprefix, b.nT), b.nT, b.lgT, CT, 0u, E, b.ctr,
                           b.live);
    }
    if (n == 0) return hipGetLastError();
    {
        Mark m(tm, s, K_SCATTER);
        hipLaunchKernelGGL(k_scatter, dim3(nb), dim3(256), 0, s, b.key, b.rank, b.offset, b.tmp, n,
                           kB ? b.in_off + b.nscenes : (const uint32_t*)nullptr, b.big, &b.ctr[CTR_BIGCELLS], b.cap, b.bslot,
                           direct ? ClearArgs{b.count, b.tflag, CT + 1u, b.nT + 1u} : ClearArgs{});
        // the histogram ranks are dead after the scatter: their array holds the huge cells' chunks
        static_assert(CTR_HUGECELLS == CTR_BIGCELLS + 1, "the sort reads the two cell counts together");
        hipLaunchKernelGGL(k_sort_cells, dim3(256), dim3(1024), 0, s, b.offset, b.big, &b.ctr[CTR_BIGCELLS], b.tmp,
                           b.rank, b.cap);
        if (n > kSortMax)  // else no cell is huge
            hipLaunchKernelGGL(k_merge_huge, dim3(256), dim3(256), 0, s, b.offset, b.big, &b.ctr[CTR_BIGCELLS], b.tmp,
                               (const uint32_t*)b.rank, b.cap);
    }
    {
        Mark m(tm, s, K_REORDER);
        hipLaunchKernelGGL(k_reorder<kB>, dim3(nb), dim3(256), 0, s, x, v, b, SC, b.key, b.tmp, n);
    }
    {
        Mark m(tm, s, K_BIG_SEG);
        hipLaunchKernelGGL(k_big_seg<kB>, dim3(kBigBlocks), dim3(1024), 0, s, b, SC);
    }
    {
        Mark m(tm, s, K_NS);
        by_width(b.cap, [&](auto wide) {
            const uint32_t ng = ceil_div(n, kGroups);
            if (n <= kOneListMax) {
                hipLaunchKernelGGL((k_ns_groups<kB, wide(), true>), dim3(ng + stat_blocks(n)), dim3(kBlock), 0, s, b, SC,
                                   T.tile_cap, ng);
                return;
            }
            hipLaunchKernelGGL((k_ns_groups<kB, wide(), false>), dim3(ng + stat_blocks(n)), dim3(kBlock), 0, s, b, SC,
                               T.tile_cap, ng);
            hipLaunchKernelGGL((k_ns_big<kB, wide()>), big_grid(n), dim3(kBlock), 0, s, b, SC);
        });
    }
    for (int it = 0; it < iters; ++it) {
        Bufs bi = b;
        if (qtape) bi.Q = qtape + (size_t)it * b.cap;
        {
            Mark m(tm, s, K_LAMBDA);
            by_lanes(n, [&](auto L) {
                hipLaunchKernelGGL((k_lambda<kB, L()>), lane_grid(n, L()), dim3(256), 0, s, bi, SC);
            });
        }
        Mark m(tm, s, K_DELTAP);
        by_lanes(n, [&](auto L) {
            hipLaunchKernelGGL((k_deltap<kB, L()>), lane_grid(n, L()), dim3(256), 0, s, bi, SC);
        });
    }
    if (!any_vort && !any_xsph) {
        Mark m(tm, s, K_OUT);
        hipLaunchKernelGGL(k_out<kB>, dim3(nb), dim3(256), 0, s, b, SC, (const float4*)nullptr, x, v);
        return hipGetLastError();
    }
    // runs of at most eight final cells with four counters each (fewer in narrower
    // runs): CR counters, never more than CT, lgrun of them per work unit of uw
    // cells; scanned in tiles of up to 4096 that divide CR
    const uint32_t lgsub = std::min(lguw, 3u), lgnc = std::min(lgsub, 2u);
    const uint32_t lgrun = lgnc + lguw - lgsub, CR = (CT >> lguw) << lgrun;
    uint32_t lgTr = 0;
    while (lgTr < 12u && ((CR >> (lgTr + 1)) << (lgTr + 1)) == CR && (1u << (lgTr + 1)) <= CR) ++lgTr;
    const uint32_t nTr = CR >> lgTr;
    {
        Mark m(tm, s, K_CUR_SORT);
        hipLaunchKernelGGL(k_cur_hash<kB>, dim3(nb), dim3(256), 0, s, b, SC, lgsub, lgnc, lgTr, CR);
        const bool direct = nTr <= kDirectTiles;
        scan_totals(b.ccount, b.ctsum, b.ctflag, b.ctprefix, nTr, lgTr, CR, lgnc, direct, s, nullptr);
        const EmitArgs E{uw, lguw, lgrun, 0u, b.cunits, &b.ctr[CTR_CUNITS]};
        hipLaunchKernelGGL(k_scan_cells<EMIT_FINAL>, dim3(nTr + 1), dim3(kScanBlock), 0, s, b.ccount, b.coffset,
                           totals_of(b.ctsum, direct), b.ctflag, prefix_of(b.ctprefix, nTr), nTr, lgTr, CR, lgnc, E,
                           (uint32_t*)nullptr, (uint32_t*)nullptr);
        hipLaunchKernelGGL(k_cur_scatter, dim3(nb), dim3(256), 0, s, b.offset, CT, b.ckey, b.crank, b.coffset, b.cperm,
                           b.oslot, direct ? ClearArgs{b.ccount, b.ctflag, CR + 1u, nTr + 1u} : ClearArgs{});
    }
    {
        Mark m(tm, s, K_FINAL_LIST);
        by_width(b.cap, [&](auto wide) {
            const uint32_t ng = ceil_div(n, kGroups);
            if (n <= kOneListMax) {
                hipLaunchKernelGGL((k_final_groups<kB, wide(), true>), dim3(ng + stat_blocks(n)), dim3(kBlock), 0, s, b, SC,
                                   kFinalTile, lguw, lgrun, ng);
                return;
            }
            hipLaunchKernelGGL((k_final_groups<kB, wide(), false>), dim3(ng + stat_blocks(n)), dim3(kBlock), 0, s, b, SC,
                               kFinalTile, lguw, lgrun, ng);
            hipLaunchKernelGGL((k_final_big<kB, wide()>), big_grid(n), dim3(kBlock), 0, s, b, SC);
        });
    }
    // the overflow positions' per-cell partials, before each pass that adds them
    auto ovf_part = [&](auto pass) {
        hipLaunchKernelGGL((k_ovf_part<kB, pass()>), dim3(ovf_blocks(n)), dim3(256), 0, s, b, SC);
    };
    if (any_vort) {
        {
            Mark m(tm, s, K_VORT);
            ovf_part(std::integral_constant<int, PASS_VORT>{});
            by_lanes(n, [&](auto L) {
                hipLaunchKernelGGL((k_vort<kB, L()>), lane_grid(n, L()), dim3(kBlock), 0, s, b, SC);
            });
        }
        Mark m(tm, s, K_CONFINE);
        ovf_part(std::integral_constant<int, PASS_CONF>{});
        by_lanes(n, [&](auto L) {
            hipLaunchKernelGGL((k_confine<kB, L()>), lane_grid(n, L()), dim3(kBlock), 0, s, b, SC);
        });
    }
    if (any_xsph) {
        Mark m(tm, s, K_XSPH_OUT);
        ovf_part(std::integral_constant<int, PASS_XSPH>{});
        by_lanes(n, [&](auto L) {
            hipLaunchKernelGGL((k_xsph_out<kB, L()>), lane_grid(n, L()), dim3(kBlock), 0, s, b, SC, x, v);
        });
    } else {
        Mark m(tm, s, K_OUT);
        hipLaunchKernelGGL(k_out<kB>, dim3(nb), dim3(256), 0, s, b, SC, (const float4*)b.R, x, v);
    }
    return hipGetLastError();
}

}  // namespace

hipError_t launch_step(const Bufs& b, const Scene& s0, const Tuning& T, float* x, float* v, uint32_t n, int iters,
                       int any_xsph, int any_vort, uint32_t uw, hipStream_t s, Timer* tm, float4* qtape) {
    if (b.nscenes == 1) {
        const Scenes<false> SC{b.scenes, s0};
        return step_seq<false>(b, SC, T, x, v, n, iters, any_xsph, any_vort, uw, s, tm, qtape);
    }
    if (qtape) return hipErrorInvalidValue;
    const Scenes<true> SC{b.scenes, s0};
    return step_seq<true>(b, SC, T, x, v, n, iters, any_xsph, any_vort, uw, s, tm, nullptr);
}

hipError_t launch_count_scan(uint32_t* count, uint32_t* offset, uint32_t* tsum, uint32_t* tflag, uint32_t* tprefix,
                             uint32_t nT, uint32_t lgT, uint32_t C, hipStream_t s) {
    scan_totals(count, tsum, tflag, tprefix, nT, lgT, C, 0u, false, s, nullptr);
    hipLaunchKernelGGL(k_scan_cells<EMIT_NONE>, dim3(nT + 1), dim3(kScanBlock), 0, s, count, offset, tsum, tflag,
                       prefix_of(tprefix, nT), nT, lgT, C, 0u, EmitArgs{}, (uint32_t*)nullptr, (uint32_t*)nullptr);
    return hipGetLastError();
}

hipError_t launch_scene_offsets(const Bufs& b, uint32_t* out, hipStream_t s) {
    hipLaunchKernelGGL(k_scene_offsets, dim3(ceil_div(b.nscenes + 1u, 256)), dim3(256), 0, s, b, out);
    return hipGetLastError();
}

hipError_t launch_neighbors_view(const Bufs& b, uint32_t* out, uint32_t* counts, uint32_t max_pair, hipStream_t s) {
    hipLaunchKernelGGL(k_neighbors_view, dim3(ceil_div(b.cap > 0 ? b.cap : 1, 256)), dim3(256), 0, s, b, out, counts,
                       max_pair);
    return hipGetLastError();
}

hipError_t launch_cell_ranges(const Bufs& b, uint32_t C, uint32_t* start, uint32_t* end, hipStream_t s) {
    hipLaunchKernelGGL(k_cell_ranges, dim3(ceil_div(C, 256)), dim3(256), 0, s, b.offset, C, start, end);
    return hipGetLastError();
}

hipError_t launch_copy_lambda(const Bufs& b, float* out, hipStream_t s) {
    hipLaunchKernelGGL(k_copy_lambda, dim3(ceil_div(b.cap > 0 ? b.cap : 1, 256)), dim3(256), 0, s, b.offset, b.CT,
                       (const float4*)b.Q, out);
    return hipGetLastError();
}

hipError_t launch_sort_cells(const uint32_t* offset, const uint32_t* cells, const uint32_t* ncells, uint32_t* vals,
                             uint32_t* scratch, uint32_t cap, hipStream_t s) {
    hipLaunchKernelGGL(k_sort_cells, dim3(256), dim3(1024), 0, s, offset, cells, ncells, vals, scratch, cap);
    hipLaunchKernelGGL(k_merge_huge, dim3(256), dim3(256), 0, s, offset, cells, ncells, vals,
                       (const uint32_t*)scratch, cap);
    return hipGetLastError();
}

hipError_t launch_density(const Bufs& b, const Scene& s0, const float* x, float* rho, hipStream_t s) {
    const dim3 g(ceil_div(b.cap > 0 ? b.cap : 1, 256));
    if (b.nscenes == 1) {
        const Scenes<false> SC{b.scenes, s0};
        hipLaunchKernelGGL(k_density<false>, g, dim3(256), 0, s, b, SC, x, rho);
    } else {
        const Scenes<true> SC{b.scenes, s0};
        hipLaunchKernelGGL(k_density<true>, g, dim3(256), 0, s, b, SC, x, rho);
    }
    return hipGetLastError();
}

hipError_t launch_restore(const Bufs& b, const float* xs, const float* vs, float* xo, float* vo, hipStream_t s) {
    hipLaunchKernelGGL(k_restore, dim3(ceil_div(b.cap > 0 ? b.cap : 1, 256)), dim3(256), 0, s, b, xs, vs, xo, vo);
    return hipGetLastError();
}

hipError_t launch_selftest_inv_sqrt(uint32_t lo, uint32_t hi, unsigned long long* mismatches, uint32_t* first,
                                    hipStream_t s) {
    hipLaunchKernelGGL(k_selftest_inv_sqrt, dim3(16384), dim3(256), 0, s, lo, hi, mismatches, first);
    return hipGetLastError();
}

hipError_t launch_clear_counts(const Bufs& b, hipStream_t s) {
    hipLaunchKernelGGL(k_clear_counts, dim3(std::min(1024u, ceil_div(b.CT + 1u, 256u))), dim3(256), 0, s,
                       ClearArgs{b.count, b.tflag, b.CT + 1u, b.nT + 1u}, ClearArgs{b.ccount, b.ctflag, b.CT + 1u, b.nT + 1u});
    return hipGetLastError();
}

hipError_t launch_selftest(const float* a, const float* bb, float* out, uint32_t n, hipStream_t s) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_selftest, dim3(ceil_div(n, 256)), dim3(256), 0, s, a, bb, out, n);
    return hipGetLastError();
}

}  // namespace pbfx
