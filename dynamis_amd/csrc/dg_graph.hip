// dg_graph.hip -- PBC radius-graph build for gfx950 (MI355X), C ABI in
// include/dynamis_graph.h.
//
// Pipeline of one build (all on the caller's stream, one host sync in the Python layer
// to size the outputs, none inside this file):
//   1. tile_rank                   Morton (SFC) rank of every tile of bins
//   2. bin_atoms                   fractional coords -> floor (wrap), bin, SFC key, and the
//                                  atom's cell-list record
//   3-5. tile_hist, tile_scatter, tile_sort   counting sort into the cell list: fp32 position
//                                  relative to the bin origin + id, packed floor, in SFC order
//   6. search<0>                   per-target degree and row words (one workgroup per tile,
//                                  region of (T+2P)^3 bins staged in LDS, one lane per target),
//                                  and the tile's region map
//   7. scan                        per-tile edge offsets in SFC tile order
//   8. expand, search<1>           edges: row words decoded into LDS, then streamed out with
//                                  16-byte stores; the few tiles the count flagged swept again
//
// Reference stages replaced (dynamis_state/src/csrc/graph/radius_graph_kernels.cu):
// wrap :596-605, selective images :18-141 (here: periodic bin wrap, no image atoms),
// grid + sort :146-194,662-714, target sort :731-769, count :197-258, write :320-442,
// outputs :925-933.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <mutex>
#include <string>
#include <type_traits>
#include <utility>
#include <vector>

#include "../../include/dynamis_graph.h"
#include "dg_common.hpp"
#include "dg_plan.hpp"
#include "dg_scan.hpp"
#include "dg_segsort.hpp"

namespace dg {

thread_local std::string g_last_error;

dg_status fail(dg_status st, const std::string& msg)
{
    g_last_error = msg;
    return st;
}

constexpr int kRegPerThread = (kMaxRegion + kBlock - 1) / kBlock;
constexpr int kBinSortMax = 128;

// Whether a device-wide flag word still reads 0 (a device-scope load, so a flag another
// XCD set is seen): raising flags only then keeps the atomics on one address few.
__device__ __forceinline__ bool flag_clear(int64_t* w)
{
    return __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0;
}

// search_kernel<1> work of a tile, set by the count pass
constexpr int kFixOver = 1;     // a target has more row words than its list holds
constexpr int kFixChunked = 2;  // no row words: the region needs more than two LDS chunks, the
                                // region map is full, or the count recorded none
#ifndef DG_FIXGRID
#define DG_FIXGRID 512
#endif
constexpr int64_t kFixGrid = DG_FIXGRID;  // workgroups of the fix-up pass (it loops over the tiles)

// Value known to be uniform across the wave, moved to a scalar register.
__device__ __forceinline__ int rfl(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ uint32_t rfl(uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); }

__device__ __forceinline__ void load_pos(const void* pos, int f64, int64_t i, double* p)
{
    if (f64) {
        const double* q = (const double*)pos + 3 * i;
        p[0] = q[0]; p[1] = q[1]; p[2] = q[2];
    } else {
        const float* q = (const float*)pos + 3 * i;
        p[0] = q[0]; p[1] = q[1]; p[2] = q[2];
    }
}

struct GridArgs {
    double C[9], Cinv[9];
    int nb[3], T[3], ntl[3], mb[3];
    int tb;
};

// Offset of a cell-list record along the cell's a axis inside its bin, as a Cartesian x
// length (lower-triangular cells): x less the b and c shears of its y and z offsets, so the
// key is fa * hax for the record's fraction fa of the bin along a.  The tile sort orders
// bins by it and the count pass counts quarter-bin prefixes of it: both evaluate it with
// these explicit operations on the same inputs, so the counts are prefixes of the order.
struct XKey {
    float hbx, hcx, hcy, inv_hby, inv_hcz;
};
__device__ __forceinline__ float bin_xkey(const float4& e, const XKey& k)
{
    const float fc = e.z * k.inv_hcz;
    const float fb = fmaf(-fc, k.hcy, e.y) * k.inv_hby;
    return fmaf(-fc, k.hcx, fmaf(-fb, k.hbx, e.x));
}

// ---------------------------------------------------------------- tile SFC ranks
// Rank of every tile in the compact Morton order (morton_encode) among the tiles of the
// grid, computed directly: for each 1 bit of the tile's code, the tiles whose codes share
// the bits above it and have a 0 there all come first; per axis, their coordinate has its
// high bits fixed and f free low bits, so the axis admits clamp(n - lo, 0, 2^f) values.
// Also clears the bin counts (bcnt) for the binning that follows.
__global__ void tile_rank_kernel(GridArgs g, int64_t ntiles, int* __restrict__ tile_of_rank,
                                 int* __restrict__ rank_of_tile, int* __restrict__ bcnt,
                                 int64_t nbins, int64_t* __restrict__ totals, int64_t* __restrict__ tbase)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    if (blockIdx.x == 0 && threadIdx.x < 8) totals[threadIdx.x] = 0;  // the build's totals and flags
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < nbins; q += stride) bcnt[q] = 0;
    for (int64_t lin = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; lin < ntiles; lin += stride) {
        tbase[lin] = 0;  // (the cursors of the region map lie there until the tiles are counted)
        const int X[3] = {(int)(lin % g.ntl[0]), (int)((lin / g.ntl[0]) % g.ntl[1]),
                          (int)(lin / ((int64_t)g.ntl[0] * g.ntl[1]))};
        int f[3] = {0, 0, 0};
        int64_t r = 0;
        const int top = max(max(g.mb[0], g.mb[1]), g.mb[2]);
        for (int k = 0; k < top; ++k) {
            for (int dp = 0; dp < 3; ++dp) {
                if (k >= g.mb[dp]) continue;
                if ((X[dp] >> k) & 1) {
                    int64_t cnt = 1;
#pragma unroll
                    for (int d = 0; d < 3; ++d) {
                        const int lo = d == dp ? (X[d] >> (k + 1)) << (k + 1) : (X[d] >> f[d]) << f[d];
                        cnt *= (int64_t)min(max(g.ntl[d] - lo, 0), 1 << f[d]);
                    }
                    r += cnt;
                }
                ++f[dp];
            }
        }
        tile_of_rank[r] = (int)lin;
        rank_of_tile[lin] = (int)r;
    }
}

// ---------------------------------------------------------------- binning
// Canonical wrap of one atom: floor of the fractional coordinate (all axes, as the
// reference, radius_graph_kernels.cu:603-605), wrapped fraction s in [0,1) and bin b.
__device__ __forceinline__ int wrap_atom(const GridArgs& g, const double* p, int* f, double* s,
                                         int* b)
{
    int st = 0;
    double q[3] = {p[0], p[1], p[2]};
    if (!(isfinite(q[0]) && isfinite(q[1]) && isfinite(q[2]))) {
        st |= kStatusNonFinite;
        q[0] = q[1] = q[2] = 0.0;
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        double fr = canon_frac(q[0], q[1], q[2], g.Cinv, j);
        double fl = floor(fr);
        if (!(fabs(fl) <= (double)kFloorMax)) {
            st |= kStatusRange;
            fl = 0.0;
            fr = 0.0;
        }
        f[j] = (int)fl;
        s[j] = fr - fl;
        int bj = (int)(s[j] * (double)g.nb[j]);
        b[j] = bj < 0 ? 0 : (bj >= g.nb[j] ? g.nb[j] - 1 : bj);
    }
    return st;
}

__device__ __forceinline__ uint32_t bin_key(const GridArgs& g, const int* b,
                                            const int* __restrict__ rank_of_tile)
{
    int t0 = b[0] / g.T[0], t1 = b[1] / g.T[1], t2 = b[2] / g.T[2];
    int l0 = b[0] - t0 * g.T[0], l1 = b[1] - t1 * g.T[1], l2 = b[2] - t2 * g.T[2];
    int lin = t0 + g.ntl[0] * (t1 + g.ntl[1] * t2);
    return (uint32_t)rank_of_tile[lin] * (uint32_t)g.tb + (uint32_t)(l0 + g.T[0] * (l1 + g.T[1] * l2));
}

// Per atom: wrap, bin, SFC key and an atomic slot inside the key's bin; and the atom's
// cell-list record (fp32 position relative to its bin origin, packed floor), which
// finish_bins moves to the atom's sorted place.
__global__ void bin_atoms_kernel(GridArgs g, const void* __restrict__ pos, int f64, int64_t n,
                                 const int* __restrict__ rank_of_tile, uint32_t* __restrict__ key,
                                 uint32_t* __restrict__ rank, int* __restrict__ bcnt,
                                 float4* __restrict__ rec, int64_t* __restrict__ totals)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double p[3], s[3];
    int f[3], b[3];
    load_pos(pos, f64, i, p);
    int st = wrap_atom(g, p, f, s, b);
    if (st) atomicOr((unsigned long long*)&totals[1], (unsigned long long)st);
    uint32_t k = bin_key(g, b, rank_of_tile);
    key[i] = k;
    if (bcnt) rank[i] = (uint32_t)atomicAdd(&bcnt[k], 1);
    // position relative to the bin origin: (s - b/nb) . C
    double o[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) o[d] = s[d] - (double)b[d] / (double)g.nb[d];
    float4 e;
    e.x = (float)fma(o[2], g.C[6], fma(o[1], g.C[3], o[0] * g.C[0]));
    e.y = (float)fma(o[2], g.C[7], fma(o[1], g.C[4], o[0] * g.C[1]));
    e.z = (float)fma(o[2], g.C[8], fma(o[1], g.C[5], o[0] * g.C[2]));
    e.w = __uint_as_float(pack3(f[0], f[1], f[2]));
    rec[i] = e;
}

__global__ void scatter_atoms_kernel(int64_t n, const uint32_t* __restrict__ key,
                                     const uint32_t* __restrict__ rank,
                                     const int* __restrict__ bstart, int* __restrict__ sid)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    sid[bstart[key[i]] + rank[i]] = (int)i;
}

// Insertion sort of a[lo, hi) ascending (bins hold a handful of entries).
__device__ __forceinline__ void small_sort(int* a, int lo, int hi)
{
    for (int j = lo + 1; j < hi; ++j) {
        int v = a[j];
        int k = j - 1;
        while (k >= lo && a[k] > v) {
            a[k + 1] = a[k];
            --k;
        }
        a[k + 1] = v;
    }
}

// Sorts every segment [start[b], start[b + 1]) of v longer than kBinSortMax (by value,
// ascending; ids < 2^31) in place, tmp its scratch: the bins that order_atoms_kernel and
// finish_targets_kernel leave as they are.  Workgroup g scans its own range of segments,
// 256 at a time, and sorts the long ones of each batch in turn.
__global__ __launch_bounds__(kSegSortThreads) void sort_big_bins_kernel(int64_t nseg, const int* __restrict__ start,
                                                                        uint32_t* __restrict__ v,
                                                                        uint32_t* __restrict__ tmp)
{
    __shared__ SegSortLds L;
    __shared__ int big[kSegSortThreads];
    const int64_t per = (nseg + gridDim.x - 1) / gridDim.x;
    const int64_t b0 = (int64_t)blockIdx.x * per, b1 = min(nseg, b0 + per);
    for (int64_t c = b0; c < b1; c += kSegSortThreads) {
        const int64_t b = c + threadIdx.x;
        big[threadIdx.x] = b < b1 && start[b + 1] - start[b] > kBinSortMax;
        __syncthreads();
        for (int k = 0; k < kSegSortThreads; ++k) {
            if (!big[k]) continue;  // (the same for every thread)
            const int lo = start[c + k], hi = start[c + k + 1];
            segment_sort<uint32_t>(v + lo, tmp + lo, hi - lo, 32, L);
        }
        __syncthreads();
    }
}

// One thread per cell-list entry j (in arrival order inside its bin, from scatter_atoms):
// the entry's place in its bin ordered by atom id (the number of smaller ids in the bin),
// then the SoA cell list.  Bins of more than kBinSortMax atoms were put in id order by
// sort_big_bins_kernel already: there the place is j.
__global__ void order_atoms_kernel(int64_t n, const uint32_t* __restrict__ key,
                                   const int* __restrict__ bstart, const int* __restrict__ arr,
                                   const float4* __restrict__ rec, float4* __restrict__ spos,
                                   uint32_t* __restrict__ sflr, int* __restrict__ sid,
                                   int* __restrict__ inv)
{
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const int i = arr[j];
    const uint32_t b = key[i];
    const int lo = bstart[b], hi = bstart[b + 1];
    int d = (int)j;
    if (hi - lo > 1 && hi - lo <= kBinSortMax) {
        int below = 0;
        for (int m = lo; m < hi; ++m) below += arr[m] < i;
        d = lo + below;
    }
    const float4 r = rec[i];
    spos[d] = make_float4(r.x, r.y, r.z, __int_as_float(i));
    sflr[d] = __float_as_uint(r.w);
    sid[d] = i;
    if (inv) inv[i] = d;
}

// ---------------------------------------------------------------- tile-level counting sort
// Without per-atom device atomics (about 25 G/s on this part, the dominant cost of a
// per-bin counting sort): kSortChunks workgroups each histogram the tiles of one chunk of
// atoms in LDS and reserve their share of every tile with one device atomic per tile;
// the same chunks then place their atoms into tile buckets; one workgroup per tile then
// orders its bucket by (bin, offset along the a axis in the bin for lower-triangular cells,
// atom id) in LDS and writes the bin starts and the cell list.

// Chunk c of the atoms: [c n / G, (c + 1) n / G).
__device__ __forceinline__ void sort_chunk(int64_t n, int64_t* lo, int64_t* hi)
{
    *lo = n * blockIdx.x / gridDim.x;
    *hi = n * (blockIdx.x + 1) / gridDim.x;
}

__global__ __launch_bounds__(1024) void tile_hist_kernel(int64_t n, int tb, int64_t ntiles,
                                                         const uint32_t* __restrict__ key,
                                                         int* __restrict__ tcnt, int* __restrict__ wgb,
                                                         const int64_t* __restrict__ run_if)
{
    if (run_if && *run_if == 0) return;  // (explicit targets that need no sort)
    extern __shared__ int h[];
    for (int64_t r = threadIdx.x; r < ntiles; r += blockDim.x) h[r] = 0;
    __syncthreads();
    int64_t lo, hi;
    sort_chunk(n, &lo, &hi);
    for (int64_t i = lo + threadIdx.x; i < hi; i += blockDim.x) atomicAdd(&h[key[i] / (uint32_t)tb], 1);
    __syncthreads();
    for (int64_t r = threadIdx.x; r < ntiles; r += blockDim.x) {
        const int c = h[r];
        wgb[blockIdx.x * ntiles + r] = c ? atomicAdd(&tcnt[r], c) : 0;
    }
}

// Places every atom of the chunk in its tile's bucket as (atom id, bin inside the tile);
// the atoms are read in order, the scattered side is the 8-byte stores.
// Each workgroup scans the tile totals itself (workgroup 0 also stores the tile starts,
// with tstart[ntiles] = n, for tile_sort_kernel).
// A tile-bucket entry: an id and the bin inside the tile (< 256).  32 bits (24 + 8) when
// every id fits 24 bits, else 64 (32 + 32).
__device__ __forceinline__ uint32_t bk_pack(uint32_t i, uint32_t l, uint32_t*) { return i | (l << 24); }
__device__ __forceinline__ uint64_t bk_pack(uint32_t i, uint32_t l, uint64_t*) { return (uint64_t)i | ((uint64_t)l << 32); }
__device__ __forceinline__ int bk_id(uint32_t w) { return (int)(w & 0xFFFFFFu); }
__device__ __forceinline__ int bk_id(uint64_t w) { return (int)(uint32_t)w; }
__device__ __forceinline__ int bk_bin(uint32_t w) { return (int)(w >> 24); }
__device__ __forceinline__ int bk_bin(uint64_t w) { return (int)(w >> 32); }

template <typename BT>
__global__ __launch_bounds__(1024) void tile_scatter_kernel(int64_t n, int tb, int64_t ntiles,
                                                            const uint32_t* __restrict__ key,
                                                            const int* __restrict__ tcnt,
                                                            int* __restrict__ tstart,
                                                            const int* __restrict__ wgb,
                                                            BT* __restrict__ bucket,
                                                            const int64_t* __restrict__ run_if)
{
    if (run_if && *run_if == 0) return;  // (explicit targets that need no sort)
    extern __shared__ int h[];  // this chunk's next place in every tile's bucket
    __shared__ int s_w[1024 / 64];
    {
        const int per = (int)((ntiles + 1023) / 1024);
        const int64_t r0 = (int64_t)threadIdx.x * per;
        int loc = 0;
        for (int k = 0; k < per; ++k)
            if (r0 + k < ntiles) loc += tcnt[r0 + k];
        int tot;
        int ex = block_excl_scan<int, 1024>(loc, s_w, &tot);
        for (int k = 0; k < per; ++k) {
            const int64_t r = r0 + k;
            if (r < ntiles) {
                h[r] = ex + wgb[blockIdx.x * ntiles + r];
                if (blockIdx.x == 0) tstart[r] = ex;
                ex += tcnt[r];
            }
        }
        if (blockIdx.x == 0 && threadIdx.x == 0) tstart[ntiles] = tot;
    }
    __syncthreads();
    int64_t lo, hi;
    sort_chunk(n, &lo, &hi);
    // four atoms per thread and step, their loads issued together
    for (int64_t i0 = lo + threadIdx.x; i0 < hi; i0 += 4 * (int64_t)blockDim.x) {
        uint32_t k[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int64_t i = i0 + (int64_t)u * blockDim.x;
            k[u] = i < hi ? key[i] : 0u;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int64_t i = i0 + (int64_t)u * blockDim.x;
            if (i < hi) {
                const uint32_t r = k[u] / (uint32_t)tb;
                const int d = atomicAdd(&h[r], 1);
                bucket[d] = bk_pack((uint32_t)i, k[u] - r * (uint32_t)tb, (BT*)nullptr);
            }
        }
    }
}

constexpr int kTileSortCap = 2048;  // bucket entries ordered in LDS (larger: sorted by segment_sort)
constexpr int kTileSortPer = kTileSortCap / 256;
struct TileSortLds {
    union {
        int by[kTileSortCap];  // ids grouped by bin
        SegSortLds seg;        // a larger bucket: sorted in global memory
    };
    uint32_t bx[kTileSortCap];  // atoms: order key of each grouped entry's x in its bin
    int cnt[kTileMax * kTileMax * kTileMax];
    int st[kTileMax * kTileMax * kTileMax + 1];
    int w32[4];
};

// What tile_sort_kernel writes for one sorted entry.  Atoms (TGT false): the cell-list
// record (position in the bin and id, floor, id, and the inverse map); ids are atom ids.
// Explicit targets (TGT true): ids are caller positions t; the caller position and the
// cell-list index of target t's atom.
struct TileSortOut {
    const float4* rec;  // atoms: records by atom id
    float4* spos;
    uint32_t* sflr;
    int* sid;
    int* inv;           // atoms: written when given; targets: read (atom -> cell-list index)
    const int64_t* tgt; // targets: atom of each caller position
    int64_t natoms;
    int* tslot;
    int* tsidx;
    const int64_t* run_if;  // targets: skipped when *run_if == 0 (they need no sort)
    void* stmp;             // scratch for a bucket of more than kTileSortCap entries (one per entry)
    int64_t* xflag;         // atoms: raised when a bucket's bins are left in id order
    int xorder;             // atoms: order bins by (bin_xkey, id) (else by id)
    XKey xk;
};

// Order key of a float: unsigned compare of the keys is the float order (-0 below +0).
__device__ __forceinline__ uint32_t float_order_key(float x)
{
    const uint32_t u = __float_as_uint(x);
    return u ^ ((uint32_t)((int32_t)u >> 31) | 0x80000000u);
}

// One workgroup per tile: orders its bucket by bin, writes the tile's bin starts and its
// part of the sorted list.  Inside a bin, atoms go by (x relative to the bin origin, id),
// so that the count pass can cut a stencil row's end bins at quarter-bin x boundaries;
// explicit targets go by caller position.  A bucket too large for LDS is ordered by (bin,
// id) and raises *xflag (the count pass then uses whole bins).  Each entry's payload is
// gathered into registers as soon as its id is known, so the gathers overlap the ordering
// in LDS.
template <bool TGT, typename BT>
__global__ __launch_bounds__(256) void tile_sort_kernel(int64_t n, int tb, int64_t ntiles,
                                                        const int* __restrict__ tstart,
                                                        BT* __restrict__ bucket,
                                                        int* __restrict__ bstart, TileSortOut o)
{
    if (o.run_if && *o.run_if == 0) return;
    __shared__ TileSortLds S;
    typedef typename std::conditional<TGT, int, float4>::type Pay;
    auto gather = [&](int i) -> Pay {
        if constexpr (TGT) {
            int64_t at = o.tgt[i];
            at = at < 0 || at >= o.natoms ? 0 : at;  // (out of range: flagged by target_keys_kernel)
            return o.inv[at];
        } else {
            return o.rec[i];
        }
    };
    const int64_t r = blockIdx.x;
    const int base = tstart[r], m = tstart[r + 1] - base;
    const bool fits = m <= kTileSortCap;
    for (int l = threadIdx.x; l < tb; l += 256) S.cnt[l] = 0;
    __syncthreads();
    Pay q[kTileSortPer];
    int qi[kTileSortPer], ql[kTileSortPer];
#pragma unroll
    for (int u = 0; u < kTileSortPer; ++u) {
        const int e = threadIdx.x + 256 * u;
        qi[u] = -1;
        if (fits && e < m) {
            const BT w = bucket[base + e];
            qi[u] = bk_id(w);
            ql[u] = bk_bin(w);
            q[u] = gather(qi[u]);
            atomicAdd(&S.cnt[ql[u]], 1);
        }
    }
    if (!fits)
        for (int e = threadIdx.x; e < m; e += 256) atomicAdd(&S.cnt[bk_bin(bucket[base + e])], 1);
    __syncthreads();
    // bin starts inside the bucket (tb <= 216: one pass of a 256-thread scan)
    {
        const int c = (int)threadIdx.x < tb ? S.cnt[threadIdx.x] : 0;
        int tot;
        const int ex = block_excl_scan<int, 256>(c, S.w32, &tot);
        if ((int)threadIdx.x < tb) {
            S.st[threadIdx.x] = ex;
            S.cnt[threadIdx.x] = ex;  // placement cursors
            bstart[r * tb + threadIdx.x] = base + ex;
        }
        if (threadIdx.x == 0) {
            S.st[tb] = tot;
            if (r == ntiles - 1) bstart[ntiles * tb] = (int)n;
        }
    }
    __syncthreads();
    auto emit = [&](int d, int i, Pay v) {
        if constexpr (TGT) {
            o.tslot[d] = i;
            o.tsidx[d] = v;
        } else {
            o.spos[d] = make_float4(v.x, v.y, v.z, __int_as_float(i));
            o.sflr[d] = __float_as_uint(v.w);
            o.sid[d] = i;
            if (o.inv) o.inv[i] = d;
        }
    };
    if (!fits) {
        // a very dense tile: the bucket sorted by (bin, id) in global memory (an entry's
        // bin sits above its id), then each entry goes to its place
        if constexpr (!TGT)
            if (o.xorder && threadIdx.x == 0 && flag_clear(o.xflag))
                atomicOr((unsigned long long*)o.xflag, 1ull);
        segment_sort<BT>(bucket + base, (BT*)o.stmp + base, m, sizeof(BT) == 4 ? 32 : 40, S.seg);
        for (int e = threadIdx.x; e < m; e += 256) {
            const int i = bk_id(bucket[base + e]);
            emit(base + e, i, gather(i));
        }
        return;
    }
    uint32_t qx[kTileSortPer];
#pragma unroll
    for (int u = 0; u < kTileSortPer; ++u) {
        qx[u] = 0;
        if constexpr (!TGT)
            if (qi[u] >= 0 && o.xorder) qx[u] = float_order_key(bin_xkey(q[u], o.xk));
        if (qi[u] >= 0) {
            const int d = atomicAdd(&S.cnt[ql[u]], 1);
            S.by[d] = qi[u];
            S.bx[d] = qx[u];
        }
    }
    __syncthreads();
    // each entry's place in its bin: the number of entries there with a smaller (x, id)
    // (targets, and atoms without xorder: x keys all 0, so by id)
#pragma unroll
    for (int u = 0; u < kTileSortPer; ++u) {
        if (qi[u] < 0) continue;
        const int i = qi[u], l = ql[u];
        const uint32_t x = qx[u];
        int below = 0;
        for (int k = S.st[l]; k < S.st[l + 1]; ++k) {
            const uint32_t xk = S.bx[k];
            below += (xk < x) | ((xk == x) & (S.by[k] < i));
        }
        emit(base + S.st[l] + below, i, q[u]);
    }
}

// ---------------------------------------------------------------- explicit targets
// Bin key of every target's atom (tile-level sort of the targets); out-of-range targets
// are flagged and take atom 0.  Also clears the tile totals for the targets' histogram.
__global__ void target_keys_kernel(int64_t nt, int64_t n, const int64_t* __restrict__ tgt,
                                   const uint32_t* __restrict__ key, uint32_t* __restrict__ tkey,
                                   int* __restrict__ tcnt, int64_t ntiles, int64_t* __restrict__ totals)
{
    if (totals[2] == 0) return;  // the targets are 0 .. nt - 1: no sort (target_prefix_kernel)
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (int64_t r = i0; r < ntiles; r += stride) tcnt[r] = 0;
    for (int64_t t = i0; t < nt; t += stride) {
        int64_t a = tgt[t];
        if (a < 0 || a >= n) {
            atomicOr((unsigned long long*)&totals[1], (unsigned long long)DG_FLAG_TARGET);
            a = 0;
        }
        tkey[t] = key[a];
    }
}

// Raises totals[2] unless the explicit targets are exactly 0, 1, ..., nt - 1 with nt <= n
// (then the count takes the atoms of each tile with ids < nt as its targets, in cell-list
// order, with no target sort).  totals[2] was cleared by tile_rank_kernel.
__global__ void target_prefix_kernel(int64_t nt, int64_t n, const int64_t* __restrict__ tgt,
                                     int64_t* __restrict__ totals)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    bool other = nt > n;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < nt && !other; t += stride)
        other = tgt[t] != t;
    // one device atomic per workgroup at most, and none once the flag is seen set (atomics
    // on one address serialise: one per wave of a large list costs tens of microseconds)
    __shared__ int s_w[256 / 64];
    if (block_any<256>(other, s_w) && threadIdx.x == 0 && flag_clear(&totals[2]))
        atomicOr((unsigned long long*)&totals[2], 1ull);
}

__global__ void bin_targets_kernel(int64_t nt, int64_t n, const int64_t* __restrict__ tgt,
                                   const uint32_t* __restrict__ key, uint32_t* __restrict__ tkey,
                                   uint32_t* __restrict__ trank, int* __restrict__ tbcnt,
                                   int64_t* __restrict__ totals)
{
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nt) return;
    int64_t a = tgt[t];
    if (a < 0 || a >= n) {
        atomicOr((unsigned long long*)&totals[1], (unsigned long long)DG_FLAG_TARGET);
        a = 0;
    }
    uint32_t k = key[a];
    tkey[t] = k;
    trank[t] = (uint32_t)atomicAdd(&tbcnt[k], 1);
}

__global__ void scatter_targets_kernel(int64_t nt, const uint32_t* __restrict__ tkey,
                                       const uint32_t* __restrict__ trank,
                                       const int* __restrict__ tbstart, int* __restrict__ tslot)
{
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nt) return;
    tslot[tbstart[tkey[t]] + trank[t]] = (int)t;
}

__global__ void finish_targets_kernel(int64_t nbins, int64_t n, const int* __restrict__ tbstart,
                                      int* __restrict__ tslot, const int64_t* __restrict__ tgt,
                                      const int* __restrict__ inv, int* __restrict__ tsidx)
{
    int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= nbins) return;
    int lo = tbstart[q], hi = tbstart[q + 1];
    if (hi - lo > 1 && hi - lo <= kBinSortMax) small_sort(tslot, lo, hi);
    for (int j = lo; j < hi; ++j) {
        int64_t a = tgt[tslot[j]];
        if (a < 0 || a >= n) a = 0;
        tsidx[j] = inv[a];
    }
}

// ---------------------------------------------------------------- neighbour search
struct SearchArgs {
    double C[9];
    double Cinv[9];
    double hC[9];  // bin step vectors: row d = C[d] / nb[d]
    double r2;
    int lowtri;    // lower-triangular cell (a along x, b in the xy plane, positive diagonal):
                   // stencil rows are trimmed to the padded cutoff sphere; 2: orthorhombic
    float hax, hbx, hby, hcx, hcy, hcz;  // bin step vectors C[d] / nb[d] (lower triangle)
    float rprune2, pmargin;
    float gy_off, gz_off;             // -hby - pmargin, -hcz - pmargin (orthorhombic rows)
    float inv_hax, inv_hby, inv_hcz;  // reciprocals of the diagonal bin steps
    int nb[3], P[3], T[3], ntl[3], R[3], pbc[3];
    int tb, nregion;
    float inv_R0, inv_R01, inv_T[3];  // 1 / R0, 1 / (R0 R1), 1 / T (small_div)
    int wrap1;  // a region bin lies at most one cell outside the grid on every periodic axis
    int64_t ntiles;
    float toff, hi_off;  // d2' = d2 - toff: edge iff bits(d2') < lo_bits, band iff d2' <= hi_off
    uint32_t lo_bits;
    // the count pass's bounds on d2'' = d2 - mid (mid = fl(r^2)): edge iff d2'' < 0 unless
    // |d2''| <= band or d2'' <= low, which the exact test settles
    float mid, band, low;
    const float4* spos;
    const uint32_t* sflr;
    const int* sid;    // atom id of every cell-list entry
    const void* cpos;  // the positions in cell-list order (pos dtype; set for vector outputs)
    const int* bstart;
    const int* tile_of_rank;
    const int* rank_of_tile;
    const void* pos;
    int f64;
    // explicit targets (subset != 0)
    int subset;
    // Explicit targets that are exactly 0, 1, ..., ntarg - 1 (checked on the device: the
    // local atoms of a partition, DistGraphBuilder's mode B) need no target sort: every atom
    // of a tile is a lane, and atoms with ids >= ntarg (the ghosts) stay idle.  pmis is the
    // device word that is nonzero when the list is not that prefix (null: never masked).
    const int64_t* pmis;
    int64_t ntarg;
    const int* tbstart;
    const int* tsidx;
    const int* tslot;  // caller position of each sorted target
    // count pass
    int* cnt;          // per target, processing order
    int* counts_user;  // per target, caller order (nullable)
    int* ttot;         // per tile (rank order)
    int* tfix;         // per tile: kFix* bits, work left to search_kernel<1>
    // write pass
    int64_t* tbase;
    int64_t* out_src;
    int64_t* out_dst;
    float* out_shift;
    void* out_vec;
    void* out_dist;
    int vout_f64;
    int64_t capacity;
    int64_t* totals;
    const int64_t* out_ids;  // written for atom i: out_ids[i] (null: i); positions use i
    const int* wid;  // the id written for cell-list entry g (sid, or out_ids of it)
    // Row words (null: none recorded).  A target's edges are kept as one 32-bit word per stencil
    // row that holds any: the region index of the row's last candidate (12 bits) above the
    // row's edge mask (20 bits, bit i: candidate last - i); a longer row takes two words, the
    // first candidates first.  Words go in groups of four (16 bytes), group-major: group g of
    // target j at words + 4 * (g * nrow + j), so that the groups that neighbouring targets fill
    // at about the same time share cache lines.  nw[j]: words of target j (kWordsOver: its list
    // was too short, and search_kernel<1> writes its edges).
    uint32_t* words;
    uint8_t* nw;
    int Kw;          // words a target's list holds (a multiple of 4)
    int64_t nrow;    // targets (group row length)
    // The region map: for each tile, from entry tmap[tile].x on, one pair per region entry (its
    // cell-list index, packed image shift of its bin - floor of its atom).  Tiles take their
    // part of the map in the order in which they finish, from one of npools pools of equal size
    // (cursors in the tile offsets' place, which are written after the count, one 128-byte line
    // each; taken from a single cursor, 4860 tiles' atomics alone took 0.37 ms); what a part
    // holds is the same whatever the order.
    int2* map;
    int64_t mapcap;
    int npools;
    int2* tmap;  // (its first entry, its entries)
    int64_t* n_out;  // (write) where the number of edges goes too, or null
    int xsplit;     // bins ordered by x unless *xflag (see tile_sort_kernel): quarter-bin row ends
};

// Whether this build's targets are the atoms of the tile with ids < ntarg (see SearchArgs).
__device__ __forceinline__ bool masked_targets(const SearchArgs& a)
{
    return a.subset && a.pmis != nullptr && *a.pmis == 0;
}
// Whether targets come from the explicit (sorted) target list.
__device__ __forceinline__ bool listed_targets(const SearchArgs& a)
{
    return a.subset && !masked_targets(a);
}

// The kernel's arguments (a SearchArgs by value, the first parameter) read again from the
// kernarg segment, behind an opaque pointer: what a cold part of the search needs is then loaded
// there, instead of being held in scalar registers (and spilled) across the sweep.
__device__ __forceinline__ const SearchArgs& kernarg_search()
{
    auto p = (const __attribute__((address_space(4))) char*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const SearchArgs*)(const char*)p;
}

// Output order -> tile rank.  Consecutive workgroups go round-robin to the 8 XCDs; the
// Morton order is dealt out to them in runs of kXcdRun tiles (run q to XCD q mod 8), so a
// run of neighbouring tiles shares its halo bins in one L2, and every XCD's share is
// spread over the whole box.  (One contiguous eighth of the Morton order per XCD puts all
// the work of a half-empty box -- a slab, a two-phase cell -- on four XCDs: C4's count
// took 0.317 ms that way against 0.256 ms with runs.)  The output holds the tiles in this
// order; the last ntiles mod (8 kXcdRun) tiles keep their Morton rank.
constexpr int64_t kXcdRun = 16;
__device__ __forceinline__ int64_t xcd_tile_rank(int64_t b, int64_t ntiles)
{
    const int64_t full = ntiles / (8 * kXcdRun) * (8 * kXcdRun);
    if (b >= full) return b;
    const int64_t x = b & 7, j = b >> 3;
    return ((j / kXcdRun) * 8 + x) * kXcdRun + (j % kXcdRun);
}

// LDS of one search workgroup.
//   qbuf   the staged region: position relative to the tile centre per entry (the fix-up pass:
//          and the atom id); in the count pass with room for the three candidates read past a
//          row's end, and before its start;
//   rt     region bin table: the byte offset of each region bin's first entry, as 32-bit words
//          (rp) or, with quarter-bin row ends, as four 16-bit words per bin (rq): its quarters'.
// Positions alone (12 bytes an entry) let the count pass fit five workgroups per CU; the fix-up
// write pass adds the per-entry shift table T.
constexpr int kWordBits = 20;                 // candidates in a row word's mask
constexpr int kCountWaves = 5;                // waves per SIMD of the count pass
constexpr int kWordsOver = 255;               // nw of a target whose list was too short
constexpr int kRowMax = 28;                   // candidates of a row swept at a time (one mask register)
static_assert(2 * kCap <= 1 << (32 - kWordBits), "a region index fits the row word");

template <int ENT>
struct SearchLds {
    static constexpr int kEnt = ENT;  // bytes of a region entry
    static constexpr int kFront = ENT == 12 ? 3 * ENT : 0;  // bytes before the first one
    __align__(16) unsigned char qbuf[kFront + ENT * (kCap + 3)];
    union {
        int tbs[kTileMax * kTileMax * kTileMax + 1];  // bin starts of the tile, while a batch's targets
                                                      // are looked up
        __align__(16) uint32_t ring[kBlock][4];       // (count) then per-lane groups of row words
    };
    uint32_t rt[2 * kMaxRegion + 2];
    int64_t w64[kBlock / 64];
    int w32[kBlock / 64];
    int64_t bc[2];  // workgroup broadcasts
};
struct CountLds : SearchLds<12> {};
struct FixLds : SearchLds<16> {
    uint32_t T[kCap + 1];  // packed (bin image shift - source floor) per entry
};
static_assert(sizeof(CountLds) <= 32000, "count pass must fit five workgroups per CU (LDS goes in 1280 bytes)");
template <int MODE>
struct LdsOf { typedef CountLds type; };
template <>
struct LdsOf<1> { typedef FixLds type; };

// Cartesian offset of region bin (rx, ry, rz) from the centre of its tile: positions in
// LDS are relative to the tile centre, which keeps their magnitudes (and so their
// rounding) small.
__device__ __forceinline__ void region_offset(const SearchArgs& a, int rx, int ry, int rz,
                                              float* o)
{
    const double u0 = (double)(rx - a.P[0]) - 0.5 * a.T[0], u1 = (double)(ry - a.P[1]) - 0.5 * a.T[1],
                 u2 = (double)(rz - a.P[2]) - 0.5 * a.T[2];
#pragma unroll
    for (int c = 0; c < 3; ++c) o[c] = (float)fma(u2, a.hC[6 + c], fma(u1, a.hC[3 + c], u0 * a.hC[c]));
}

// Exact (canonical fp64) decision for a candidate the fp32 prefilter cannot settle: atom
// src as seen from target tgt, (dq0, dq1, dq2) = its fp32 LDS position minus the target's.
// The integer image shift is recovered by rounding: dq - (pos[src] - pos[tgt]) is S.C up
// to the LDS rounding (~1e-5 A), far below half a cell.
__device__ __forceinline__ bool exact_edge(const SearchArgs& a, int src, int tgt, double dq0,
                                        double dq1, double dq2)
{
    double ps[3], pt[3], v[3];
    load_pos(a.pos, a.f64, src, ps);
    load_pos(a.pos, a.f64, tgt, pt);
    const double w0 = dq0 - (ps[0] - pt[0]), w1 = dq1 - (ps[1] - pt[1]), w2 = dq2 - (ps[2] - pt[2]);
    const int S0 = (int)rint(canon_frac(w0, w1, w2, a.Cinv, 0));
    const int S1 = (int)rint(canon_frac(w0, w1, w2, a.Cinv, 1));
    const int S2 = (int)rint(canon_frac(w0, w1, w2, a.Cinv, 2));
    if (src == tgt && S0 == 0 && S1 == 0 && S2 == 0) return false;
    const double d2 = canon_d2(ps, pt, S0, S1, S2, a.C, v);
    return d2 > kSelfThr && d2 <= a.r2;
}

// One edge: edge_index columns, integer cell shift, optional canonical vector / distance.
__device__ __forceinline__ int out_id(const SearchArgs& a, int i)
{
    return a.out_ids ? (int)a.out_ids[i] : i;
}

// src, dst: atom indices (of pos); the ids written go through a.out_ids.
__device__ __forceinline__ void emit_edge(const SearchArgs& a, int64_t o, int src, int dst, int S0,
                                          int S1, int S2)
{
    a.out_src[o] = out_id(a, src);
    a.out_dst[o] = out_id(a, dst);
    *(float3*)(a.out_shift + 3 * o) = make_float3((float)S0, (float)S1, (float)S2);
    if (a.out_vec || a.out_dist) {
        double ps[3], pt[3], vv[3];
        load_pos(a.pos, a.f64, src, ps);
        load_pos(a.pos, a.f64, dst, pt);
        const double dd = canon_d2(ps, pt, S0, S1, S2, a.C, vv);
        if (a.vout_f64) {
            if (a.out_vec) {
                double* ov = (double*)a.out_vec + 3 * o;
                ov[0] = vv[0]; ov[1] = vv[1]; ov[2] = vv[2];
            }
            if (a.out_dist) ((double*)a.out_dist)[o] = sqrt(dd);
        } else {
            if (a.out_vec) {
                float* ov = (float*)a.out_vec + 3 * o;
                ov[0] = (float)vv[0]; ov[1] = (float)vv[1]; ov[2] = (float)vv[2];
            }
            if (a.out_dist) ((float*)a.out_dist)[o] = (float)sqrt(dd);
        }
    }
}

// ---------------------------------------------------------------- region bins
// x / y for 0 <= x < 2^16 and 1 <= y < 2^11, inv = fl(1 / y): the quotient is at least 1 / (2 y)
// from the next integer, far more than its rounding (an integer division by a run-time divisor
// takes about twenty instructions, and staging a region takes eight of them per bin).
__device__ __forceinline__ int small_div(int x, float inv) { return (int)(((float)x + 0.5f) * inv); }

// Coordinates of region bin rb inside the region.
__device__ __forceinline__ void region_coords(const SearchArgs& a, int rb, int* r)
{
    r[2] = small_div(rb, a.inv_R01);
    const int q = rb - r[2] * (a.R[0] * a.R[1]);
    r[1] = small_div(q, a.inv_R0);
    r[0] = q - r[1] * a.R[0];
}

// Grid bin w and periodic image sb of region bin r (region_coords) of the tile at bin g0; false
// outside the grid on a non-periodic axis (an empty bin).
__device__ __forceinline__ bool region_wrap(const SearchArgs& a, const int* g0, const int* r, int* w, int* sb)
{
    bool ok = true;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const int gg = g0[d] - a.P[d] + r[d], nb = a.nb[d];
        int q = 0;
        if (a.pbc[d]) {
            if (a.wrap1)
                q = gg < 0 ? -1 : (gg >= nb ? 1 : 0);
            else
                q = floor_div(gg, nb);
        } else {
            ok = ok && gg >= 0 && gg < nb;
        }
        sb[d] = q;
        w[d] = gg - q * nb;
    }
    return ok;
}

// Bin-list key of region bin rb of the tile at bin g0 (periodic wrap on pbc axes); false
// outside the grid on a non-periodic axis (an empty bin).
__device__ __forceinline__ bool region_bin_key(const SearchArgs& a, const int* g0, int rb,
                                               int64_t* key)
{
    int r[3], w[3], sb[3];
    region_coords(a, rb, r);
    if (!region_wrap(a, g0, r, w, sb)) return false;
    const int t0 = small_div(w[0], a.inv_T[0]), t1 = small_div(w[1], a.inv_T[1]), t2 = small_div(w[2], a.inv_T[2]);
    const int l0 = w[0] - t0 * a.T[0], l1 = w[1] - t1 * a.T[1], l2 = w[2] - t2 * a.T[2];
    const int tl = t0 + a.ntl[0] * (t1 + a.ntl[1] * t2);
    *key = (int64_t)a.rank_of_tile[tl] * a.tb + (l0 + a.T[0] * (l1 + a.T[1] * l2));
    return true;
}

// Cell-list start of region bin rb (0 for a bin outside the grid, which is empty).
__device__ __forceinline__ int region_bin_start(const SearchArgs& a, const int* g0, int rb)
{
    int64_t key;
    return region_bin_key(a, g0, rb, &key) ? a.bstart[key] : 0;
}

// Cell-list range of the region bins rb = kRegPerThread * threadIdx.x + h of the tile at
// bin g0; returns the thread's total.
__device__ __forceinline__ int region_bins(const SearchArgs& a, const int* g0, int* rcnt, int* rst)
{
    int sum = 0;
#pragma unroll
    for (int h = 0; h < kRegPerThread; ++h) {
        rcnt[h] = 0;
        rst[h] = 0;
        const int rb = kRegPerThread * threadIdx.x + h;
        int64_t key;
        if (rb < a.nregion && region_bin_key(a, g0, rb, &key)) {
            rst[h] = a.bstart[key];
            rcnt[h] = a.bstart[key + 1] - rst[h];
        }
        sum += rcnt[h];
    }
    return sum;
}

typedef float v3f __attribute__((ext_vector_type(3)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef int v4i __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------- edge expansion
// The edges of a tile are written by a few workgroups (parts), each a range of its outputs that
// starts on a 128-byte line (32 edges are 256 bytes of ids, 384 of shifts), in blocks of kSub
// edges: the row words of the block's targets are decoded into LDS, one entry per edge, and the
// edges then go out in 16-byte stores that fill whole lines.  The targets' ids may lie off the
// sources' lines (row 1 of a [2, E] array): a block then writes those of the edges `skew` further
// on.
//
// Bound by the stores: 1M atoms (90.5M edges, 2.53 GB) in 0.50-0.515 ms, against 0.595 ms with
// one workgroup per tile and the target ids off their lines; a probe that only stores the same
// pattern takes 0.46 ms with every line whole and 0.53 ms with the ids 80 bytes off.  Plain
// stores instead of non-temporal ones take 0.63 ms, and the same kernel without the next
// block's words fetched ahead (its loads then wait for the stores before them) 0.67 ms.
constexpr int kLine = 32;                       // edges whose outputs span whole lines
constexpr int kSub = 1024;                      // edges of a block
constexpr int kWaveEdges = kSub / (kBlock / 64);
constexpr int kSkewMax = 16;                    // 8-byte ids of a line
// A part's setup (region pairs, target tables) costs about as much as a block: parts grow with
// the tiles' number, to whole tiles in large boxes (1M atoms: 0.67 ms at two blocks a part, 0.55
// at four, 0.50-0.515 at eight to sixteen; 100k atoms: 0.067 ms at two, 0.088 at one).
constexpr double kPartBlocks = 10;              // blocks of a part, at most
constexpr double kPartsWanted = 4096;           // parts that fill the chip for a few rounds

template <typename VT, bool GROUPS>
struct ExpandLds {
    // per edge of the block: target in the batch and region entry (kNoEdge: the edge is written
    // by search_kernel<1>); then its packed shift
    uint32_t ent[kSub + kSkewMax];
    __align__(16) uint32_t shift[kSub + 2];
    // the region's pairs: id to write, packed shift (where there are no vectors)
    int2 pair[GROUPS && std::is_void<VT>::value ? kCap : 1];
    // the batch's targets: first edge and first row word (with the batch's totals behind them),
    // id to write, floor, cell-list index (vectors)
    int off[kBlock + 1];
    int woff[kBlock + 1];
    int tid[kBlock];
    uint32_t tf[kBlock];
    int tg[std::is_void<VT>::value ? 1 : kBlock];
    int t01[2][2];  // the first and last target of a block and of the next
    int2 s2[kBlock / 64];
    int w32[kBlock / 64];
    // edge vectors and distances as the bytes they take in the outputs
    __align__(16) typename std::conditional<std::is_void<VT>::value, int, VT>::type
        v[std::is_void<VT>::value ? 4 : 3 * kSub],
        d[std::is_void<VT>::value ? 4 : kSub];
};
constexpr int kPoolLine = 16;  // 64-bit words between the region map's cursors
// waves per SIMD of the expansion (fp64 vectors: three by their LDS)
template <typename VT>
constexpr int expand_waves = std::is_same<VT, double>::value ? 3 : 5;
constexpr uint32_t kNoEdge = 0xFFFFFFFFu;
constexpr uint32_t kZero3 = (uint32_t)kFloorBias * 0x00100401u;  // pack3(0, 0, 0)

// Part s of S of tile ord for workgroup b: the parts of a tile go to one XCD (the dispatch deals
// consecutive workgroups to the 8 XCDs in turn), so that they share its region map and words.
__device__ __forceinline__ void part_of(int64_t b, int64_t ntiles, int S, int64_t* ord, int* s)
{
    const int64_t grp = b / (8 * S);
    const int r = (int)(b - grp * (8 * S));
    const int m = (int)min<int64_t>(8, ntiles - 8 * grp);
    *s = r / m;
    *ord = 8 * grp + (r - *s * m);
}

// Two neighbouring row words of a lane, on their way from memory.
struct WordPair {
    uint32_t w[2];
    int t[2];  // their targets in the batch (the second's, or the first's again)
    int live;  // how many there are
};

// Writes part s of S of the edges of tile ord (of the target ids, those skew further on), from
// the row words of its targets and its region map.
// GROUPS: the edges go out in 16-byte groups, with VT (float or double) the edge vectors and
// distances too; otherwise every edge is written by its lane (emit_edge).
template <typename VT, bool GROUPS>
__device__ __forceinline__ void expand_part(const SearchArgs& a, ExpandLds<VT, GROUPS>& sh, int64_t ord, int s, int S,
                                            int skew)
{
    constexpr bool kVec = !std::is_void<VT>::value;
    constexpr bool kStaged = GROUPS && !kVec;
    typedef typename std::conditional<kVec, VT, float>::type VTn;  // (a type when VT is void)
    const int tt = a.ttot[ord];
    if (tt == 0) return;
    const int64_t tb = a.tbase[ord];
    if (tb + tt > a.capacity) {
        if (threadIdx.x == 0 && !(__hip_atomic_load(&a.totals[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & kStatusCapacity))
            atomicOr((unsigned long long*)&a.totals[1], (unsigned long long)kStatusCapacity);
        return;
    }
    const int fix = a.tfix[ord];
    if (fix & kFixChunked) return;  // written by search_kernel<1>
    // the part's outputs [p0, p1), and where the last ones of its target ids end
    // (a part that would start at or before the tile is empty, but for one, the tile's first)
    auto cut = [&](int q) {
        const int64_t g = (tb + (int64_t)tt * q / S) & ~(int64_t)(kLine - 1);
        return q == S ? tb + tt : (g <= tb ? tb & ~(int64_t)(kLine - 1) : g);
    };
    const int64_t r0 = cut(s), p1 = cut(s + 1), p0 = max(tb, r0);
    if (p0 >= p1) return;
    const int64_t q1 = min(tb + tt, p1 + skew);
    const bool listed = listed_targets(a);
    const int64_t kb = xcd_tile_rank(ord, a.ntiles) * a.tb;
    const int* const tstart = listed ? a.tbstart : a.bstart;
    const int tbeg = tstart[kb], ntg = tstart[kb + a.tb] - tbeg;
    const int2 tm = a.tmap[ord];
    const int2* const __restrict__ map = a.map + tm.x;
    const int nreg = tm.y;  // region entries
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint64_t gstep = 16ull * (uint64_t)a.nrow;  // bytes between a target's word groups
    // The region's pairs (id to write, shift) in LDS when they fit: a block's stores then wait
    // for no load behind them (loads and stores share one in-order counter).
    const bool staged = kStaged && nreg <= kCap;
    constexpr int kPer = kStaged ? (kCap + kBlock - 1) / kBlock : 1;
    int2 pr[kPer];
    if (staged)
#pragma unroll
        for (int u = 0; u < kPer; ++u) pr[u] = map[min(tid + kBlock * u, nreg - 1)];

    int64_t gb = tb;  // output of the batch's first edge
    for (int k0 = 0; k0 < ntg && gb < q1; k0 += kBlock) {
        const int j = min(tbeg + k0 + tid, tbeg + ntg - 1);
        const bool in = k0 + tid < ntg;
        const int sidx = listed ? a.tsidx[j] : j;
        const int cnt = in ? a.cnt[j] : 0;
        const int nw0 = in ? a.nw[j] : 0;
        const int my_id = GROUPS ? a.wid[sidx] : a.sid[sidx];
        const uint32_t my_f = a.sflr[sidx];
        if (staged && k0 == 0) {
#pragma unroll
            for (int u = 0; u < kPer; ++u) pr[u].x = a.wid[pr[u].x];
        }
        // (a target without words has one that stands for all its edges)
        const int nw = nw0 == kWordsOver ? 1 : nw0;
        int btot, wtot;
        const int2 ex2 = block_excl_scan2<kBlock>(make_int2(cnt, nw), sh.s2, &btot, &wtot);
        const int ex = ex2.x;
        sh.off[tid] = ex;
        sh.woff[tid] = ex2.y;
        if (tid == 0) {
            sh.off[kBlock] = btot;
            sh.woff[kBlock] = wtot;
        }
        sh.tid[tid] = my_id;
        sh.tf[tid] = my_f;
        if constexpr (kVec) sh.tg[tid] = sidx;
        if (staged && k0 == 0) {
#pragma unroll
            for (int u = 0; u < kPer; ++u)
                if (tid + kBlock * u < nreg) sh.pair[tid + kBlock * u] = pr[u];
        }
        const int64_t g0 = gb;
        gb += btot;
        // (uniform; a batch without edges, ghosts only, names no target for a block either, and
        // t01 would hold another batch's)
        if (gb <= p0 || btot == 0) {
            __syncthreads();
            continue;
        }
        // the batch's edges [b0, b1) are the part's, those from b2 on for their target ids only
        const int b0 = (int)(max(p0, g0) - g0), b1 = (int)(min(q1, gb) - g0), b2 = (int)(min(p1, gb) - g0);
        // the edges [lo, hi) of the block at output `block` (hi: target ids included), and of its
        // place in LDS, at, the batch's edge 0
        auto range = [&](int64_t block, int& lo, int& hi, int& at) {
            lo = max(b0, (int)(block - g0));
            hi = min(b1, (int)(block + kSub + skew - g0));
            at = (int)(g0 - block);
        };
        // notes the first and last target of a block, for the lanes that read sh.t01[slot] after
        // the next barrier
        auto mark = [&](int64_t block, int slot) {
            int lo, hi, at;
            range(block, lo, hi, at);
            if (cnt > 0 && ex <= lo && ex + cnt > lo) sh.t01[slot][0] = tid;
            if (cnt > 0 && ex < hi && ex + cnt >= hi) sh.t01[slot][1] = tid;
        };
        auto word_at = [&](int t, int w) {
            return *(const uint32_t*)((const char*)a.words + 16ull * (uint64_t)(tbeg + k0 + t) +
                                      (uint64_t)(uint32_t)(w >> 2) * gstep + 4 * (w & 3));
        };
        // words i and i + 1 of the batch (i = the first of the block's, + 2 tid + skip); the
        // loads go out unconditionally
        auto fetch = [&](int slot, int skip) {
            const int tf = sh.t01[slot][0], tl = sh.t01[slot][1];
            const int wend = sh.woff[tl + 1], i = sh.woff[tf] + 2 * tid + skip;
            int t = tf, th = tl + 1;  // the target with woff[t] <= i < woff[t + 1]
            while (th - t > 1) {
                const int mid = (t + th) >> 1;
                const bool up = sh.woff[mid] <= i;
                t = up ? mid : t;
                th = up ? th : mid;
            }
            WordPair P;
            P.live = min(max(wend - i, 0), 2);
            int t2 = t;
            if (P.live == 2)
                while (sh.woff[t2 + 1] <= i + 1) ++t2;
            P.t[0] = t;
            P.t[1] = t2;
            P.w[0] = word_at(t, P.live > 0 ? i - sh.woff[t] : 0);
            P.w[1] = word_at(t2, P.live > 1 ? i + 1 - sh.woff[t2] : 0);
            return P;
        };
        // writes a block's entries from its words, two per lane: a word's edges start where the
        // words before it end.  first: the batch's edge that the first of them starts at;
        // returns where the last ends.
        auto decode = [&](const WordPair& P, int lo, int hi, int at, int first) {
            uint32_t bits[2];
            int n[2];
            const bool over_tile = (fix & kFixOver) != 0;
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                bits[k] = P.live > k ? P.w[k] & ((1u << kWordBits) - 1u) : 0u;
                n[k] = __popc(bits[k]);
                if (__builtin_expect(over_tile, 0) && P.live > k && a.nw[tbeg + k0 + P.t[k]] == kWordsOver) {
                    bits[k] = 0;
                    n[k] = a.cnt[tbeg + k0 + P.t[k]];
                }
            }
            int rtot;
            int e0 = first + block_excl_scan_dpp<kBlock>(n[0] + n[1], sh.w32, &rtot);
            if (__builtin_expect(over_tile, 0)) {  // (those edges are written by search_kernel<1>)
                int e1 = e0;
                for (int k = 0; k < 2; ++k) {
                    if (bits[k] == 0)
                        for (int e = max(e1, lo); e < min(e1 + n[k], hi); ++e) sh.ent[at + e] = kNoEdge;
                    e1 += n[k];
                }
            }
            uint32_t* const ent = sh.ent + (at + lo);
            const uint32_t len = (uint32_t)(hi - lo);
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                // the mask's bits from the first candidate on; q: entry of the candidate before
                // the leading bit
                uint32_t m = bits[k] << (32 - kWordBits);
                uint32_t q = ((uint32_t)P.t[k] << 12) + (P.w[k] >> kWordBits) - (uint32_t)kWordBits;
                uint32_t e = (uint32_t)(e0 - lo);
                while (m != 0u) {
                    const uint32_t c = (uint32_t)__builtin_clz(m) + 1u;
                    q += c;
                    m <<= c;
                    if (e < len) ent[e] = q;
                    ++e;
                }
                e0 += n[k];
            }
            return first + rtot;
        };
        auto pair_of = [&](uint32_t en) -> int2 {
            const uint32_t k = en == kNoEdge ? 0u : en & 4095u;
            if constexpr (kStaged) {
                if (staged) return sh.pair[k];
                int2 p = map[k];
                p.x = a.wid[p.x];
                return p;
            } else {
                return map[k];
            }
        };
        // the shifts of this wave's edges, from LDS: 16-byte chunks, of the groups of 4 edges in
        // [a0, a1)
        const int wb = kWaveEdges * wave;
        auto store_shifts = [&](int64_t block, bool full, int a0, int a1) {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            v4f* const __restrict__ of = (v4f*)(a.out_shift + 3 * block);
#pragma unroll
            for (int h = 0; h < 3 * kWaveEdges / 256; ++h) {
                // chunk c: shift floats 4c .. 4c + 3, fields r .. r + 3 of the six of edges e, e + 1
                const int c = 3 * wb / 4 + 64 * h + lane;
                const int g = c / 3, r = c - 3 * g, e = 4 * g + r;  // (4c / 3 = 4g + r for r < 3)
                if (full || (4 * g >= a0 && 4 * g < a1)) {
                    const uint32_t S0 = sh.shift[e], S1 = sh.shift[e + 1];
                    const uint64_t P = ((uint64_t)S1 << 30 | S0) >> (10 * r);
                    const v4f vf = {(float)((int)(P & 1023u) - kFloorBias),
                                    (float)((int)((P >> 10) & 1023u) - kFloorBias),
                                    (float)((int)((P >> 20) & 1023u) - kFloorBias),
                                    (float)((int)((P >> 30) & 1023u) - kFloorBias)};
                    __builtin_nontemporal_store(vf, of + c);
                }
            }
        };
        // Writes a block whose edges are all the part's: straight-line code, so that the next
        // block's words, fetched before, are waited for without its stores.
        auto write_full = [&](int64_t block) {
            v4i* const __restrict__ os = (v4i*)(a.out_src + block);
            v4i* const __restrict__ od = (v4i*)(a.out_dst + block + skew);
            uint32_t en[kWaveEdges / 64], et[kWaveEdges / 64];
            int2 mp[kWaveEdges / 64];
#pragma unroll
            for (int u = 0; u < kWaveEdges / 64; ++u) {
                // a lane takes two neighbouring edges at a time
                const int i = wb + 128 * (u / 2) + 2 * lane + (u & 1);
                en[u] = sh.ent[i];
                et[u] = sh.ent[i + skew];
            }
#pragma unroll
            for (int u = 0; u < kWaveEdges / 64; ++u) mp[u] = sh.pair[en[u] & 4095u];
#pragma unroll
            for (int h = 0; h < kWaveEdges / 128; ++h) {
                const int i = wb + 128 * h + 2 * lane;
                uint32_t S3[2];
#pragma unroll
                for (int k = 0; k < 2; ++k) S3[k] = (uint32_t)mp[2 * h + k].y + sh.tf[en[2 * h + k] >> 12] - kZero3;
                *(uint2*)&sh.shift[i] = make_uint2(S3[0], S3[1]);
                const v4i vs = {mp[2 * h].x, 0, mp[2 * h + 1].x, 0};
                const v4i vd = {sh.tid[et[2 * h] >> 12], 0, sh.tid[et[2 * h + 1] >> 12], 0};
                __builtin_nontemporal_store(vs, os + i / 2);
                __builtin_nontemporal_store(vd, od + i / 2);
            }
            store_shifts(block, true, 0, 0);
        };
        // Any block.
        auto write_any = [&](int64_t block, int lo, int hi, int at, int tf0) {
            const int i0 = max(at + lo, wb), i1 = min(at + b2, wb + kWaveEdges);
            if constexpr (!GROUPS) {
                for (int i = i0 + lane; i < i1; i += 64) {
                    const uint32_t en = sh.ent[i];
                    if (en == kNoEdge) continue;
                    const int2 mp = map[en & 4095u];
                    const uint32_t S3 = (uint32_t)mp.y + sh.tf[en >> 12] - kZero3;
                    emit_edge(a, block + i, a.sid[mp.x], sh.tid[en >> 12], unpack3(S3, 0), unpack3(S3, 1), unpack3(S3, 2));
                }
                return;
            }
            // the sources of two neighbouring edges are one 16-byte store, and the shifts of four
            // are three, where the edges are all the part's: groups of 4 at multiples of 4 outputs
            // in [a0, a1); the up-to-3 edges before and after go per lane
            const int a0 = (i0 + 3) & ~3, a1 = i1 & ~3;
            const bool any = i0 < i1;
            uint32_t en[kWaveEdges / 64];
            int2 mp[kWaveEdges / 64];
            int src[kWaveEdges / 64];
#pragma unroll
            for (int u = 0; u < kWaveEdges / 64; ++u) {
                const int i = wb + 128 * (u / 2) + 2 * lane + (u & 1);
                en[u] = i >= i0 && i < i1 ? sh.ent[i] : kNoEdge;
                mp[u] = pair_of(en[u]);
            }
#pragma unroll
            for (int u = 0; u < kWaveEdges / 64; ++u) src[u] = kStaged ? mp[u].x : a.wid[mp[u].x];
            uint32_t S3[kWaveEdges / 64];
#pragma unroll
            for (int u = 0; u < kWaveEdges / 64; ++u) {
                const int i = wb + 128 * (u / 2) + 2 * lane + (u & 1);
                const uint32_t t = en[u] == kNoEdge ? (uint32_t)tf0 : en[u] >> 12;
                // (the fields of pack3 add without carries: a shift fits 10 bits)
                S3[u] = en[u] == kNoEdge ? kZero3 : (uint32_t)mp[u].y + sh.tf[t] - kZero3;
                sh.shift[i] = S3[u];
                if constexpr (kVec) {
                    double ps[3], pt[3], vv[3];
                    load_pos(a.cpos, a.f64, mp[u].x, ps);
                    load_pos(a.cpos, a.f64, sh.tg[t], pt);
                    const double dd = canon_d2(ps, pt, unpack3(S3[u], 0), unpack3(S3[u], 1), unpack3(S3[u], 2), a.C, vv);
                    sh.v[3 * i] = (VTn)vv[0];
                    sh.v[3 * i + 1] = (VTn)vv[1];
                    sh.v[3 * i + 2] = (VTn)vv[2];
                    sh.d[i] = (VTn)sqrt(dd);
                }
            }
            // the target ids of the wave's edges, skew further on (at the tile's start, the first
            // ones too)
            {
                const int j0 = max(at + lo, r0 <= tb && block == r0 && wave == 0 ? 0 : wb + skew);
                const int j1 = min(at + hi, wb + kWaveEdges + skew);
                auto target = [&](int i) {
                    const uint32_t e = sh.ent[i];
                    return sh.tid[e == kNoEdge ? (uint32_t)tf0 : e >> 12];
                };
                if (j0 == wb + skew && j1 - j0 == kWaveEdges) {
#pragma unroll
                    for (int h = 0; h < kWaveEdges / 128; ++h) {
                        const int i = wb + skew + 128 * h + 2 * lane;
                        const v4i vd = {target(i), 0, target(i + 1), 0};
                        __builtin_nontemporal_store(vd, (v4i*)(a.out_dst + block + i));
                    }
                } else {
                    for (int i = j0 + lane; i < j1; i += 64) a.out_dst[block + i] = target(i);
                }
            }
            if (!any) return;
            v4i* const __restrict__ os = (v4i*)(a.out_src + block);
#pragma unroll
            for (int h = 0; h < kWaveEdges / 128; ++h) {
                const int i = wb + 128 * h + 2 * lane;
                if (i >= a0 && i < a1) {
                    const v4i vs = {src[2 * h], 0, src[2 * h + 1], 0};
                    __builtin_nontemporal_store(vs, os + i / 2);
                } else {
#pragma unroll
                    for (int k = 0; k < 2; ++k)
                        if (i + k >= i0 && i + k < i1) {
                            const int64_t o = block + i + k;
                            const uint32_t S = S3[2 * h + k];
                            a.out_src[o] = src[2 * h + k];
                            *(float3*)(a.out_shift + 3 * o) =
                                make_float3((float)unpack3(S, 0), (float)unpack3(S, 1), (float)unpack3(S, 2));
                            if constexpr (kVec) {
                                if (a.out_vec)
                                    for (int c = 0; c < 3; ++c) ((VTn*)a.out_vec)[3 * o + c] = sh.v[3 * (i + k) + c];
                                if (a.out_dist) ((VTn*)a.out_dist)[o] = sh.d[i + k];
                            }
                        }
                }
            }
            const bool full = i1 - i0 == kWaveEdges;
            store_shifts(block, full, a0, a1);
            if constexpr (kVec) {
                // the staged rows are the outputs' bytes
                constexpr int kPer = 16 / (int)sizeof(VTn);  // VT per chunk
                if (a.out_vec) {
                    v4i* const __restrict__ ov = (v4i*)((VTn*)a.out_vec + 3 * block);
#pragma unroll
                    for (int h = 0; h < 3 * kWaveEdges / kPer / 64; ++h) {
                        const int c = 3 * wb / kPer + 64 * h + lane;
                        const int q = kPer * c / 12 * 4;  // of the edges q .. q + 3
                        if (full || (q >= a0 && q < a1)) __builtin_nontemporal_store(((const v4i*)sh.v)[c], ov + c);
                    }
                }
                if (a.out_dist) {
                    v4i* const __restrict__ odd = (v4i*)((VTn*)a.out_dist + block);
#pragma unroll
                    for (int h = 0; h < kWaveEdges / kPer / 64; ++h) {
                        const int c = wb / kPer + 64 * h + lane;
                        const int q = kPer * c & ~3;
                        if (full || (q >= a0 && q < a1)) __builtin_nontemporal_store(((const v4i*)sh.d)[c], odd + c);
                    }
                }
            }
        };

        // The blocks of kSub outputs (the first may hold target ids only, those of the batch's
        // first edges).  A block's words are fetched while the block before it is written.
        int64_t block = r0 + (max(g0 + b0 - skew - r0, (int64_t)0) & ~(int64_t)(kSub - 1));
        const int64_t bend = min(g0 + (int64_t)b1, p1);  // blocks start below it
        if (block >= bend) {
            __syncthreads();
            continue;
        }
        mark(block, 0);
        __syncthreads();
        WordPair P = fetch(0, 0);
        int slot = 0;
        auto is_full = [&](int64_t b) {
            return kStaged && staged && fix == 0 && !(r0 <= tb && b == r0) && g0 + b0 <= b && b + kSub + skew <= g0 + b1 && b + kSub <= g0 + b2;
        };
        auto words_in = [&](int sl) { return sh.woff[sh.t01[sl][1] + 1] - sh.woff[sh.t01[sl][0]]; };
        while (block < bend) {
            int lo, hi, at;
            if constexpr (kStaged) {
                if (is_full(block) && words_in(slot) <= 2 * kBlock) {
                    // (the first pair is waited for here, so that the wait inside the loop is the
                    // one behind the loop's own stores)
                    asm volatile("" : "+v"(P.w[0]), "+v"(P.w[1]));
                    bool again;
                    do {
                        range(block, lo, hi, at);
                        decode(P, lo, hi, at, sh.off[sh.t01[slot][0]]);
                        const int64_t next = block + kSub;
                        const bool more = next < bend;
                        mark(more ? next : block, slot ^ 1);
                        __syncthreads();
                        P = fetch(slot ^ 1, 0);
                        write_full(block);
                        slot ^= 1;
                        block = next;
                        again = more && is_full(next) && words_in(slot) <= 2 * kBlock;
                        __syncthreads();  // before the next block's entries are written
                    } while (again);
                    if (block >= bend) break;
                }
            }
            range(block, lo, hi, at);
            const int tf0 = sh.t01[slot][0], nwords = words_in(slot);
            int first = decode(P, lo, hi, at, sh.off[tf0]);
            for (int skip = 2 * kBlock; skip < nwords; skip += 2 * kBlock)
            {
                const WordPair Q = fetch(slot, skip);
                __syncthreads();  // (before the scan's sums are written again)
                first = decode(Q, lo, hi, at, first);
            }
            const int64_t next = block + kSub;
            if (next < bend) mark(next, slot ^ 1);
            __syncthreads();
            if (next < bend) P = fetch(slot ^ 1, 0);
            write_any(block, lo, hi, at, tf0);
            slot ^= 1;
            block = next;
            __syncthreads();  // before the next block's entries, or the next batch's tables
        }
    }
}

// Takes n entries of pool p of the region map; where they start in the pool.
__device__ __forceinline__ unsigned long long map_take(const SearchArgs& a, int p, int n)
{
    return atomicAdd((unsigned long long*)a.tbase + kPoolLine * p, (unsigned long long)n);
}

// Neighbour search, one tile of bins per workgroup.
//
// The region of (T+2P)^3 bins around the tile is staged in LDS (in chunks if it does
// not fit).  Both passes share the per-target sweep below (one lane per target, rows of
// the stencil trimmed to the cutoff sphere for lower-triangular cells), so they agree on
// every edge and on its order.
//
// MODE 0 (count): per-target degree, per-tile total, and -- for tiles whose region fits two
//   chunks -- the target's row words and the tile's region map.
// MODE 1 (fix-up write, only tiles the count pass flagged): targets with more words than their
//   list holds, and tiles without words, are swept again and written directly.  Every other
//   edge is written by expand_kernel.
// What the count of one tile leaves for the publication / expansion of its edges.
struct TileOut {
    int64_t tt;  // edges of the tile
    int fix;     // kFix* bits
    int tbeg, ntg;
    int g0[3];
};

// QS (count pass, cell list ordered by bin_xkey inside bins): the quarter-bin row ends
// described below, for orthorhombic (1) or other lower-triangular cells (2); 0: whole
// bins, any cell.
template <int MODE, int QS = 0>
__device__ __forceinline__ TileOut search_tile(const SearchArgs& a,
                                               typename LdsOf<MODE>::type& sh, int64_t ord)
{
    constexpr bool WRITE = MODE == 1;
    constexpr int kEnt = LdsOf<MODE>::type::kEnt;
    char* const qb = (char*)sh.qbuf + LdsOf<MODE>::type::kFront;
    int* const rp = (int*)sh.rt;
    uint16_t* const rq = (uint16_t*)sh.rt;
    TileOut out;
    out.tt = 0;
    out.fix = 0;
    // ord: the tile's place in the output (and index of its per-tile records); rank: its
    // Morton rank.  Tiles go to the output in ord order; ord -> rank is xcd_tile_rank.
    const int64_t rank = xcd_tile_rank(ord, a.ntiles);
    const int lin = a.tile_of_rank[rank];
    const int tx = lin % a.ntl[0];
    const int ty = (lin / a.ntl[0]) % a.ntl[1];
    const int tz = lin / (a.ntl[0] * a.ntl[1]);
    const int g0[3] = {tx * a.T[0], ty * a.T[1], tz * a.T[2]};
    const bool listed = listed_targets(a), masked = a.subset && !listed;
    const int* tstart = listed ? a.tbstart : a.bstart;
    const int64_t kb = rank * a.tb;
    const int tbeg = tstart[kb], tend = tstart[kb + a.tb];
    const int ntg = tend - tbeg;
    out.tbeg = tbeg;
    out.ntg = ntg;
    for (int d = 0; d < 3; ++d) out.g0[d] = g0[d];
    if (ntg == 0) {
        if (MODE == 0 && threadIdx.x == 0) {
            a.ttot[ord] = 0;
            a.tfix[ord] = 0;
        }
        return out;
    }
    if (WRITE && a.tfix[ord] == 0) return out;  // written by the expansion
    if (!WRITE && masked) {
        // a tile of ghosts only (atoms with ids >= ntarg) has no targets: nothing to count
        bool mine = false;
        for (int k = threadIdx.x; k < ntg; k += kBlock) mine = mine || a.sid[tbeg + k] < a.ntarg;
        if (!block_any<kBlock>(mine, sh.w32)) {
            if (threadIdx.x == 0) {
                a.ttot[ord] = 0;
                a.tfix[ord] = 0;
            }
            return out;
        }
    }
    int64_t ebase = 0;
    if (WRITE) {
        ebase = a.tbase[ord];
        if (ebase + a.ttot[ord] > a.capacity) {
            if (threadIdx.x == 0)
                atomicOr((unsigned long long*)&a.totals[1], (unsigned long long)kStatusCapacity);
            return out;
        }
    }

    // ---- region table: (T+2P)^3 bins around the tile, periodic wrap on pbc axes
    const int R0 = a.R[0], R1 = a.R[1];
    int rcnt[kRegPerThread], rst[kRegPerThread];
    const int mysum = region_bins(kernarg_search(), g0, rcnt, rst);
    int total;
    int rex[kRegPerThread];  // first region entry of this thread's bins
    {
        int ex = block_excl_scan<int, kBlock>(mysum, sh.w32, &total);
#pragma unroll
        for (int h = 0; h < kRegPerThread; ++h) {
            rex[h] = ex;
            ex += rcnt[h];
        }
    }
    const int nchunks = (total + kCap - 1) / kCap;
    // Quarter-bin row ends (QS: count pass, lower-triangular cell; a one-chunk region whose
    // bins are ordered by bin_xkey): the bin table holds where each quarter of a bin starts,
    // counted by the entries whose key lies below each quarter boundary while staging, and a
    // row then starts at the quarter of its first bin that the cutoff reaches and ends after
    // the quarter of its last.  Entries cut off this way lie beyond the padded cutoff along x
    // alone, so they are never edges: every target's edge sequence is unchanged (the fix-up
    // pass, which sweeps whole bins, numbers edges alike).
    static_assert(12 * kCap < 65536, "a one-chunk region's offsets fit 16 bits");
    const bool qsplit = QS != 0 && nchunks == 1 && a.totals[4] == 0;
    if (!qsplit) {
#pragma unroll
        for (int h = 0; h < kRegPerThread; ++h) {
            const int rb = kRegPerThread * threadIdx.x + h;
            if (rb < a.nregion) rp[rb] = kEnt * rex[h];
        }
        if (threadIdx.x == 0) rp[a.nregion] = kEnt * total;
    } else if (threadIdx.x == 0) {
        rq[4 * a.nregion] = (uint16_t)(kEnt * total);
    }
    // byte offset of region bin rb's first entry, in the whole region
    auto bin_first = [&](int rb) -> int { return qsplit ? (int)rq[4 * rb] : rp[rb]; };
    // row words name up to two chunks' entries; a larger region is written directly by
    // search_kernel<1>, which follows what the count pass recorded: a tile flagged as chunked
    // is swept again
    const bool slotted = WRITE ? !(a.tfix[ord] & kFixChunked) : nchunks <= 2 && a.words != nullptr;
    unsigned long long map_at = 0;  // (count, thread 0) the tile's first region-map entry
    int loaded = -1;

    // packed (image shift of region bin rb - floor of cell-list entry gidx)
    auto entry_T = [&](int rb, int gidx) -> uint32_t {
        const uint32_t fl = a.sflr[gidx];
        int r[3], w[3], sb[3];
        region_coords(a, rb, r);
        region_wrap(a, g0, r, w, sb);
        return pack3(sb[0] - unpack3(fl, 0), sb[1] - unpack3(fl, 1), sb[2] - unpack3(fl, 2));
    };
    // every thread copies the entries of its own region bins (cnt, first cell-list entry st,
    // first region entry ex0) that fall in chunk c
    auto copy_bins = [&](int c, const int* cnt, const int* st, const int* ex0) {
        const SearchArgs& k = kernarg_search();
        const float qb1 = 0.25f * k.hax, qb2 = 0.5f * k.hax, qb3 = 0.75f * k.hax;
        XKey xkey;
        xkey.hbx = k.hbx; xkey.hcx = k.hcx; xkey.hcy = k.hcy; xkey.inv_hby = k.inv_hby; xkey.inv_hcz = k.inv_hcz;
        const int c0 = c * kCap;
        const int c1 = min(total, c0 + kCap);
#pragma unroll
        for (int h = 0; h < kRegPerThread; ++h) {
            const int rb = kRegPerThread * threadIdx.x + h;
            const int b0 = max(ex0[h], c0), b1 = min(ex0[h] + cnt[h], c1);
            int s1 = 0, s2 = 0, s3 = 0;  // entries below the quarter boundaries
            if (b0 < b1) {
                int r[3];
                region_coords(k, rb, r);
                float o[3];
                region_offset(k, r[0], r[1], r[2], o);
                const int g = st[h] - ex0[h];  // cell-list index minus region index
                for (int vv = b0; vv < b1; vv += 4) {
                    float4 e[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        if (vv + u < b1) e[u] = k.spos[g + vv + u];
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        if (vv + u < b1) {
                            const float x = e[u].x + o[0], y = e[u].y + o[1], z = e[u].z + o[2];
                            if constexpr (WRITE) {
                                ((float4*)qb)[vv + u - c0] = make_float4(x, y, z, e[u].w);
                                sh.T[vv + u - c0] = entry_T(rb, g + vv + u);
                            } else {
                                float* const to = (float*)(qb + kEnt * (vv + u - c0));
                                to[0] = x; to[1] = y; to[2] = z;
                            }
                            if constexpr (QS != 0) {
                                const float xk = QS == 1 ? e[u].x : bin_xkey(e[u], xkey);
                                s1 += xk < qb1;
                                s2 += xk < qb2;
                                s3 += xk < qb3;
                            }
                        }
                }
            }
            if (QS != 0 && qsplit && rb < k.nregion) {  // (one chunk: [b0, b1) is the whole bin)
                const uint32_t f = (uint32_t)(kEnt * ex0[h]);
                sh.rt[2 * rb] = f | ((f + kEnt * s1) << 16);
                sh.rt[2 * rb + 1] = (f + kEnt * s2) | ((f + kEnt * s3) << 16);
            }
        }
    };
    auto ensure_chunk = [&](int c) {  // uniform
        if (loaded != c) {
            __syncthreads();
            if (loaded < 0 && c == 0) {
                copy_bins(0, rcnt, rst, rex);
            } else {
                // (looked up again: the bins of the first chunk need not stay in registers)
                int cnt[kRegPerThread], st[kRegPerThread], ex0[kRegPerThread];
                region_bins(kernarg_search(), g0, cnt, st);
#pragma unroll
                for (int h = 0; h < kRegPerThread; ++h)
                    ex0[h] = cnt[h] ? bin_first(kRegPerThread * threadIdx.x + h) / kEnt : 0;
                copy_bins(c, cnt, st, ex0);
            }
            __syncthreads();
            loaded = c;
        }
    };
    // the first chunk is resident before the first target is looked up
    ensure_chunk(0);

    const int nrx = 2 * a.P[0] + 1, nry = 2 * a.P[1] + 1, nrz = 2 * a.P[2] + 1;
    int tile_found = 0;  // (this lane's; a tile's total is kept as an int too)
    bool over_any = false;

    for (int k0 = 0; k0 < ntg; k0 += kBlock) {
        const int nbatch = min(kBlock, ntg - k0);
        for (int k = threadIdx.x; k <= a.tb; k += kBlock) sh.tbs[k] = tstart[kb + k];
        __syncthreads();
        const int kk = k0 + threadIdx.x;
        const int j = tbeg + kk;
        const bool in_batch = (int)threadIdx.x < nbatch;
        bool active = in_batch;

        // ---- per-lane target state
        int lx = 0, ly = 0, lz = 0, my_id = 0, caller = 0;
        int v_self = -kEnt;  // byte offset of the target's own region entry
        uint32_t my_f = 0;
        float t0 = 0.f, t1 = 0.f, t2 = 0.f, ux = 0.f, uy = 0.f, uz = 0.f;
        if (active) {
            int lo = 0, hi = a.tb;
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (sh.tbs[mid] <= j) lo = mid; else hi = mid;
            }
            const int q = small_div(lo, a.inv_T[0]);
            lz = small_div(q, a.inv_T[1]);
            ly = q - lz * a.T[1];
            lx = lo - q * a.T[0];
            const int sidx = listed ? a.tsidx[j] : j;
            const float4 e = a.spos[sidx];
            my_f = a.sflr[sidx];
            my_id = __float_as_int(e.w);
            caller = listed ? a.tslot[j] : my_id;
            active = !masked || my_id < a.ntarg;  // (masked: a ghost atom's lane idles)
            ux = e.x; uy = e.y; uz = e.z;  // position inside its own bin
            float o[3];
            region_offset(kernarg_search(), lx + a.P[0], ly + a.P[1], lz + a.P[2], o);
            t0 = e.x + o[0]; t1 = e.y + o[1]; t2 = e.z + o[2];
            // the target's own region entry (same atom, zero shift) is never an edge
            const int rb_self = ((lz + a.P[2]) * R1 + (ly + a.P[1])) * R0 + (lx + a.P[0]);
            const int bin_start = listed ? a.bstart[kb + lo] : sh.tbs[lo];
            v_self = bin_first(rb_self) + kEnt * (sidx - bin_start);
        }
        __syncthreads();  // (tbs is read; its place is the ring's)
        const int fx = unpack3(my_f, 0), fy = unpack3(my_f, 1), fz = unpack3(my_f, 2);
        // the target's position inside its bin in bin units (lower-triangular cells)
        // (reciprocals and the hardware square root below: their few-ulp errors are far
        // inside the trimming margin pmargin)
        const float Oz = uz * a.inv_hcz, Oy = (uy - Oz * a.hcy) * a.inv_hby,
                    Ox = (ux - Oy * a.hbx - Oz * a.hcx) * a.inv_hax;
        const float Oxp = Ox + (float)a.P[0];  // (orthorhombic rows: x bins from the region's first)
        const float Oxp4 = 4.f * Oxp, inv_hax4 = 4.f * a.inv_hax;  // in quarter bins (exact scalings)

        // (QS 1: rprune2 - gz^2 of the layer oz = gz_oz, kept while the rows of one z
        // layer go by; gz_oz is uniform)
        float gzz = 0.f;
        int gz_oz = -1;
        const int rb_lane = (lz * R1 + ly) * R0 + lx;  // the first bin of the lane's first row
        // candidate range of row (oz, oy) of this lane, as chunk-local byte offsets;
        // empty when the padded cutoff sphere misses the row
        auto row_range = [&](int oz, int oy, int c0, int c1) -> int2 {
            int xlo = 0, xhi = nrx - 1;
            int ql = 0, qh = 0;  // first and last quarter, in the row's quarters
            if (QS == 1 || (QS == 0 && a.lowtri == 2)) {
                // orthorhombic: the row's bins span y in [py, py + 1] hby and z in
                // [pz, pz + 1] hcz around the target; their gaps (less the margin) bound the
                // distance from below, and the x range follows without shear
                const float py = (float)(oy - a.P[1]) - Oy;
                const float gy = fmaxf(fmaxf(fmaf(py, a.hby, -a.pmargin), fmaf(-py, a.hby, a.gy_off)), 0.f);
                float rem2;
                if constexpr (QS == 1) {
                    if (oz != gz_oz) {
                        const float pz = (float)(oz - a.P[2]) - Oz;
                        const float gz = fmaxf(fmaxf(fmaf(pz, a.hcz, -a.pmargin), fmaf(-pz, a.hcz, a.gz_off)), 0.f);
                        gzz = fmaf(-gz, gz, a.rprune2);
                        gz_oz = oz;
                    }
                    rem2 = fmaf(-gy, gy, gzz);
                } else {
                    const float pz = (float)(oz - a.P[2]) - Oz;
                    const float gz = fmaxf(fmaxf(fmaf(pz, a.hcz, -a.pmargin), fmaf(-pz, a.hcz, a.gz_off)), 0.f);
                    rem2 = fmaf(-gz, gz, fmaf(-gy, gy, a.rprune2));
                }
                if (rem2 < 0.f) return make_int2(0, 0);
                const float rem = __builtin_amdgcn_sqrtf(rem2);
                if constexpr (QS == 1) {
                    // (4 floor(u) + quarter = floor(4 u): the bins are those of floor(u))
                    ql = max((int)floorf(fmaf(-rem, inv_hax4, Oxp4)), 0);
                    qh = min((int)floorf(fmaf(rem, inv_hax4, Oxp4)), 4 * nrx - 1);
                } else {
                    xlo = max((int)floorf(fmaf(-rem, a.inv_hax, Oxp)), 0);
                    xhi = min((int)floorf(fmaf(rem, a.inv_hax, Oxp)), nrx - 1);
                    if (xlo > xhi) return make_int2(0, 0);
                }
            } else if (QS == 2 || (QS == 0 && a.lowtri)) {
                // bounding box of the row (bins py, pz relative to the target's bin, all x)
                // in Cartesian y and z, from the target: its gaps gy, gz bound the distance
                // from below; the x range that the (padded) cutoff sphere can reach then
                // follows from the row's x shear
                const float py = (float)(oy - a.P[1]) - Oy, pz = (float)(oz - a.P[2]) - Oz;
                const float zl = pz * a.hcz, zh = zl + a.hcz;
                const float cyl = fminf(pz * a.hcy, (pz + 1.f) * a.hcy);
                const float cyh = fmaxf(pz * a.hcy, (pz + 1.f) * a.hcy);
                const float yl = py * a.hby + cyl, yh = (py + 1.f) * a.hby + cyh;
                float gy = fmaxf(fmaxf(yl, -yh), 0.f), gz = fmaxf(fmaxf(zl, -zh), 0.f);
                gy = fmaxf(gy - a.pmargin, 0.f);
                gz = fmaxf(gz - a.pmargin, 0.f);
                const float rem2 = a.rprune2 - gy * gy - gz * gz;
                if (rem2 < 0.f) return make_int2(0, 0);
                const float rem = __builtin_amdgcn_sqrtf(rem2);
                const float sl = fminf(py * a.hbx, (py + 1.f) * a.hbx) + fminf(pz * a.hcx, (pz + 1.f) * a.hcx);
                const float sh = fmaxf(py * a.hbx, (py + 1.f) * a.hbx) + fmaxf(pz * a.hcx, (pz + 1.f) * a.hcx);
                if constexpr (QS == 2) {
                    // in quarter bins, as the orthorhombic rows: an entry of the first bin
                    // whose a fraction is below u - xlo lies at least rem below the target
                    // in x (its shear is at most sh), one of the last bin at or above
                    // w - xhi at least rem above it (its shear is at least sl)
                    ql = max((int)floorf(4.f * (Ox + (-rem - sh) * a.inv_hax)) + 4 * a.P[0], 0);
                    qh = min((int)floorf(4.f * (Ox + (rem - sl) * a.inv_hax)) + 4 * a.P[0], 4 * nrx - 1);
                } else {
                    xlo = max((int)floorf(Ox + (-rem - sh) * a.inv_hax) + a.P[0], 0);
                    xhi = min((int)floorf(Ox + (rem - sl) * a.inv_hax) + a.P[0], nrx - 1);
                    if (xlo > xhi) return make_int2(0, 0);
                }
            }
            const int rb = rb_lane + (oz * R1 + oy) * R0;
            if constexpr (QS != 0) {
                if (qsplit) {  // (uniform: the region's only chunk)
                    const int va = rq[4 * rb + ql], vb = rq[4 * rb + qh + 1];
                    return make_int2(va, max(va, vb));
                }
                xlo = ql >> 2;
                xhi = qh >> 2;
                if (xlo > xhi) return make_int2(0, 0);
            }
            const int va = max(rp[rb + xlo] - kEnt * c0, 0), vb = min(rp[rb + xhi + 1], kEnt * c1) - kEnt * c0;
            return va < vb ? make_int2(va, vb) : make_int2(0, 0);
        };
        if constexpr (!WRITE) {
            // ---------------- count pass
            const bool slots = slotted;
            uint32_t* const ring = sh.ring[threadIdx.x];
            // group g of this target's list
            auto group = [&](int g) { return (uint4*)a.words + ((uint64_t)(uint32_t)g * (uint64_t)(uint32_t)a.nrow + (uint32_t)j); };
            int found = 0, w = 0;  // edges, and row words recorded
            // Records the row whose last candidate is region index last, of n candidates with
            // the edge mask bits (bit i: candidate last - i).
            auto put_word = [&](uint32_t word, bool put) {  // (not put: overwritten by the next)
                ring[w & 3] = word;
                w += put ? 1 : 0;
                if (put && (w & 3) == 0 && w <= a.Kw) *group((w >> 2) - 1) = *(const uint4*)ring;
            };
            auto put_row = [&](uint32_t bits, int last) {
                found += __popc(bits);
                if (!slots) return;
                if (__builtin_expect(__builtin_amdgcn_ballot_w64(bits >> kWordBits != 0u) != 0ull, 0)) {
                    put_word(((uint32_t)(last - kWordBits) << kWordBits) | (bits >> kWordBits), bits >> kWordBits != 0u);
                    bits &= (1u << kWordBits) - 1u;
                }
                put_word(((uint32_t)last << kWordBits) | bits, bits != 0u);
            };

            // Bound by VALU issue and, per row, by the latency of its few LDS reads: 113M VALU
            // instructions at 1M atoms (r = 6, 90.5M edges) in 0.257 ms, against 159M in 0.345 ms
            // for a sweep that wrote a 2-byte entry per edge (two candidates a step, 34 VALU;
            // this one: four a step, 39), at four workgroups per CU to this one's five.
            // Where a row holds three candidates the width gains nothing: 35 against 33 us for the
            // degrees of 20000 atoms of 0.05 per cubic A, r = 4.5; 41 against 37 with the row words
            // and the region map, which take 5 us off the expansion.
            //
            // Sweeps this lane's target over the resident chunk c, in the fixed order (dz, dy, x,
            // atom) -- ascending region index.  The edge test is the sign bit of d2 - mid, shifted
            // into a mask register, one bit per candidate and four candidates per step; a row's
            // mask becomes its row word, so the loop holds no compare, counter or store per
            // candidate.  The rare candidate within the band around the cutoff, or at a distance
            // near zero, shows in two running minima: its row is then decided again, candidate
            // by candidate, with the exact test.  (The target itself is never read: as one of the
            // three past its piece's end, it had nearly every wave decide two pieces again, 121M
            // VALU instructions and 24 us more.)
            //
            // Rows are swept with one row of lookahead: the wave stays on row r until every
            // lane has finished its row r, and a lane that finishes early goes on into its row
            // r + 1 meanwhile, so a wave waits for its longest row less often.  Rows of more than
            // kRowMax candidates go in pieces.
            auto sweep = [&](int c) {
                constexpr int kPieceB = kEnt * kRowMax;
                static_assert(kRowMax % 4 == 0 && kRowMax < 32, "a piece's steps fit the mask register");
                // (entries of a byte offset b < 65536 that is a multiple of 12: b / 12)
                auto entries = [](int b) { return (int)(__umul24((uint32_t)b, 5462u) >> 16); };
                const int c0 = c * kCap;
                const int c1 = min(total, c0 + kCap);
                const int vs = v_self - kEnt * c0;
                const float nmid = -a.mid;
                int oz = 0, oy = 0;    // the next row (uniform); oz = nrz: none
                int fa = 0, fe = 0;    // what is left of the row taken last
                bool pend = false;     // some lane has some left
                bool center = false;   // that row is the target's own
                int lead = 0;          // candidates read before the start of the piece that ends there
                // The next piece: at most kRowMax candidates of the row, and up to the target's own
                // entry, which is skipped.  The piece that ends there takes its steps up to it, so
                // that none reads it; they start at up to three entries before the piece.
                auto next_piece = [&]() -> int2 {
                    if (!pend) {
                        const int2 r = row_range(oz, oy, c0, c1);
                        fa = r.x;
                        fe = active ? r.y : r.x;
                        center = oz == a.P[2] && oy == a.P[1];
                        const bool wrap = oy + 1 == nry;
                        oz += wrap ? 1 : 0;
                        oy = wrap ? 0 : oy + 1;
                    }
                    int pv = fa;
                    int pe = min(fe, pv + kPieceB);
                    fa = pe;
                    if (center) {
                        const bool self = vs >= pv && vs < pe;
                        pe = self ? vs : pe;
                        fa = self ? vs + kEnt : pe;
                        lead = self ? -entries(vs - pv) & 3 : lead;
                        pv = self ? pv - kEnt * lead : pv;
                    }
                    pend = __builtin_amdgcn_ballot_w64(fa < fe) != 0ull;
                    return make_int2(pv, pe);
                };
                const int2 piece0 = next_piece();
                int v = piece0.x, e = piece0.y;  // [v, e): this lane's unswept part of its current piece
                int ncur = e - v, ecur = e;   // the wave's piece: its bytes, and its end
                int2 nxt = next_piece();      // this lane's next piece
                uint32_t M = 0;               // the masks of this lane's pieces, newest bit lowest
                float near_hi = INFINITY, near_lo = INFINITY;  // least |d2 - mid|, least d2 - mid
                uint64_t again = 0ull;        // lanes whose next piece is to be decided again
                bool more = true, more2 = true;  // there is a next piece, and one after it
                do {
                    const int pv = nxt.x, pe = nxt.y;
                    more = more2;
                    // (the piece after the next is looked up before the steps, which hide its LDS
                    // reads)
                    more2 = more && (pend || oz < nrz);
                    nxt = make_int2(0, 0);
                    if (more2) nxt = next_piece();
                    const int nnext = pe - pv;
                    uint32_t Mp = M;              // the mask of this lane's current piece, when done
                    const bool done = v >= e;
                    uint64_t live = __builtin_amdgcn_ballot_w64(!done);
                    v = done ? pv : v;
                    e = done ? pe : e;
                    while (live != 0ull) {
                        if (v < e) {
                            // four candidates per step: those past the end or before the start
                            // (at most three, inside qbuf) leave bits that the piece's mask drops
                            struct F3 { float x, y, z; };
                            const F3* const q = (const F3*)(qb + v);
                            const F3 q0 = q[0], q1 = q[1], q2 = q[2], q3 = q[3];
                            auto dist = [&](const F3& p) {
                                const float dx = p.x - t0, dy = p.y - t1, dz = p.z - t2;
                                return fmaf(dz, dz, fmaf(dy, dy, fmaf(dx, dx, nmid)));
                            };
                            float d0 = dist(q0), d1 = dist(q1), d2 = dist(q2), d3 = dist(q3);
                            M = __builtin_amdgcn_alignbit(M, __float_as_uint(d0), 31);
                            M = __builtin_amdgcn_alignbit(M, __float_as_uint(d1), 31);
                            M = __builtin_amdgcn_alignbit(M, __float_as_uint(d2), 31);
                            M = __builtin_amdgcn_alignbit(M, __float_as_uint(d3), 31);
                            near_hi = fminf(fminf(near_hi, fabsf(d0)), fabsf(d1));
                            near_hi = fminf(fminf(near_hi, fabsf(d2)), fabsf(d3));
                            near_lo = fminf(fminf(near_lo, d0), d1);
                            near_lo = fminf(fminf(near_lo, d2), d3);
                        }
                        // (a lane at rest is not live, and stays at or past e)
                        const int nv = v + 4 * kEnt;
                        const uint64_t firstm = __builtin_amdgcn_ballot_w64(nv >= e) & live;
                        const bool first = __builtin_amdgcn_inverse_ballot_w64(firstm);
                        Mp = first ? M : Mp;
                        e = first ? pe : e;
                        v = first ? pv : nv;
                        live &= ~firstm;
                    }
                    // the piece is done in every lane: its candidates' bits, less those swept past
                    // its end or (in the piece that ends at the target) before its start
                    const int n = entries(ncur), before = ecur == vs ? lead : 0;
                    uint32_t bits = (Mp >> (-n & 3)) & ((1u << (n - before)) - 1u);
                    const uint64_t nearm = __builtin_amdgcn_ballot_w64(near_hi <= a.band) |
                                           __builtin_amdgcn_ballot_w64(near_lo <= a.low);
                    if (__builtin_expect((nearm | again) != 0ull, 0)) {
                        // (what the minima saw lies in this piece or, in the lookahead, the next)
                        if (__builtin_amdgcn_inverse_ballot_w64(nearm | again)) {
                            bits = 0;
                            for (int q = ecur - ncur + kEnt * before; q < ecur; q += kEnt) {
                                const float* const x = (const float*)(qb + q);
                                const float dx = x[0] - t0, dy = x[1] - t1, dz = x[2] - t2;
                                const float d = fmaf(dz, dz, fmaf(dy, dy, fmaf(dx, dx, nmid)));
                                bool edge = d < 0.f;
                                if (fabsf(d) <= a.band || d <= a.low) {
                                    // the source: its bin is the last that starts at or before it
                                    const SearchArgs& k = kernarg_search();
                                    const int at = q + kEnt * c0;
                                    int lo = 0, hi = k.nregion;
                                    while (hi - lo > 1) {
                                        const int mid = (lo + hi) >> 1;
                                        if (bin_first(mid) <= at) lo = mid; else hi = mid;
                                    }
                                    const int g = region_bin_start(k, g0, lo) + (at - bin_first(lo)) / kEnt;
                                    edge = exact_edge(k, k.sid[g], my_id, (double)dx, (double)dy, (double)dz);
                                }
                                bits = (bits << 1) | (edge ? 1u : 0u);
                            }
                            near_hi = near_lo = INFINITY;
                        }
                        again = nearm;
                    }
                    put_row(bits, entries(ecur) - 1 + c0);
                    ncur = nnext;
                    ecur = pe;
                } while (more);
            };

            const bool wave_active = __builtin_amdgcn_ballot_w64(active) != 0ull;
            for (int c = 0; c < nchunks; ++c) {
                ensure_chunk(c);
                if (c == 0 && k0 == 0 && slotted && threadIdx.x == 0)  // (its result is used after the sweep)
                    map_at = map_take(a, (int)(ord % a.npools), total);
                if (wave_active) sweep(c);
            }
            if (in_batch) {  // (inactive in the batch: masked, a ghost without edges)
                a.cnt[j] = found;
                if (slots) {
                    const bool over = w > a.Kw;
                    if ((w & 3) && !over) *group(w >> 2) = *(const uint4*)ring;
                    a.nw[j] = (uint8_t)(over ? kWordsOver : w);
                    over_any = over_any || over;
                }
                if (active && a.counts_user) a.counts_user[caller] = found;
                tile_found += found;
            }
            __syncthreads();
            continue;
        }

        // Sweeps this lane's target over the resident chunk c, in the count pass's order;
        // on_edge(v, k) receives every edge's byte offset in the chunk and its number.
        int found = 0;
        auto sweep = [&](int c, auto&& on_edge) {
            const int c0 = c * kCap;
            const int c1 = min(total, c0 + kCap);
            const int vs = v_self - kEnt * c0;
            for (int ri = 0; ri < nrz * nry; ++ri) {
                const int2 r = row_range(ri / nry, ri % nry, c0, c1);
                for (int v = r.x; v < r.y; v += kEnt) {
                    const float4 q = *(const float4*)(qb + v);
                    // d2 - toff with the offset in the innermost fma; edge iff its bits are
                    // below lo_bits (0 <= d2' < lo_off), band iff d2' <= hi_off
                    const float dx = q.x - t0, dy = q.y - t1, dz = q.z - t2;
                    const float d = fmaf(dz, dz, fmaf(dy, dy, fmaf(dx, dx, -a.toff)));
                    bool edge = __float_as_uint(d) < a.lo_bits;
                    if (!edge && d <= a.hi_off && v != vs)
                        edge = exact_edge(a, __float_as_int(q.w), my_id, (double)dx, (double)dy, (double)dz);
                    if (edge) on_edge(v, found++);
                }
            }
        };
        if constexpr (WRITE) {
        // ---------------- write pass
        const int mycnt = active ? a.cnt[j] : 0;
        int btot;
        const int ex = block_excl_scan<int, kBlock>(mycnt, sh.w32, &btot);
        // all of a tile without row words, or the targets whose list was too short
        const bool mine = active && (!slotted || a.nw[j] == kWordsOver);
        if (block_any<kBlock>(mine, sh.w32)) {
            const int64_t base = ebase + ex;
            for (int c = 0; c < nchunks; ++c) {
                ensure_chunk(c);
                if (!mine) continue;
                sweep(c, [&](int vb, int k) {
                    const int v = vb / kEnt;
                    if (k < mycnt) {
                        const uint32_t Tp = sh.T[v];
                        emit_edge(a, base + k, __float_as_int(((const float4*)qb)[v].w), my_id,
                                  unpack3(Tp, 0) + fx, unpack3(Tp, 1) + fy, unpack3(Tp, 2) + fz);
                    }
                });
            }
        }
        ebase += btot;
        }
        __syncthreads();
    }

    if constexpr (!WRITE) {
        // the tile's part of the region map, bin by bin (the last sweep is done: w64, bc free)
        bool mapped = false;
        int64_t mb = 0;
        if (slotted) {
            if (threadIdx.x == 0) {
                // (a full pool: the next ones are tried)
                const int64_t cap = a.mapcap / a.npools;
                int pool = (int)(ord % a.npools);
                for (int k = 1; (int64_t)map_at + total > cap && k < a.npools; ++k) {
                    pool = (pool + 1) % a.npools;
                    map_at = map_take(a, pool, total);
                }
                sh.bc[0] = (int64_t)map_at + total <= cap ? pool * cap + (int64_t)map_at : -1;
            }
            __syncthreads();
            mb = sh.bc[0];
            mapped = mb >= 0;
        }
        if (mapped) {
            // (the sweeps are done: the region's buffer holds the pairs, which then go out
            // side by side)
            const SearchArgs& k = kernarg_search();
            int2* const pair = (int2*)sh.qbuf;
            static_assert(sizeof(sh.qbuf) >= 8 * kCap, "the pairs of a chunk fit the region's buffer");
            for (int v0 = 0; v0 < total; v0 += kCap) {
#pragma unroll
                for (int h = 0; h < kRegPerThread; ++h) {
                    const int rb = kRegPerThread * threadIdx.x + h;
                    if (rb >= k.nregion) continue;
                    const int first = bin_first(rb) / kEnt - v0, end = bin_first(rb + 1) / kEnt - v0;
                    if (first >= end || end <= 0 || first >= kCap) continue;
                    int r[3], w[3], sb[3];
                    region_coords(k, rb, r);
                    region_wrap(k, g0, r, w, sb);
                    // (the fields of pack3 subtract without borrows: each stays within 10 bits)
                    const int T0 = (int)(pack3(sb[0], sb[1], sb[2]) + kZero3);
                    for (int v = max(first, 0); v < min(end, kCap); ++v)
                        pair[v] = make_int2(rst[h] + v - first, T0);
                }
                __syncthreads();
                int2* const to = k.map + mb + v0;
                for (int v = threadIdx.x; v < min(total - v0, kCap); v += kBlock) {
                    const int2 p = pair[v];
                    to[v] = make_int2(p.x, p.y - (int)k.sflr[p.x]);
                }
                __syncthreads();
            }
        }
        int64_t tt;
        block_excl_scan<int64_t, kBlock>(tile_found, sh.w64, &tt);
        const bool over = block_any<kBlock>(over_any, sh.w32);
        const int fix = mapped ? (over ? kFixOver : 0) : kFixChunked;
        out.tt = tt;
        out.fix = fix;
        if (threadIdx.x == 0) {
            a.ttot[ord] = (int)tt;
            a.tfix[ord] = fix;
            a.tmap[ord] = make_int2((int)mb, total);
            if (fix && flag_clear(&a.totals[3]))  // the fix-up pass has work
                atomicOr((unsigned long long*)&a.totals[3], 1ull);
        }
    }
    return out;
}

// MODE 0 (count) and MODE 1 (fix-up write): one tile per workgroup.
// QS: the count with quarter-bin row ends (1: orthorhombic cells, 2: other lower-triangular
// cells; cell list ordered by bin_xkey).
template <int MODE, int QS = 0>
__global__ __launch_bounds__(kBlock, MODE == 0 ? kCountWaves : 1) void search_kernel(SearchArgs a)
{
    if constexpr (MODE == 0) {
        __shared__ CountLds sh;
        search_tile<0, QS>(a, sh, blockIdx.x);
    } else {
        __shared__ FixLds f;
        // (written here, in the build's last launch: a fill of its own took 4.5 us)
        if (a.n_out && blockIdx.x == 0 && threadIdx.x == 0) *a.n_out = a.totals[0];
        // a grid of at most DG_FIXGRID workgroups walks the tiles: most have nothing to do,
        // and in most builds no tile has (the count pass raises totals[3] when one does)
        if (a.totals[3] == 0) return;
        for (int64_t ord = blockIdx.x; ord < a.ntiles; ord += gridDim.x) {
            if (a.tfix[ord] == 0) continue;
            search_tile<1>(a, f, ord);
            __syncthreads();  // before the next tile reuses the LDS
        }
    }
}

// The positions in cell-list order (entry g: atom sid[g]), for the edge vectors: the
// expansion then reads a tile's sources from a few contiguous runs instead of from all
// over the caller's order.
__global__ void cell_pos_kernel(int64_t n, const int* __restrict__ sid, const void* __restrict__ pos,
                                int f64, void* __restrict__ cpos)
{
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n) return;
    const int64_t i = sid[g];
    if (f64) {
        const double* ps = (const double*)pos + 3 * i;
        double* pc = (double*)cpos + 3 * g;
        pc[0] = ps[0]; pc[1] = ps[1]; pc[2] = ps[2];
    } else {
        const float* ps = (const float*)pos + 3 * i;
        float* pc = (float*)cpos + 3 * g;
        pc[0] = ps[0]; pc[1] = ps[1]; pc[2] = ps[2];
    }
}

// The ids to write for the cell-list entries.
__global__ void cell_ids_kernel(int64_t n, const int* __restrict__ sid, const int64_t* __restrict__ out_ids,
                                int* __restrict__ wid)
{
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g < n) wid[g] = (int)out_ids[sid[g]];
}

// The write stage: every edge the count pass left as row words, S workgroups per tile.
// VT: the type of vector / distance outputs written in groups, else void.
template <typename VT, bool GROUPS>
__global__ __launch_bounds__(kBlock, expand_waves<VT>) void expand_kernel(SearchArgs a, int S)
{
    __shared__ ExpandLds<VT, GROUPS> sh;
    int64_t ord;
    int s;
    part_of(blockIdx.x, a.ntiles, S, &ord, &s);
    const int skew = GROUPS ? (int)(kSkewMax - (((uintptr_t)a.out_dst >> 3) & (kSkewMax - 1))) & (kSkewMax - 1) : 0;
    expand_part<VT, GROUPS>(a, sh, ord, s, S, skew);
}

// ---------------------------------------------------------------- all-pairs fallback
// Used only when the search region of a tile would exceed kMaxRegion bins (cutoff much
// larger than the cell).  One thread per target, every atom, and for each pair every
// periodic shift that can put the source within the cutoff (brute_kernel: the exact
// per-pair range).
struct BruteArgs {
    double C[9], Cinv[9];
    double r2;
    double cf[3];  // r / face distance per axis: the fractional reach of the cutoff sphere
    int pbc[3];
    const void* pos;
    int f64;
    int64_t n, nt;
    const int64_t* tgt;
    int* cnt;
    int* counts_user;
    const int64_t* offs;
    int64_t* out_src;
    int64_t* out_dst;
    float* out_shift;
    void* out_vec;
    void* out_dist;
    int vout_f64;
    int64_t capacity;
    int64_t* totals;
    const int64_t* out_ids;  // written for atom i: out_ids[i] (null: i)
    int64_t* n_out;          // as in SearchArgs
};

template <bool WRITE>
__global__ void brute_kernel(BruteArgs a)
{
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (WRITE && a.n_out && t == 0) *a.n_out = a.totals[0];
    if (t >= a.nt) return;
    int64_t tg = a.tgt ? a.tgt[t] : t;
    if (tg < 0 || tg >= a.n) {
        atomicOr((unsigned long long*)&a.totals[1], (unsigned long long)DG_FLAG_TARGET);
        if (!WRITE) { a.cnt[t] = 0; if (a.counts_user) a.counts_user[t] = 0; }
        return;
    }
    double pt[3], frt[3];
    load_pos(a.pos, a.f64, tg, pt);
    for (int d = 0; d < 3; ++d) frt[d] = canon_frac(pt[0], pt[1], pt[2], a.Cinv, d);
    int64_t o = WRITE ? a.offs[t] : 0;
    if (WRITE && a.offs[t + 1] > a.capacity) {
        atomicOr((unsigned long long*)&a.totals[1], (unsigned long long)kStatusCapacity);
        return;
    }
    int found = 0;
    for (int64_t j = 0; j < a.n; ++j) {
        double ps[3];
        load_pos(a.pos, a.f64, j, ps);
        // an edge's shift is its periodic image plus the floor difference of the two atoms
        // (radius_graph_kernels.cu:282-303); on a periodic axis every S with
        // |frt - frs - S| <= cf can be one (the source image is at least that fractional
        // distance times the face distance from the target), widened by 1e-9 against
        // rounding; without PBC only the floor difference
        int lo[3], hi[3];
        for (int d = 0; d < 3; ++d) {
            const double frs = canon_frac(ps[0], ps[1], ps[2], a.Cinv, d);
            if (a.pbc[d]) {
                lo[d] = (int)ceil(frt[d] - frs - a.cf[d] - 1e-9);
                hi[d] = (int)floor(frt[d] - frs + a.cf[d] + 1e-9);
            } else {
                lo[d] = hi[d] = (int)floor(frt[d]) - (int)floor(frs);
            }
        }
        for (int s0 = lo[0]; s0 <= hi[0]; ++s0)
            for (int s1 = lo[1]; s1 <= hi[1]; ++s1)
                for (int s2 = lo[2]; s2 <= hi[2]; ++s2) {
                    double v[3];
                    double d2 = canon_d2(ps, pt, s0, s1, s2, a.C, v);
                    if (!(d2 > kSelfThr && d2 <= a.r2)) continue;
                    if (WRITE) {
                        int64_t e = o + found;
                        a.out_src[e] = a.out_ids ? a.out_ids[j] : j;
                        a.out_dst[e] = a.out_ids ? a.out_ids[tg] : tg;
                        a.out_shift[3 * e] = (float)s0;
                        a.out_shift[3 * e + 1] = (float)s1;
                        a.out_shift[3 * e + 2] = (float)s2;
                        if (a.out_vec) {
                            if (a.vout_f64) {
                                double* ov = (double*)a.out_vec + 3 * e;
                                ov[0] = v[0]; ov[1] = v[1]; ov[2] = v[2];
                            } else {
                                float* ov = (float*)a.out_vec + 3 * e;
                                ov[0] = (float)v[0]; ov[1] = (float)v[1]; ov[2] = (float)v[2];
                            }
                        }
                        if (a.out_dist) {
                            if (a.vout_f64) ((double*)a.out_dist)[e] = sqrt(d2);
                            else ((float*)a.out_dist)[e] = (float)sqrt(d2);
                        }
                    }
                    ++found;
                }
    }
    if (!WRITE) {
        a.cnt[t] = found;
        if (a.counts_user) a.counts_user[t] = found;
    }
}

// ---------------------------------------------------------------- small utilities
__global__ void zero_i32_kernel(int* __restrict__ p, int64_t n)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

__global__ void zero_i64_kernel(int64_t* __restrict__ p, int64_t n)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

inline unsigned nblocks(int64_t n, int b = 256) { return (unsigned)((n + b - 1) / b); }

template <typename T>
inline T* at(void* ws, size_t off)
{
    return (T*)((char*)ws + off);
}

dg_status check_launch(const char* what)
{
    hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return fail(DG_ERR_HIP, std::string(what) + ": " + hipGetErrorString(e));
    return DG_OK;
}

// Opt-in stage timer: with RADIUS_PBC_PROFILE set in the environment (the switch of
// radius_graph_kernels.cu:444-465), a count or write call records a HIP event on its
// stream at every stage boundary, waits for the last one and prints each stage's time to
// stderr.  Off (the default) it does nothing: no events, no synchronisation.
struct StageTimer {
    static constexpr int kMax = 8;
    hipEvent_t ev[kMax];
    const char* name[kMax];
    int n = 0;
    bool on;
    hipStream_t s;
    explicit StageTimer(hipStream_t st) : on(getenv("RADIUS_PBC_PROFILE") != nullptr), s(st) {}
    // marks the end of stage `what` (the first mark opens the clock)
    void mark(const char* what)
    {
        if (!on || n >= kMax) return;
        if (hipEventCreate(&ev[n]) != hipSuccess) { on = false; return; }
        (void)hipEventRecord(ev[n], s);
        name[n++] = what;
    }
    void report(const char* call, const Plan& p, int64_t capacity)
    {
        if (!on || n < 2) { release(); return; }
        (void)hipEventSynchronize(ev[n - 1]);
        float total = 0;
        fprintf(stderr, "[radius_graph_pbc profile] %s: N=%lld targets=%lld bins=%dx%dx%d tiles=%lld "
                        "(%dx%dx%d bins) Kw=%d%s", call, (long long)p.n, (long long)p.nt, p.nb[0], p.nb[1],
                p.nb[2], (long long)p.ntiles, p.T[0], p.T[1], p.T[2], p.Kw, p.brute ? " all-pairs" : "");
        if (capacity >= 0) fprintf(stderr, " edge capacity=%lld", (long long)capacity);
        fprintf(stderr, "\n");
        for (int i = 1; i < n; ++i) {
            float ms = 0;
            (void)hipEventElapsedTime(&ms, ev[i - 1], ev[i]);
            total += ms;
            fprintf(stderr, "  %-22s %8.3f ms\n", name[i], ms);
        }
        fprintf(stderr, "  %-22s %8.3f ms\n", "total", total);
        release();
    }
    void release()
    {
        for (int i = 0; i < n; ++i) (void)hipEventDestroy(ev[i]);
        n = 0;
    }
    ~StageTimer() { release(); }
};

// Validates the description and builds the plan (host only).
dg_status make_plan(const dg_graph_desc* d, Plan& p)
{
    if (!d) return fail(DG_ERR_INVALID, "desc is NULL");
    if (d->n_atoms < 0 || d->n_atoms > 0x7ffffff0LL)
        return fail(DG_ERR_INVALID, "n_atoms must be in [0, 2^31)");
    if (d->has_targets && (d->n_targets < 0 || d->n_targets > 0x7ffffff0LL))
        return fail(DG_ERR_INVALID, "n_targets must be in [0, 2^31)");
    if (d->pos_dtype != DG_F32 && d->pos_dtype != DG_F64)
        return fail(DG_ERR_INVALID, "pos must be float32 or float64");
    if (!(d->radius > 0.0) || !isfinite(d->radius))
        return fail(DG_ERR_INVALID, "radius must be positive, got " + std::to_string(d->radius));
    for (int k = 0; k < 9; ++k)
        if (!isfinite(d->cell[k])) return fail(DG_ERR_INVALID, "cell must be finite");
    p = Plan();
    p.n = d->n_atoms;
    p.subset = d->has_targets ? 1 : 0;
    p.nt = d->has_targets ? d->n_targets : d->n_atoms;
    p.f64 = d->pos_dtype == DG_F64;
    if (plan_geometry(p, d->cell, d->pbc, d->radius)) return fail(DG_ERR_INVALID, "cell is singular");
    if (!(pair_images(p.cf, p.pbc) <= kMaxPairImages))
        return fail(DG_ERR_INVALID, "cell too thin for the radius: more than 2^24 periodic images per atom pair");
    plan_grid(p);
    plan_layout(p);
    if (p.nbins >= 0x7fffffffLL || p.ncodes >= 0x7fffffffLL)
        return fail(DG_ERR_INVALID, "grid too large");
    return DG_OK;
}

// 2: orthorhombic cell; 1: other lower-triangular cell (a along x, b in the xy plane,
// positive diagonal); 0: any other.
int cell_shape(const Plan& p)
{
    const bool low = p.C[1] == 0.0 && p.C[2] == 0.0 && p.C[5] == 0.0 && p.C[0] > 0.0 && p.C[4] > 0.0 &&
                     p.C[8] > 0.0;
    if (!low) return 0;
    return p.C[3] == 0.0 && p.C[6] == 0.0 && p.C[7] == 0.0 ? 2 : 1;
}

// The bin steps bin_xkey needs, as the search's arguments hold them.
XKey xkey_of(const Plan& p)
{
    XKey k;
    k.hbx = (float)(p.C[3] / p.nb[1]);
    k.hcx = (float)(p.C[6] / p.nb[2]);
    k.hcy = (float)(p.C[7] / p.nb[2]);
    k.inv_hby = (float)(p.nb[1] / p.C[4]);
    k.inv_hcz = (float)(p.nb[2] / p.C[8]);
    return k;
}

GridArgs grid_args(const Plan& p)
{
    GridArgs g;
    memcpy(g.C, p.C, sizeof g.C);
    memcpy(g.Cinv, p.Cinv, sizeof g.Cinv);
    for (int d = 0; d < 3; ++d) {
        g.nb[d] = p.nb[d]; g.T[d] = p.T[d]; g.ntl[d] = p.ntl[d]; g.mb[d] = p.mb[d];
    }
    g.tb = p.tb;
    return g;
}

SearchArgs search_args(const Plan& p, const void* pos, void* ws)
{
    SearchArgs a;
    memset(&a, 0, sizeof a);
    memcpy(a.C, p.C, sizeof a.C);
    memcpy(a.Cinv, p.Cinv, sizeof a.Cinv);
    for (int d = 0; d < 3; ++d)
        for (int c = 0; c < 3; ++c) a.hC[3 * d + c] = p.C[3 * d + c] / (double)p.nb[d];
    a.r2 = p.r2;
    a.lowtri = cell_shape(p);
    a.hax = (float)(p.C[0] / p.nb[0]);
    a.hbx = (float)(p.C[3] / p.nb[1]);
    a.hby = (float)(p.C[4] / p.nb[1]);
    a.hcx = (float)(p.C[6] / p.nb[2]);
    a.hcy = (float)(p.C[7] / p.nb[2]);
    a.hcz = (float)(p.C[8] / p.nb[2]);
    a.inv_hax = (float)(p.nb[0] / p.C[0]);
    a.inv_hby = (float)(p.nb[1] / p.C[4]);
    a.inv_hcz = (float)(p.nb[2] / p.C[8]);
    // row trimming must never drop a candidate the exact test could accept: pad the
    // cutoff by far more than the fp32 position error
    a.pmargin = (float)(1e-4 * p.r + 1e-3);
    a.rprune2 = (float)((p.r + 2.0 * a.pmargin) * (p.r + 2.0 * a.pmargin));
    a.gy_off = -a.hby - a.pmargin;
    a.gz_off = -a.hcz - a.pmargin;
    for (int d = 0; d < 3; ++d) {
        a.nb[d] = p.nb[d]; a.P[d] = p.P[d]; a.T[d] = p.T[d]; a.ntl[d] = p.ntl[d];
        a.R[d] = p.R[d]; a.pbc[d] = p.pbc[d];
    }
    a.tb = p.tb;
    a.nregion = p.nregion;
    a.inv_R0 = 1.0f / (float)p.R[0];
    a.inv_R01 = 1.0f / (float)(p.R[0] * p.R[1]);
    a.wrap1 = 1;
    for (int d = 0; d < 3; ++d) {
        a.inv_T[d] = 1.0f / (float)p.T[d];
        // (a region bin runs from -P to ntl T - 1 + P, and ntl T < nb + T)
        if (p.pbc[d] && p.nb[d] < p.T[d] + p.P[d]) a.wrap1 = 0;
    }
    a.xsplit = p.ntiles <= kSortTilesMax;  // (the per-bin sort above keeps bins in id order)
    a.ntiles = p.ntiles;
    a.toff = p.toff; a.hi_off = p.hi_off; a.lo_bits = p.lo_bits;
    a.spos = at<float4>(ws, p.o_spos);
    a.sflr = at<uint32_t>(ws, p.o_sflr);
    a.sid = at<int>(ws, p.o_sid);
    a.bstart = at<int>(ws, p.o_bstart);
    a.tile_of_rank = at<int>(ws, p.o_tor);
    a.rank_of_tile = at<int>(ws, p.o_rot);
    a.pos = pos;
    a.f64 = p.f64;
    a.subset = p.subset;
    a.tbstart = at<int>(ws, p.o_tbstart);
    a.tsidx = at<int>(ws, p.o_tsidx);
    a.tslot = at<int>(ws, p.o_tslot);
    a.cnt = at<int>(ws, p.o_cnt);
    a.ttot = at<int>(ws, p.o_ttot);
    a.tfix = at<int>(ws, p.o_tfix);
    a.tbase = at<int64_t>(ws, p.o_tbase);
    a.totals = at<int64_t>(ws, p.o_tot);
    // word rows: one per target, or per atom when the targets are the atoms with ids < nt
    // (every atom of a tile is then a lane)
    a.mid = p.mid; a.band = p.band; a.low = p.low;
    a.words = at<uint32_t>(ws, p.o_slot);
    a.nw = at<uint8_t>(ws, p.o_nw);
    a.Kw = p.Kw;
    a.nrow = p.nrow;
    a.map = at<int2>(ws, p.o_map);
    a.mapcap = p.mapcap;
    a.npools = p.npools;  // (64 tiles or more to one: their sizes even out; 128 bytes fit 8 per tile)
    a.tmap = at<int2>(ws, p.o_wgb);  // (free once the atoms and targets are sorted)
    a.wid = a.sid;
    a.ntarg = p.nt;
    // the prefix test runs with the tile-level sort only (the per-bin fallback sorts the
    // explicit targets as listed)
    a.pmis = p.subset && p.ntiles <= kSortTilesMax ? at<int64_t>(ws, p.o_tot) + 2 : nullptr;
    return a;
}

BruteArgs brute_args(const Plan& p, const void* pos, const int64_t* tgt, void* ws)
{
    BruteArgs b;
    memset(&b, 0, sizeof b);
    memcpy(b.C, p.C, sizeof b.C);
    memcpy(b.Cinv, p.Cinv, sizeof b.Cinv);
    b.r2 = p.r2;
    for (int d = 0; d < 3; ++d) { b.pbc[d] = p.pbc[d]; b.cf[d] = p.cf[d]; }
    b.pos = pos;
    b.f64 = p.f64;
    b.n = p.n;
    b.nt = p.nt;
    b.tgt = p.subset ? tgt : nullptr;
    b.cnt = at<int>(ws, p.o_cnt);
    b.offs = at<int64_t>(ws, p.o_tbase);
    b.totals = at<int64_t>(ws, p.o_tot);
    return b;
}

// Dynamic LDS beyond the default 64 KiB for kernel fn (gfx950 allows up to 160 KiB per
// workgroup); the attribute is raised once per kernel and size.
static void allow_dyn_lds(const void* fn, size_t bytes)
{
    if (bytes <= 65536) return;
    static std::mutex mu;
    static std::vector<std::pair<const void*, size_t>> done;
    std::lock_guard<std::mutex> lock(mu);
    for (auto& d : done)
        if (d.first == fn && d.second >= bytes) return;
    if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) == hipSuccess)
        done.emplace_back(fn, bytes);
}

// Workgroups of sort_big_bins_kernel: about 1024 bins each, at most 2048.
static unsigned big_bins_grid(int64_t nbins)
{
    return (unsigned)std::max<int64_t>(1, std::min<int64_t>(2048, (nbins + 1023) / 1024));
}

// Steps 1-5 of a build: Morton tile ranks, counting sort of the atoms (and of the
// explicit targets) into the SFC-ordered cell list.
void launch_sort(const Plan& p, const void* pos, const int64_t* target_idx, void* ws,
                 int64_t* totals, hipStream_t s)
{
    GridArgs g = grid_args(p);
    int* bcnt = at<int>(ws, p.o_bcnt);
    int* bstart = at<int>(ws, p.o_bstart);
    if (p.ntiles <= kSortTilesMax) {
        // 1. Morton rank of the tiles (and cleared tile counts)
        int* tcnt = at<int>(ws, p.o_tcnt);
        int* tstart = at<int>(ws, p.o_tstart);
        int* wgb = at<int>(ws, p.o_wgb);
        hipLaunchKernelGGL(tile_rank_kernel, dim3((unsigned)std::min<int64_t>(nblocks(p.ntiles), 2048)),
                           dim3(256), 0, s, g, p.ntiles, at<int>(ws, p.o_tor), at<int>(ws, p.o_rot), tcnt,
                           p.ntiles, totals, at<int64_t>(ws, p.o_tbase));
        // 2. wrap, bin key and cell-list record of every atom
        hipLaunchKernelGGL(bin_atoms_kernel, dim3(nblocks(p.n)), dim3(256), 0, s, g, pos, p.f64, p.n,
                           (const int*)at<int>(ws, p.o_rot), at<uint32_t>(ws, p.o_key),
                           (uint32_t*)nullptr, (int*)nullptr, at<float4>(ws, p.o_rec), totals);
        // 3-5. tile buckets, then each tile's bins in LDS
        const unsigned nch = (unsigned)std::max<int64_t>(1, std::min<int64_t>(kSortChunks, (p.n + 4095) / 4096));
        const size_t hl = 4 * (size_t)p.ntiles;
        allow_dyn_lds((const void*)tile_hist_kernel, hl);
        // 32-bit bucket entries when every id (atom, and target position) fits 24 bits
        const bool narrow = p.n < (1 << 24) && (!p.subset || p.nt < (1 << 24));
        allow_dyn_lds(narrow ? (const void*)tile_scatter_kernel<uint32_t> : (const void*)tile_scatter_kernel<uint64_t>, hl);
        const int64_t* always = nullptr;
        hipLaunchKernelGGL(tile_hist_kernel, dim3(nch), dim3(1024), hl, s, p.n, p.tb, p.ntiles,
                           (const uint32_t*)at<uint32_t>(ws, p.o_key), tcnt, wgb, always);
        if (narrow)
            hipLaunchKernelGGL(tile_scatter_kernel<uint32_t>, dim3(nch), dim3(1024), hl, s, p.n, p.tb, p.ntiles,
                               (const uint32_t*)at<uint32_t>(ws, p.o_key), (const int*)tcnt, tstart,
                               (const int*)wgb, at<uint32_t>(ws, p.o_arr), always);
        else
            hipLaunchKernelGGL(tile_scatter_kernel<uint64_t>, dim3(nch), dim3(1024), hl, s, p.n, p.tb, p.ntiles,
                               (const uint32_t*)at<uint32_t>(ws, p.o_key), (const int*)tcnt, tstart,
                               (const int*)wgb, at<uint64_t>(ws, p.o_arr), always);
        TileSortOut o;
        memset(&o, 0, sizeof o);
        o.rec = at<float4>(ws, p.o_rec);
        o.spos = at<float4>(ws, p.o_spos);
        o.sflr = at<uint32_t>(ws, p.o_sflr);
        o.sid = at<int>(ws, p.o_sid);
        o.inv = p.subset ? at<int>(ws, p.o_inv) : (int*)nullptr;
        o.stmp = at<void>(ws, p.o_stmp);
        o.xflag = totals + 4;
        o.xorder = cell_shape(p) != 0;  // (the count cuts bins by x in lower-triangular cells)
        o.xk = xkey_of(p);
        if (narrow)
            hipLaunchKernelGGL((tile_sort_kernel<false, uint32_t>), dim3((unsigned)p.ntiles), dim3(256), 0, s, p.n,
                               p.tb, p.ntiles, (const int*)tstart, at<uint32_t>(ws, p.o_arr), bstart, o);
        else
            hipLaunchKernelGGL((tile_sort_kernel<false, uint64_t>), dim3((unsigned)p.ntiles), dim3(256), 0, s, p.n,
                               p.tb, p.ntiles, (const int*)tstart, at<uint64_t>(ws, p.o_arr), bstart, o);
        if (p.subset) {
            // the explicit targets through the same tile-level sort: keyed by their atom's
            // bin, ordered by caller position inside a bin -- unless they are exactly
            // 0 .. nt - 1 (target_prefix_kernel leaves totals[2] at 0): then the kernels below
            // exit at once and the count takes the atoms of each tile with ids < nt
            hipLaunchKernelGGL(target_prefix_kernel, dim3((unsigned)std::min<int64_t>(nblocks(p.nt), 2048)), dim3(256),
                               0, s, p.nt, p.n, target_idx, totals);
            const int64_t* listed = totals + 2;
            uint32_t* tkey = at<uint32_t>(ws, p.o_tkey);
            hipLaunchKernelGGL(target_keys_kernel, dim3((unsigned)std::min<int64_t>(nblocks(std::max(p.nt, p.ntiles)), 4096)),
                               dim3(256), 0, s, p.nt, p.n, target_idx, (const uint32_t*)at<uint32_t>(ws, p.o_key),
                               tkey, tcnt, p.ntiles, totals);
            const unsigned tch = (unsigned)std::max<int64_t>(1, std::min<int64_t>(kSortChunks, (p.nt + 4095) / 4096));
            hipLaunchKernelGGL(tile_hist_kernel, dim3(tch), dim3(1024), hl, s, p.nt, p.tb, p.ntiles,
                               (const uint32_t*)tkey, tcnt, wgb, listed);
            if (narrow)
                hipLaunchKernelGGL(tile_scatter_kernel<uint32_t>, dim3(tch), dim3(1024), hl, s, p.nt, p.tb, p.ntiles,
                                   (const uint32_t*)tkey, (const int*)tcnt, tstart, (const int*)wgb,
                                   at<uint32_t>(ws, p.o_tarr), listed);
            else
                hipLaunchKernelGGL(tile_scatter_kernel<uint64_t>, dim3(tch), dim3(1024), hl, s, p.nt, p.tb, p.ntiles,
                                   (const uint32_t*)tkey, (const int*)tcnt, tstart, (const int*)wgb,
                                   at<uint64_t>(ws, p.o_tarr), listed);
            TileSortOut ot;
            memset(&ot, 0, sizeof ot);
            ot.inv = at<int>(ws, p.o_inv);
            ot.tgt = target_idx;
            ot.natoms = p.n;
            ot.tslot = at<int>(ws, p.o_tslot);
            ot.tsidx = at<int>(ws, p.o_tsidx);
            ot.run_if = listed;
            ot.stmp = at<void>(ws, p.o_stmp);
            if (narrow)
                hipLaunchKernelGGL((tile_sort_kernel<true, uint32_t>), dim3((unsigned)p.ntiles), dim3(256), 0, s,
                                   p.nt, p.tb, p.ntiles, (const int*)tstart,
                                   at<uint32_t>(ws, p.o_tarr), at<int>(ws, p.o_tbstart), ot);
            else
                hipLaunchKernelGGL((tile_sort_kernel<true, uint64_t>), dim3((unsigned)p.ntiles), dim3(256), 0, s,
                                   p.nt, p.tb, p.ntiles, (const int*)tstart,
                                   at<uint64_t>(ws, p.o_tarr), at<int>(ws, p.o_tbstart), ot);
        }
        return;
    } else {
    // 1. Morton rank of the tiles (and cleared bin counts)
    hipLaunchKernelGGL(tile_rank_kernel, dim3((unsigned)std::min<int64_t>(nblocks(p.nbins), 2048)), dim3(256),
                       0, s, g, p.ntiles, at<int>(ws, p.o_tor), at<int>(ws, p.o_rot), bcnt, p.nbins, totals,
                       at<int64_t>(ws, p.o_tbase));
    // 2-5. counting sort of the atoms into SFC-ordered bins (per-bin device atomics)
    hipLaunchKernelGGL(bin_atoms_kernel, dim3(nblocks(p.n)), dim3(256), 0, s, g, pos, p.f64, p.n,
                       (const int*)at<int>(ws, p.o_rot), at<uint32_t>(ws, p.o_key),
                       at<uint32_t>(ws, p.o_rank), bcnt, at<float4>(ws, p.o_rec), totals);
    device_excl_scan<int, int>(bcnt, p.nbins, bstart, at<int>(ws, p.o_part), s);
    hipLaunchKernelGGL(scatter_atoms_kernel, dim3(nblocks(p.n)), dim3(256), 0, s, p.n,
                       (const uint32_t*)at<uint32_t>(ws, p.o_key),
                       (const uint32_t*)at<uint32_t>(ws, p.o_rank), (const int*)bstart,
                       at<int>(ws, p.o_arr));
    hipLaunchKernelGGL(sort_big_bins_kernel, dim3(big_bins_grid(p.nbins)), dim3(kSegSortThreads), 0, s, p.nbins,
                       (const int*)bstart, at<uint32_t>(ws, p.o_arr), at<uint32_t>(ws, p.o_stmp));
    hipLaunchKernelGGL(order_atoms_kernel, dim3(nblocks(p.n)), dim3(256), 0, s, p.n,
                       (const uint32_t*)at<uint32_t>(ws, p.o_key), (const int*)bstart,
                       (const int*)at<int>(ws, p.o_arr), (const float4*)at<float4>(ws, p.o_rec),
                       at<float4>(ws, p.o_spos), at<uint32_t>(ws, p.o_sflr), at<int>(ws, p.o_sid),
                       p.subset ? at<int>(ws, p.o_inv) : (int*)nullptr);
    }
    if (p.subset) {
        int* tbcnt = at<int>(ws, p.o_tbcnt);
        int* tbstart = at<int>(ws, p.o_tbstart);
        hipLaunchKernelGGL(zero_i32_kernel, dim3(nblocks(p.nbins)), dim3(256), 0, s, tbcnt, p.nbins);
        hipLaunchKernelGGL(bin_targets_kernel, dim3(nblocks(p.nt)), dim3(256), 0, s, p.nt, p.n,
                           target_idx, (const uint32_t*)at<uint32_t>(ws, p.o_key),
                           at<uint32_t>(ws, p.o_tkey), at<uint32_t>(ws, p.o_trank), tbcnt, totals);
        device_excl_scan<int, int>(tbcnt, p.nbins, tbstart, at<int>(ws, p.o_part), s);
        hipLaunchKernelGGL(scatter_targets_kernel, dim3(nblocks(p.nt)), dim3(256), 0, s, p.nt,
                           (const uint32_t*)at<uint32_t>(ws, p.o_tkey),
                           (const uint32_t*)at<uint32_t>(ws, p.o_trank), (const int*)tbstart,
                           at<int>(ws, p.o_tslot));
        hipLaunchKernelGGL(sort_big_bins_kernel, dim3(big_bins_grid(p.nbins)), dim3(kSegSortThreads), 0, s,
                           p.nbins, (const int*)tbstart, at<uint32_t>(ws, p.o_tslot), at<uint32_t>(ws, p.o_stmp));
        hipLaunchKernelGGL(finish_targets_kernel, dim3(nblocks(p.nbins)), dim3(256), 0, s, p.nbins,
                           p.n, (const int*)tbstart, at<int>(ws, p.o_tslot), target_idx,
                           (const int*)at<int>(ws, p.o_inv), at<int>(ws, p.o_tsidx));
    }
}

void launch_count_kernel(const SearchArgs& a, unsigned grid, hipStream_t s)
{
    if (a.lowtri == 2 && a.xsplit)
        hipLaunchKernelGGL((search_kernel<0, 1>), dim3(grid), dim3(kBlock), 0, s, a);
    else if (a.lowtri == 1 && a.xsplit)
        hipLaunchKernelGGL((search_kernel<0, 2>), dim3(grid), dim3(kBlock), 0, s, a);
    else
        hipLaunchKernelGGL((search_kernel<0, 0>), dim3(grid), dim3(kBlock), 0, s, a);
}

}  // namespace dg

using namespace dg;

extern "C" {

const char* dg_last_error(void) { return g_last_error.c_str(); }

const char* dg_version(void) { return "dynamis_graph 0.1 gfx950"; }

size_t dg_graph_workspace_size(const dg_graph_desc* desc)
{
    Plan p;
    if (make_plan(desc, p) != DG_OK) return 0;
    return p.ws_bytes;
}

// The count stage; without words (counts only) the sweep records no row words, and a
// dg_graph_write that follows writes every tile from its fix-up pass instead.  Without sums
// (degrees only) the tiles' offsets and the total are not made: one launch less, 5 us where the
// degrees of 62500 targets among 500k atoms take 124, those of the smallest boxes 98.
static dg_status count_stage(const dg_graph_desc* desc, const void* pos, const int64_t* target_idx,
                             void* ws, size_t ws_bytes, int32_t* counts_out, bool words, bool sums, hipStream_t s)
{
    Plan p;
    dg_status st = make_plan(desc, p);
    if (st != DG_OK) return st;
    if (!ws || ws_bytes < p.ws_bytes) return fail(DG_ERR_WORKSPACE, "workspace too small");
    if (p.n > 0 && !pos) return fail(DG_ERR_INVALID, "pos is NULL");
    if (p.subset && p.nt > 0 && !target_idx) return fail(DG_ERR_INVALID, "target_idx is NULL");
    g_last_error.clear();
    int64_t* totals = at<int64_t>(ws, p.o_tot);
    if (p.n == 0 || p.nt == 0 || p.brute)  // (else tile_rank_kernel clears them)
        hipLaunchKernelGGL(zero_i64_kernel, dim3(1), dim3(64), 0, s, totals, (int64_t)8);
    if (p.n == 0 || p.nt == 0) {
        if (counts_out && p.nt > 0)
            hipLaunchKernelGGL(zero_i32_kernel, dim3(nblocks(p.nt)), dim3(256), 0, s, counts_out, p.nt);
        return check_launch("dg_graph_count(empty)");
    }
    if (p.brute) {
        BruteArgs b = brute_args(p, pos, target_idx, ws);
        b.counts_user = counts_out;
        hipLaunchKernelGGL(brute_kernel<false>, dim3(nblocks(p.nt, 64)), dim3(64), 0, s, b);
        if (sums)
            excl_scan<int, int64_t>(at<int>(ws, p.o_cnt), p.nt, at<int64_t>(ws, p.o_tbase),
                                    at<int64_t>(ws, p.o_part), s, totals);
        return check_launch("dg_graph_count(brute)");
    }
    StageTimer clk(s);
    clk.mark("start");
    launch_sort(p, pos, target_idx, ws, totals, s);
    clk.mark("sfc reorder + sort");
    // 6. degrees
    SearchArgs a = search_args(p, pos, ws);
    a.counts_user = counts_out;
    if (!words) a.words = nullptr;
    launch_count_kernel(a, (unsigned)p.ntiles, s);
    clk.mark("count");
    // 7. tile offsets in output order, and the total
    if (sums)
        excl_scan<int, int64_t>(at<int>(ws, p.o_ttot), p.ntiles, at<int64_t>(ws, p.o_tbase),
                                at<int64_t>(ws, p.o_part), s, totals);
    clk.mark("tile offset scan");
    st = check_launch("dg_graph_count");
    clk.report("dg_graph_count", p, -1);
    return st;
}

dg_status dg_graph_count(const dg_graph_desc* desc, const void* pos, const int64_t* target_idx,
                         void* ws, size_t ws_bytes, int32_t* counts_out, hipStream_t s)
{
    return count_stage(desc, pos, target_idx, ws, ws_bytes, counts_out, true, true, s);
}

dg_status dg_graph_counts(const dg_graph_desc* desc, const void* pos, const int64_t* target_idx,
                          void* ws, size_t ws_bytes, int32_t* counts_out, hipStream_t s)
{
    return count_stage(desc, pos, target_idx, ws, ws_bytes, counts_out, false, true, s);
}

dg_status dg_graph_degrees(const dg_graph_desc* desc, const void* pos, const int64_t* target_idx,
                           void* ws, size_t ws_bytes, int32_t* counts_out, hipStream_t s)
{
    return count_stage(desc, pos, target_idx, ws, ws_bytes, counts_out, false, false, s);
}

dg_status dg_graph_read_totals(const dg_graph_desc* desc, const void* ws, int64_t* total_edges,
                               int64_t* flags, hipStream_t s)
{
    Plan p;
    dg_status st = make_plan(desc, p);
    if (st != DG_OK) return st;
    // a small pinned buffer per host thread (allocated on its first call, kept): the copy
    // then goes straight to it instead of through a pageable staging path
    thread_local int64_t* pinned = nullptr;
    if (!pinned && hipHostMalloc((void**)&pinned, 2 * sizeof(int64_t), hipHostMallocDefault) != hipSuccess) {
        pinned = nullptr;
        (void)hipGetLastError();  // (the pageable fallback below; no stale error for later checks)
    }
    int64_t hbuf[2] = {0, 0};
    int64_t* h = pinned ? pinned : hbuf;
    h[0] = h[1] = 0;
    hipError_t e = hipMemcpyAsync(h, at<int64_t>((void*)ws, p.o_tot), 2 * sizeof(int64_t), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return fail(DG_ERR_HIP, std::string("read totals: ") + hipGetErrorString(e));
    if (total_edges) *total_edges = h[0];
    if (flags) *flags = h[1];
    if (h[1] & (DG_FLAG_RANGE | DG_FLAG_NONFINITE | DG_FLAG_TARGET)) {
        std::string m;
        if (h[1] & DG_FLAG_NONFINITE) m += "pos contains non-finite values; ";
        if (h[1] & DG_FLAG_RANGE) m += "an atom lies more than 255 cell lengths outside the cell; ";
        if (h[1] & DG_FLAG_TARGET) m += "target_indices out of range [0, N); ";
        return fail(DG_ERR_RANGE, m);
    }
    if (h[1] & DG_FLAG_CAPACITY) return fail(DG_ERR_CAPACITY, "edge capacity exceeded");
    return DG_OK;
}

dg_status dg_graph_write_n(const dg_graph_desc* desc, const void* pos, const int64_t* target_idx,
                           void* ws, size_t ws_bytes, int64_t capacity, const int64_t* out_ids,
                           int64_t* edge_src, int64_t* edge_dst, float* cell_shift, void* edge_vec,
                           void* edge_dist, int32_t vec_dtype, int64_t* n_edges, hipStream_t s)
{
    Plan p;
    dg_status st = make_plan(desc, p);
    if (st != DG_OK) return st;
    if (!ws || ws_bytes < p.ws_bytes) return fail(DG_ERR_WORKSPACE, "workspace too small");
    if (vec_dtype != DG_F32 && vec_dtype != DG_F64) return fail(DG_ERR_INVALID, "vec_dtype");
    if (capacity < 0) return fail(DG_ERR_INVALID, "capacity < 0");
    g_last_error.clear();
    if (p.n == 0 || p.nt == 0 || capacity == 0) return DG_OK;
    if (!edge_src || !edge_dst || !cell_shift) return fail(DG_ERR_INVALID, "edge outputs are NULL");
    if (!pos) return fail(DG_ERR_INVALID, "pos is NULL");
    if (p.subset && !target_idx) return fail(DG_ERR_INVALID, "target_idx is NULL");
    if (p.brute) {
        BruteArgs b = brute_args(p, pos, target_idx, ws);
        b.out_src = edge_src; b.out_dst = edge_dst; b.out_shift = cell_shift;
        b.out_vec = edge_vec; b.out_dist = edge_dist; b.vout_f64 = vec_dtype == DG_F64;
        b.capacity = capacity;
        b.out_ids = out_ids;
        b.n_out = n_edges;
        hipLaunchKernelGGL(brute_kernel<true>, dim3(nblocks(p.nt, 64)), dim3(64), 0, s, b);
        return check_launch("dg_graph_write(brute)");
    }
    SearchArgs a = search_args(p, pos, ws);
    a.out_src = edge_src; a.out_dst = edge_dst; a.out_shift = cell_shift;
    a.out_vec = edge_vec; a.out_dist = edge_dist; a.vout_f64 = vec_dtype == DG_F64;
    a.capacity = capacity;
    a.out_ids = out_ids;
    a.n_out = n_edges;
    if (out_ids) {
        // the ids to write in cell-list order (over the sort's scratch), so that the expansion
        // reads them from a tile's few runs
        int* wid = at<int>(ws, p.o_arr);
        hipLaunchKernelGGL(cell_ids_kernel, dim3(nblocks(p.n)), dim3(256), 0, s, (int64_t)p.n, a.sid, out_ids, wid);
        a.wid = wid;
    }
    StageTimer clk(s);
    clk.mark("start");
    // vectors / distances go out in 16-byte groups from bases aligned to 16 bytes, else
    // every edge is written by its lane
    const bool vec = edge_vec || edge_dist;
    const bool vec16 = vec && (((uintptr_t)edge_vec | (uintptr_t)edge_dist) & 15u) == 0;
    if (vec16) {
        a.cpos = at<char>(ws, p.o_cpos);
        hipLaunchKernelGGL(cell_pos_kernel, dim3(nblocks(p.n, 256)), dim3(256), 0, s, (int64_t)p.n,
                           (const int*)a.sid, pos, p.f64, (void*)a.cpos);
    }
    // parts per tile, from the edges expected: as many blocks to a part (whose setup costs about
    // as much as a block) as leave the chip a few rounds of workgroups
    const double per_tile = p.deg * (double)p.nt / (double)p.ntiles;
    const double part = kSub * std::min(std::max(floor((double)p.ntiles * per_tile / ((double)kSub * kPartsWanted)), 1.0), kPartBlocks);
    const int parts = (int)std::min({std::max(ceil(per_tile / part), 1.0), 64.0, floor(2147483647.0 / (double)p.ntiles)});
    const dim3 grid((unsigned)(p.ntiles * parts));
    if (vec16 && a.vout_f64)
        hipLaunchKernelGGL((expand_kernel<double, true>), grid, dim3(kBlock), 0, s, a, parts);
    else if (vec16)
        hipLaunchKernelGGL((expand_kernel<float, true>), grid, dim3(kBlock), 0, s, a, parts);
    else if (vec)
        hipLaunchKernelGGL((expand_kernel<void, false>), grid, dim3(kBlock), 0, s, a, parts);
    else
        hipLaunchKernelGGL((expand_kernel<void, true>), grid, dim3(kBlock), 0, s, a, parts);
    clk.mark("write (slot expansion)");
    hipLaunchKernelGGL(search_kernel<1>, dim3((unsigned)std::min<int64_t>(p.ntiles, kFixGrid)), dim3(kBlock), 0, s, a);
    clk.mark("write (fix-up)");
    st = check_launch("dg_graph_write");
    clk.report("dg_graph_write", p, capacity);
    return st;
}

dg_status dg_graph_write_ids(const dg_graph_desc* desc, const void* pos, const int64_t* target_idx,
                             void* ws, size_t ws_bytes, int64_t capacity, const int64_t* out_ids,
                             int64_t* edge_src, int64_t* edge_dst, float* cell_shift, void* edge_vec,
                             void* edge_dist, int32_t vec_dtype, hipStream_t s)
{
    return dg_graph_write_n(desc, pos, target_idx, ws, ws_bytes, capacity, out_ids, edge_src, edge_dst,
                            cell_shift, edge_vec, edge_dist, vec_dtype, nullptr, s);
}

dg_status dg_graph_write(const dg_graph_desc* desc, const void* pos, const int64_t* target_idx,
                         void* ws, size_t ws_bytes, int64_t capacity, int64_t* edge_src,
                         int64_t* edge_dst, float* cell_shift, void* edge_vec, void* edge_dist,
                         int32_t vec_dtype, hipStream_t s)
{
    return dg_graph_write_ids(desc, pos, target_idx, ws, ws_bytes, capacity, nullptr, edge_src, edge_dst,
                              cell_shift, edge_vec, edge_dist, vec_dtype, s);
}

dg_status dg_graph_build(const dg_graph_desc* desc, const void* pos, const int64_t* target_idx,
                         void* ws, size_t ws_bytes, int64_t capacity, int32_t* counts_out,
                         int64_t* edge_src, int64_t* edge_dst, float* cell_shift, void* edge_vec,
                         void* edge_dist, int32_t vec_dtype, hipStream_t s)
{
    // the write pass reads only device-side results of the count pass (per-tile offsets,
    // row words), so the two run back to back with no host round trip
    dg_status st = dg_graph_count(desc, pos, target_idx, ws, ws_bytes, counts_out, s);
    if (st != DG_OK) return st;
    return dg_graph_write(desc, pos, target_idx, ws, ws_bytes, capacity, edge_src, edge_dst,
                          cell_shift, edge_vec, edge_dist, vec_dtype, s);
}

}  // extern "C"

// ---------------------------------------------------------------- allocation-free build
// A device-resident workspace for dg_graph_build_noalloc: the build's whole workspace
// (cell list, row words, tile tables, totals) lives in this array, one copy per GPU, held from
// the library's load until the process ends.  Host code never names the array itself (its
// host-side symbol is no device address): it uses the address hipGetSymbolAddress
// returns on each device, kept in g_scratch_ptr.
namespace dg {
constexpr int kMaxDevices = 64;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];
static std::mutex g_scratch_mu;
static void* g_scratch_ptr[kMaxDevices];
// Overlap guard, per device: the stream of the last call and an event recorded behind it.
// A call on another stream while that event is still pending would share the scratch with
// work in flight, and is refused.  (Created once per device, with the scratch lookup.)
// A call holds its device's array (busy) from the check until its work is enqueued, so two
// host threads cannot both pass the check.
static hipEvent_t g_scratch_done[kMaxDevices];
static hipStream_t g_scratch_stream[kMaxDevices];
static bool g_scratch_used[kMaxDevices];
static bool g_scratch_busy[kMaxDevices];

// The scratch address on the current device, looked up once per device, and the device's
// array taken for this call (*dev_out; give it back with scratch_release).
// The stream must belong to the current device: the address is that device's copy.
static dg_status scratch_on_current_device(hipStream_t s, void** out, int* dev_out)
{
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return fail(DG_ERR_HIP, std::string("hipGetDevice: ") + hipGetErrorString(e));
    if (dev < 0 || dev >= kMaxDevices) return fail(DG_ERR_INVALID, "device ordinal out of range");
    if (s != nullptr) {
        hipDevice_t sdev = -1;
        e = hipStreamGetDevice(s, &sdev);
        if (e != hipSuccess) return fail(DG_ERR_HIP, std::string("hipStreamGetDevice: ") + hipGetErrorString(e));
        if (sdev != dev)
            return fail(DG_ERR_INVALID, "dg_graph_build_noalloc: the stream belongs to device " +
                                            std::to_string(sdev) + ", the current device is " + std::to_string(dev));
    }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr)
            return fail(DG_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
        e = hipEventCreateWithFlags(&g_scratch_done[dev], hipEventDisableTiming);
        if (e != hipSuccess)
            return fail(DG_ERR_HIP, std::string("hipEventCreateWithFlags: ") + hipGetErrorString(e));
        g_scratch_ptr[dev] = ptr;
    }
    // A stream under capture records no completion to test: such calls are not guarded.
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (s != nullptr) {
        e = hipStreamIsCapturing(s, &cap);
        if (e != hipSuccess) return fail(DG_ERR_HIP, std::string("hipStreamIsCapturing: ") + hipGetErrorString(e));
    }
    if (g_scratch_busy[dev])
        return fail(DG_ERR_INVALID, "dg_graph_build_noalloc: another call on this device is being enqueued "
                                    "(calls share the static scratch and must not overlap)");
    if (cap == hipStreamCaptureStatusNone && g_scratch_used[dev] && g_scratch_stream[dev] != s) {
        e = hipEventQuery(g_scratch_done[dev]);
        if (e == hipErrorNotReady)
            return fail(DG_ERR_INVALID, "dg_graph_build_noalloc: the previous call on this device (on another "
                                        "stream) has not completed; calls on different streams share the static "
                                        "scratch and must not overlap");
        if (e != hipSuccess) return fail(DG_ERR_HIP, std::string("hipEventQuery: ") + hipGetErrorString(e));
    }
    g_scratch_busy[dev] = true;
    *out = g_scratch_ptr[dev];
    *dev_out = dev;
    return DG_OK;
}

// Gives back device dev's array after a call on stream s: records the overlap guard's event
// behind whatever the call enqueued (not on a stream under capture).
static dg_status scratch_release(int dev, hipStream_t s)
{
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (s != nullptr && hipStreamIsCapturing(s, &cap) != hipSuccess) cap = hipStreamCaptureStatusActive;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    g_scratch_busy[dev] = false;
    if (cap != hipStreamCaptureStatusNone) return DG_OK;
    const hipError_t e = hipEventRecord(g_scratch_done[dev], s);
    if (e != hipSuccess) return fail(DG_ERR_HIP, std::string("hipEventRecord: ") + hipGetErrorString(e));
    g_scratch_stream[dev] = s;
    g_scratch_used[dev] = true;
    return DG_OK;
}

// Copies the build's {edge count, flags} to the caller's device buffer.
__global__ void copy_totals_kernel(const int64_t* __restrict__ totals, int64_t* __restrict__ out)
{
    if (threadIdx.x < 2) out[threadIdx.x] = totals[threadIdx.x];
}
}  // namespace dg

extern "C" dg_status dg_graph_build_noalloc(const dg_graph_desc* desc, const void* pos,
                                            const int64_t* target_idx, int64_t capacity,
                                            int32_t* counts_out, int64_t* edge_src,
                                            int64_t* edge_dst, float* cell_shift, void* edge_vec,
                                            void* edge_dist, int32_t vec_dtype,
                                            int64_t* totals_out, hipStream_t s)
{
    Plan p;
    dg_status st = make_plan(desc, p);
    if (st != DG_OK) return st;
    if (!totals_out) return fail(DG_ERR_INVALID, "totals_out is NULL");
    if (p.ws_bytes > kScratchBytes)
        return fail(DG_ERR_WORKSPACE, "dg_graph_build_noalloc: this build needs " +
                                          std::to_string(p.ws_bytes) + " bytes of workspace; the static "
                                          "scratch holds " + std::to_string(kScratchBytes) +
                                          " (use dg_graph_build with a caller workspace)");
    void* ws = nullptr;
    int dev = -1;
    st = scratch_on_current_device(s, &ws, &dev);
    if (st != DG_OK) return st;
    st = dg_graph_build(desc, pos, target_idx, ws, kScratchBytes, capacity, counts_out, edge_src,
                        edge_dst, cell_shift, edge_vec, edge_dist, vec_dtype, s);
    if (st == DG_OK) {
        hipLaunchKernelGGL(copy_totals_kernel, dim3(1), dim3(64), 0, s,
                           (const int64_t*)at<int64_t>(ws, p.o_tot), totals_out);
        st = check_launch("dg_graph_build_noalloc");
    }
    // (also after a failed call: whatever it enqueued still uses the array)
    const std::string err = st != DG_OK ? g_last_error : std::string();
    const dg_status rs = scratch_release(dev, s);
    if (st != DG_OK) {
        g_last_error = err;
        return st;
    }
    return rs;
}
