// nb_octree.hip -- Barnes-Hut octree build for gfx950.
//
// The reference builds its octree by lock-based top-down insertion
// (ParallelOctreeTopDownSubtrees.cpp:95-813): one work-group inserts every
// body down to level 7, then one work-group per subtree finishes the job.
// The resulting tree is the unique octree in which a cell is split iff it
// holds two or more bodies; only the node ids depend on the insertion race.
// This file builds that same tree without locks:
//
//  1. AABB (FP64 min/max including the origin) and cubify, on the device.
//  2. Per body, the first 21 octant digits with the reference's own FP64
//     classification chain: mid = cellMin + edge/2, digit = 4[y>mid_y] +
//     2[x>mid_x] + [z<mid_z], child min moved to mid on the x/y bits and on a
//     cleared z bit.  Digits are packed most significant first into a 63-bit
//     key, so key order is the reference's in-order body order.
//  3. Stable sort of (key, body).
//  4. Runs of bodies sharing all 21 digits get digits 21..41 and are sorted
//     inside the run (rare: bodies closer than edge/2^21).
//  5. lcp[i] = depth of the deepest cell holding sorted bodies i and i+1.
//     The internal cells are exactly the pairs (i, depth l) with
//     lcp[i-1] < l <= lcp[i]: each cell is numbered by the first adjacent pair
//     of its body range.  An exclusive scan of the chain lengths numbers the
//     internal cells k in depth-first pre-order; internal cell k stores its 8
//     children at node ids 1 + 8k + digit.
//  6. Parents come from a galloping search for the first body of the parent
//     cell; every cell and body learns the child slot (node) it fills.
//  7. Centre of mass level by level from the deepest cells up: a cell sums its
//     8 children in digit order 0..7 from 0.0 -- the reference's summation
//     (BarnesHutOctree.cpp:299-311), so every sum is bit-identical.  Cells
//     inside a block of 1024 sorted bodies are finished by that block's
//     workgroup in LDS; the few cells that cross block boundaries by one
//     workgroup per 64 blocks and one more.
//  8. Node records for traversal (COM = numerator / mass as the reference
//     divides per visit; an FP32 hi/lo record for the group traversal).  A
//     cell's edge is rootEdge * 2^-depth wherever it is needed.
#include <algorithm>
#include <cmath>

#include "nb_internal.h"

namespace nb {
namespace {

constexpr int kThreads = 256;

__device__ inline double sycl_min(double a, double b) { return b < a ? b : a; }
__device__ inline double sycl_max(double a, double b) { return a < b ? b : a; }

__device__ inline void raise_flag(TreeHdr *h, uint32_t f) { atomicOr(&h->status, f); }

// ---- 1. AABB ---------------------------------------------------------------
// Block partial extrema.  Like the reference's partials (BarnesHutOctree.cpp:
// 58-72, value-initialised to 0.0) every partial starts at the origin.  A
// seventh value says whether the block met a position that is not finite.
constexpr int kAabbThreads = 256;
constexpr int kAabbVals = 7;
struct Extents {
    double mn[3] = {0.0, 0.0, 0.0}, mx[3] = {0.0, 0.0, 0.0};
    bool bad = false;
};
// min/max are exact, so any reduction order gives the reference's result
__device__ inline void wave_extents(Extents &e) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            e.mn[c] = sycl_min(e.mn[c], __shfl_xor(e.mn[c], off, 64));
            e.mx[c] = sycl_max(e.mx[c], __shfl_xor(e.mx[c], off, 64));
        }
    }
    e.bad = __any(e.bad);
}

__global__ void __launch_bounds__(kAabbThreads) k_aabb_partial(const double *__restrict__ x,
                                                               const double *__restrict__ y,
                                                               const double *__restrict__ z,
                                                               uint32_t n, double *part) {
    __shared__ double sh[kAabbThreads / 64][kAabbVals];
    Extents e;
#pragma unroll 8
    for (uint64_t i = (uint64_t)blockIdx.x * kAabbThreads + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * kAabbThreads) {
        const double p[3] = {x[i], y[i], z[i]};
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            e.bad |= !isfinite(p[c]);
            e.mn[c] = sycl_min(e.mn[c], p[c]);
            e.mx[c] = sycl_max(e.mx[c], p[c]);
        }
    }
    wave_extents(e);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            sh[w][c] = e.mn[c];
            sh[w][3 + c] = e.mx[c];
        }
        sh[w][6] = e.bad ? 1.0 : 0.0;
    }
    __syncthreads();
    const uint32_t c = threadIdx.x;
    if (c < kAabbVals) {
        double v = sh[0][c];
        for (int k = 1; k < kAabbThreads / 64; ++k)
            v = c < 3 ? sycl_min(v, sh[k][c]) : sycl_max(v, sh[k][c]);
        part[(uint64_t)c * gridDim.x + blockIdx.x] = v;
    }
}

// Cubify the extents ext = {min_x, min_y, min_z, max_x, max_y, max_z}
// (BarnesHutOctree.cpp:161-190) to the root cube.
struct RootCube {
    double mn[3], mx[3], edge;
    bool ok;
};
__device__ inline RootCube cubify(const double ext[6]) {
    bool ok = true;
    double min_x = ext[0], min_y = ext[1], min_z = ext[2];
    double max_x = ext[3], max_y = ext[4], max_z = ext[5];
    const double x_length = fabs(max_x - min_x);
    const double y_length = fabs(max_y - min_y);
    const double z_length = fabs(max_z - min_z);
    // std::max(a, b) == (a < b) ? b : a
    const double yz = y_length < z_length ? z_length : y_length;
    const double maxEdgeLength = x_length < yz ? yz : x_length;
    if (maxEdgeLength == x_length) {
        min_z = min_z - ((maxEdgeLength - z_length) / 2);
        min_y = min_y - ((maxEdgeLength - y_length) / 2);
        max_z = max_z + ((maxEdgeLength - z_length) / 2);
        max_y = max_y + ((maxEdgeLength - y_length) / 2);
    } else if (maxEdgeLength == y_length) {
        min_x = min_x - ((maxEdgeLength - x_length) / 2);
        min_z = min_z - ((maxEdgeLength - z_length) / 2);
        max_x = max_x + ((maxEdgeLength - x_length) / 2);
        max_z = max_z + ((maxEdgeLength - z_length) / 2);
    } else if (maxEdgeLength == z_length) {
        min_x = min_x - ((maxEdgeLength - x_length) / 2);
        min_y = min_y - ((maxEdgeLength - y_length) / 2);
        max_x = max_x + ((maxEdgeLength - x_length) / 2);
        max_y = max_y + ((maxEdgeLength - y_length) / 2);
    } else {
        ok = false;
    }
    return RootCube{{min_x, min_y, min_z}, {max_x, max_y, max_z}, maxEdgeLength, ok};
}
__device__ inline void store_cube(TreeHdr *h, const RootCube &r) {
    h->minx = r.mn[0];
    h->miny = r.mn[1];
    h->minz = r.mn[2];
    h->maxx = r.mx[0];
    h->maxy = r.mx[1];
    h->maxz = r.mx[2];
    h->edge = r.edge;
}

// ---- 2. keys ---------------------------------------------------------------
__device__ inline uint64_t key_from(Cell &c, double px, double py, double pz) {
    uint64_t key = 0;
#pragma unroll
    for (int l = 0; l < kKeyLevels; ++l) key = (key << 3) | descend(c, px, py, pz);
    return key;
}

// Keys, identity permutation, and the packed body record {x, y, z, m} that
// the centre-of-mass and node-record passes gather (one 32-byte load).  Small
// jobs ride along, each of which took a launch of its own (3 to 5 us): every
// workgroup's first wave finds the root cube from the partial extents (at most
// kAabbBlocks of each), the first workgroup resets the header, and the sort's
// first digit is counted.  So there are at most 256 workgroups, which take
// their bodies in strides.
constexpr int kKeyThreads = 1024;
constexpr uint32_t kKeyBlocks = 256;
__global__ void __launch_bounds__(kKeyThreads) k_keys(
    const double *__restrict__ x, const double *__restrict__ y, const double *__restrict__ z,
    const double *__restrict__ m, uint32_t n, const double *__restrict__ part, uint32_t np,
    TreeHdr *h, uint64_t *skey, uint32_t *sidx, double4 *body4, uint32_t *scan_part,
    uint32_t scan_parts, RadixCount rc) {
    __shared__ RootCube root;
    __shared__ uint32_t hist[kRadixBins];
    const uint32_t t = threadIdx.x;
    if (t < 64) {
        Extents e;
#pragma unroll
        for (int k = 0; k < kAabbBlocks / 64; ++k) {
            const uint32_t p = t + 64u * k;
            if (p >= np) break;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                e.mn[c] = sycl_min(e.mn[c], part[(uint64_t)c * np + p]);
                e.mx[c] = sycl_max(e.mx[c], part[(uint64_t)(3 + c) * np + p]);
            }
            e.bad |= part[6ull * np + p] != 0.0;
        }
        wave_extents(e);
        const double ext[6] = {e.mn[0], e.mn[1], e.mn[2], e.mx[0], e.mx[1], e.mx[2]};
        const RootCube r = cubify(ext);
        if (t == 0) {
            root = r;
            if (blockIdx.x == 0) {
                store_cube(h, r);
                h->internal_count = 0;
                h->max_depth = 0;
                h->status = e.bad || !r.ok ? kFlagAabb : 0u;
                h->deep_runs = 0;
                h->stack_peak = 0;
                h->group_count = 0;
                h->group_next = 0;
                h->cross_count = 0;
            }
        }
    }
    if (t < kRadixBins) hist[t] = 0;
    __syncthreads();
    const uint64_t stride = (uint64_t)gridDim.x * kKeyThreads;
    const uint64_t i0 = (uint64_t)blockIdx.x * kKeyThreads + t;
    for (uint64_t i = i0; i < rc.plane_words; i += stride) rc.plane0[i] = 0;
    for (uint64_t i = i0; i < scan_parts; i += stride) scan_part[i] = 0;
    for (uint64_t i = i0; i < n; i += stride) {
        Cell c{root.mn[0], root.mn[1], root.mn[2], root.edge};
        const double px = x[i], py = y[i], pz = z[i];
        const uint64_t key = key_from(c, px, py, pz);
        skey[i] = key;
        sidx[i] = (uint32_t)i;
        body4[i] = make_double4(px, py, pz, m[i]);
        atomicAdd(&hist[(uint32_t)key & (kRadixBins - 1)], 1u);
    }
    if (!rc.total) return;  // nothing to sort
    __syncthreads();
    if (t < kRadixBins && hist[t]) atomicAdd(&rc.total[t], hist[t]);
}

// ---- 4./5. LCP and deep runs --------------------------------------------------
__device__ inline int lcp_depth(uint64_t a, uint64_t b) {
    // number of equal leading digits of two 63-bit keys (bit 63 is always 0)
    return (__clzll((long long)(a ^ b)) - 1) / 3;
}

// lcp of adjacent pair i (i + 1 < n); the first pair of a run of equal keys
// extends and sorts the run.  Shared by the one-system build and the
// workgroup-per-system ensemble build.
__device__ inline void lcp_at(uint32_t i, const double *__restrict__ x,
                              const double *__restrict__ y, const double *__restrict__ z,
                              uint32_t n, const Cell &root, TreeHdr *h, uint64_t *skey,
                              uint32_t *sidx, uint64_t *klo, int32_t *lcp) {
    const uint64_t k0 = skey[i], k1 = skey[i + 1];
    if (k0 != k1) {
        lcp[i] = lcp_depth(k0, k1);
        return;
    }
    if (i > 0 && skey[i - 1] == k0) return;  // not the first pair of the run
    // run [a, b] of bodies sharing all 21 digits: extend their keys by 21
    // more digits from the common level-21 cell and sort the run by them.
    const uint32_t a = i;
    uint32_t b = i + 1;
    while (b + 1 < n && skey[b + 1] == k0) ++b;
    atomicAdd(&h->deep_runs, 1u);
    Cell c0 = root;
    {
        const uint32_t q = sidx[a];
        key_from(c0, x[q], y[q], z[q]);  // walk to the shared level-21 cell
    }
    for (uint32_t p = a; p <= b; ++p) {
        Cell c = c0;
        const uint32_t q = sidx[p];
        klo[p] = key_from(c, x[q], y[q], z[q]);
    }
    // insertion sort by the second key word; stable, so equal keys keep body order
    for (uint32_t p = a + 1; p <= b; ++p) {
        const uint64_t kv = klo[p];
        const uint32_t iv = sidx[p];
        uint32_t q = p;
        while (q > a && klo[q - 1] > kv) {
            klo[q] = klo[q - 1];
            sidx[q] = sidx[q - 1];
            --q;
        }
        klo[q] = kv;
        sidx[q] = iv;
    }
    for (uint32_t p = a; p < b; ++p) {
        const uint64_t d = klo[p] ^ klo[p + 1];
        if (d == 0) {
            raise_flag(h, kFlagDepth);  // not separated within kMaxDepth digits
            lcp[p] = kMaxDepth - 1;
        } else {
            lcp[p] = kKeyLevels + lcp_depth(klo[p], klo[p + 1]);
        }
    }
}

// chain[i] = number of internal cells owned by pair i = max(0, lcp[i] - lcp[i-1])
__device__ inline void chain_at(uint32_t i, const int32_t *__restrict__ lcp, uint32_t *chain) {
    const int cp = i > 0 ? lcp[i - 1] : -1;
    const int cn = lcp[i];
    chain[i] = cn > cp ? (uint32_t)(cn - cp) : 0u;
}

// lcp of every pair, and the chain lengths of each scan tile's pairs added into
// part[tile] (zeroed before).  A pair's chain needs the lcp of the pair before
// it: from the keys, or at least kKeyLevels if these are equal, which leaves a
// chain of 0.  The chains inside a run of equal keys are added by the thread
// that sorts the run.
__global__ void __launch_bounds__(kThreads) k_lcp(const double *__restrict__ x,
                                                  const double *__restrict__ y,
                                                  const double *__restrict__ z, uint32_t n,
                                                  TreeHdr *h, uint64_t *skey, uint32_t *sidx,
                                                  uint64_t *klo, int32_t *lcp, uint32_t *part) {
    static_assert(kScanTile % kThreads == 0, "a workgroup's pairs lie in one tile");
    __shared__ uint32_t ws[kThreads / 64];
    const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
    uint32_t own = 0;
    if (i + 1 < n) {
        const Cell root{h->minx, h->miny, h->minz, h->edge};
        lcp_at(i, x, y, z, n, root, h, skey, sidx, klo, lcp);
        const uint64_t k0 = skey[i], k1 = skey[i + 1];
        const uint64_t kp = i > 0 ? skey[i - 1] : 0;
        const int cp = i == 0 ? -1 : kp == k0 ? kKeyLevels : lcp_depth(kp, k0);
        if (k0 != k1) {
            const int cn = lcp_depth(k0, k1);
            own = cn > cp ? (uint32_t)(cn - cp) : 0u;
        } else if (i == 0 || kp != k0) {  // a run's first pair: the chains of the run
            int before = cp;
            for (uint32_t p = i; p + 1 < n && skey[p + 1] == k0; ++p) {
                const int d = lcp[p];
                if (d > before) atomicAdd(&part[p / kScanTile], (uint32_t)(d - before));
                before = d;
            }
        }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) own += __shfl_xor(own, off, 64);
    if ((threadIdx.x & 63u) == 0) ws[threadIdx.x >> 6] = own;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t sum = 0;
        for (int w = 0; w < kThreads / 64; ++w) sum += ws[w];
        if (sum) atomicAdd(&part[i / kScanTile], sum);
    }
}

// Numbers the internal cells: off[i] = the chain lengths of the pairs before i
// (tile sums in `part`), h->internal_count their total; and empties what the
// topology pass fills in: the child slots of the tile's own cells, and the
// table of block-crossing cells.
__global__ void __launch_bounds__(kScanThreads) k_number(const int32_t *__restrict__ lcp,
                                                         uint32_t pairs, uint32_t *off,
                                                         const uint32_t *__restrict__ part,
                                                         uint32_t nparts, bool scanned, TreeHdr *h,
                                                         uint32_t icap, int32_t *ref,
                                                         uint32_t *spanning, uint32_t spanning_cap) {
    __shared__ uint32_t sh[2 * kScanThreads / 64];
    const uint32_t t = threadIdx.x;
    const uint64_t stride = (uint64_t)gridDim.x * kScanThreads;
    for (uint64_t j = (uint64_t)blockIdx.x * kScanThreads + t; j < spanning_cap; j += stride)
        spanning[j] = kNoCell;
    const uint64_t i0 = (uint64_t)blockIdx.x * kScanTile + (uint64_t)t * kScanItems;
    uint32_t v[kScanItems], sum = 0;
    int before = i0 > 0 && i0 <= pairs ? lcp[i0 - 1] : -1;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const int d = i0 + k < pairs ? lcp[i0 + k] : -1;
        v[k] = d > before ? (uint32_t)(d - before) : 0u;
        sum += v[k];
        before = d;
    }
    const ScanPlace pl = scan_place(sum, part, nparts, scanned, sh);
    uint32_t o = pl.first + pl.before;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        if (i0 + k < pairs) off[i0 + k] = o;
        o += v[k];
    }
    if (blockIdx.x + 1 == gridDim.x && t == 0) h->internal_count = pl.first + pl.total;
    const uint64_t ob = 1ull + 8ull * min(pl.first, icap);
    const uint64_t oe = 1ull + 8ull * min(pl.first + pl.total, icap);
    for (uint64_t j = ob + t; j < oe; j += kScanThreads) ref[j] = kRefEmpty;
}

// h->max_depth = depth of the deepest leaf = 1 + the deepest cell that two
// sorted neighbours share (max lcp), for n >= 2; 0 for one body.  Run on
// demand (tree queries, cell moments), not in every build: a grid-stride
// maximum per workgroup, and the device-scope RMW only when it raises the
// stored value.
constexpr int kDepthBlocks = 256;
__global__ void __launch_bounds__(kThreads) k_max_depth(const int32_t *__restrict__ lcp, uint32_t n,
                                                        TreeHdr *h) {
    __shared__ int wmax[kThreads / 64];
    int v = -1;
    for (uint32_t i = blockIdx.x * kThreads + threadIdx.x; i + 1 < n; i += gridDim.x * kThreads)
        v = max(v, lcp[i]);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v = max(v, __shfl_xor(v, off, 64));
    if ((threadIdx.x & 63u) == 0) wmax[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        int b = wmax[0];
        for (int w = 1; w < kThreads / 64; ++w) b = max(b, wmax[w]);
        const uint32_t d = (uint32_t)(b + 1);
        if (b >= 0 &&
            d > __hip_atomic_load(&h->max_depth, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            atomicMax(&h->max_depth, d);
    }
}

// ---- 6. topology --------------------------------------------------------------
// The sorted keys, pairs' lcp and cell numbers as the topology pass reads them.
// A window [w0, w1) of each sits in LDS: the searches of one block stay mostly
// inside it, and the memory latencies of keys, lcp and numbers overlap.
struct KeyView {
    const uint64_t *skey;
    const uint64_t *klo;
    const int32_t *lcp;
    const uint32_t *off;
    const uint64_t *win;
    const int32_t *wlcp;
    const uint32_t *woff;
    uint32_t w0, w1;
    __device__ inline int lcp_of(uint32_t p) const {
        return p - w0 < w1 - w0 ? wlcp[p - w0] : lcp[p];
    }
    __device__ inline uint32_t off_of(uint32_t p) const {
        return p - w0 < w1 - w0 ? woff[p - w0] : off[p];
    }
    __device__ inline uint64_t key(uint32_t p) const {
        return p - w0 < w1 - w0 ? win[p - w0] : skey[p];
    }
    __device__ inline uint32_t digit(uint32_t p, int l) const {
        return l < kKeyLevels ? (uint32_t)(key(p) >> (3 * (kKeyLevels - 1 - l))) & 7u
                              : (uint32_t)(klo[p] >> (3 * (2 * kKeyLevels - 1 - l))) & 7u;
    }
    // do sorted bodies p and q share their first v digits?
    __device__ inline bool same(uint32_t p, uint32_t q, int v) const {
        if (v <= 0) return true;
        const uint64_t kp = key(p), kq = key(q);
        if (v <= kKeyLevels) return ((kp ^ kq) >> (63 - 3 * v)) == 0;
        return kp == kq && ((klo[p] ^ klo[q]) >> (63 - 3 * (v - kKeyLevels))) == 0;
    }
    // does the key kn of sorted body p share its first v digits with body q's?
    __device__ inline bool same_key(uint64_t kn, uint32_t p, uint32_t q, int v) const {
        if (v <= 0) return true;
        const uint64_t kq = key(q);
        if (v <= kKeyLevels) return ((kn ^ kq) >> (63 - 3 * v)) == 0;
        return kn == kq && ((klo[p] ^ klo[q]) >> (63 - 3 * (v - kKeyLevels))) == 0;
    }
    // first sorted position of the depth-v cell that holds sorted body i
    __device__ inline uint32_t cell_start(uint32_t i, int v) const {
        if (v <= 0 || i == 0) return 0;
        int64_t in = i;       // shares the prefix
        int64_t out = -1;     // does not (or -1)
        uint32_t step = 1;
        while (true) {
            const int64_t q = (int64_t)i - step;
            if (q < 0) break;
            if (!same((uint32_t)q, i, v)) {
                out = q;
                break;
            }
            in = q;
            step <<= 1;
        }
        while (in - out > 1) {
            const int64_t mid = out + (in - out) / 2;
            if (same((uint32_t)mid, i, v)) in = mid; else out = mid;
        }
        return (uint32_t)in;
    }
};

// Internal cells owned by pair i and the leaf of sorted body i.  A cell is
// "local" (int_local 1) when its bodies stay inside one com_block-body block
// of the sorted order; the others go to the table
// spanning[block * kMaxDepth + depth], with int_local 2 (and kSpanCross set in
// the table) if they also cross a boundary of the com_super-body super-blocks
// and 0 if not.
// No atomics: every cell, node slot and table entry has exactly one writer.
__device__ inline void link_at(uint32_t i, uint32_t n, uint32_t icap, TreeHdr *h, KeyView kv,
                               const uint32_t *__restrict__ sidx, int32_t *ref, uint8_t *int_depth,
                               uint32_t *int_node, uint32_t *body_node,
                               uint8_t *int_local, uint32_t *spanning, uint32_t spanning_cap,
                               uint32_t *int_first, uint32_t com_block, uint32_t com_super) {
    if (n == 1) {  // the root is a leaf holding the only body (max_depth stays 0)
        ref[0] = ref_of_body(sidx[0]);
        body_node[0] = 0;
        return;
    }
    // the next block's and super-block's first keys, read before they are needed
    const uint32_t next_block = (i / com_block + 1) * com_block;
    const uint32_t next_super = (i / com_super + 1) * com_super;
    const uint64_t key_block = kv.skey[min(next_block, n - 1)];
    const uint64_t key_super = kv.skey[min(next_super, n - 1)];
    const uint32_t body = sidx[i];
    const int cp = i > 0 ? kv.lcp_of(i - 1) : -1;
    const int cn = i + 1 < n ? kv.lcp_of(i) : -1;
    // One search serves every body: the depth-cp cell that holds it holds the top
    // of pair i's chain, or, without a chain, the body's leaf.
    uint32_t up = 0;  // that cell's number
    if (cp >= 0) {
        const uint32_t a = kv.cell_start(i, cp);
        const int ca = a > 0 ? kv.lcp_of(a - 1) : -1;
        up = kv.off_of(a) + (uint32_t)(cp - ca - 1);
    }
    const uint32_t own = cn > cp ? kv.off_of(i) : 0u;  // the chain's first cell
    // internal cells owned by pair i: depths cp+1 .. cn
    for (int l = cp + 1; l <= cn; ++l) {
        const uint32_t k = own + (uint32_t)(l - cp - 1);
        if (k >= icap) {
            raise_flag(h, kFlagNodeOverflow);
            break;
        }
        int_depth[k] = (uint8_t)l;
        int_first[k] = i;
        // The cell's bodies start at i; it crosses into the next COM block iff
        // that block's first body shares its l-digit prefix with body i.
        const bool local = !(next_block < n && kv.same_key(key_block, next_block, i, l));
        if (local) {
            int_local[k] = 1;
        } else {
            // the same test at the next super-block boundary
            const bool cross = next_super < n && kv.same_key(key_super, next_super, i, l);
            int_local[k] = cross ? 2 : 0;
            // the block of body i owns at most one crossing cell per depth:
            // the depth-l cell holding the block's last and the next block's
            // first body
            const uint64_t slot = (uint64_t)(i / com_block) * kMaxDepth + (uint32_t)l;
            if (slot < spanning_cap) spanning[slot] = cross ? k | kSpanCross : k;
            else raise_flag(h, kFlagNodeOverflow);
        }
        if (l == 0) {
            int_node[k] = 0;
            ref[0] = (int32_t)k;
            continue;
        }
        const uint32_t pk = l > cp + 1 ? k - 1 : up;
        if (pk >= icap) {
            raise_flag(h, kFlagNodeOverflow);
            break;
        }
        const uint32_t node = 1u + 8u * pk + kv.digit(i, l - 1);
        int_node[k] = node;
        ref[node] = (int32_t)k;
    }
    // the body's leaf: one level below the deepest cell it shares with a neighbour
    const int D = cp > cn ? cp : cn;
    const uint32_t pk = cn > cp ? own + (uint32_t)(cn - cp - 1) : up;
    if (pk >= icap) {
        raise_flag(h, kFlagNodeOverflow);
        body_node[i] = 0xffffffffu;
        return;
    }
    const uint32_t leaf = 1u + 8u * pk + kv.digit(i, D);
    ref[leaf] = ref_of_body(body);
    body_node[i] = leaf;
    // the deepest leaf, 1 + max lcp, is taken from the lcp array (max_depth_of)
}

constexpr uint32_t kLinkBack = 768;  // entries before a link block's own kept in LDS
// Loads the window of the block at b0: its kThreads entries and kLinkBack before
// them, all loads in flight together.  kv's arrays and window are absolute here.
// (The last pair's lcp and number, and those of one body, are never written:
// what is loaded for them is not used.)
__device__ __forceinline__ void link_window(KeyView &kv, uint32_t b0, uint32_t n) {
    constexpr int rounds = (kLinkBack + kThreads) / kThreads;
    static_assert(kLinkBack % kThreads == 0, "whole rounds");
    __shared__ uint64_t win[kLinkBack + kThreads];
    __shared__ int32_t wlcp[kLinkBack + kThreads];
    __shared__ uint32_t woff[kLinkBack + kThreads];
    const uint32_t w0 = b0 > kLinkBack ? b0 - kLinkBack : 0u;
    const uint32_t w1 = min(n, b0 + (uint32_t)kThreads);
    uint64_t k[rounds];
    int32_t l[rounds];
    uint32_t o[rounds];
#pragma unroll
    for (int r = 0; r < rounds; ++r) {
        const uint32_t p = min(w0 + threadIdx.x + (uint32_t)r * kThreads, w1 - 1);
        k[r] = kv.skey[p];
        l[r] = kv.lcp[p];
        o[r] = kv.off[p];
    }
#pragma unroll
    for (int r = 0; r < rounds; ++r) {
        const uint32_t j = threadIdx.x + (uint32_t)r * kThreads;
        win[j] = k[r];
        wlcp[j] = l[r];
        woff[j] = o[r];
    }
    __syncthreads();
    kv.win = win;
    kv.wlcp = wlcp;
    kv.woff = woff;
    kv.w0 = w0;
    kv.w1 = w1;
}

// Latency again: memory round trips and the search.  1024 bodies 10.7 us with two
// searches per body and keys alone in LDS, 7.7 now; 100,003: 18.8 and 12.9;
// 4,194,304: 149 and 117; the ensemble's 96 and 70.
__global__ void __launch_bounds__(kThreads) k_link(uint32_t n, uint32_t icap, TreeHdr *h,
                                                   KeyView kv, const uint32_t *__restrict__ sidx,
                                                   int32_t *ref, uint8_t *int_depth,
                                                   uint32_t *int_node, uint32_t *body_node,
                                                   uint8_t *int_local,
                                                   uint32_t *spanning, uint32_t spanning_cap,
                                                   uint32_t *int_first) {
    const uint32_t b0 = blockIdx.x * kThreads;
    link_window(kv, b0, n);
    const uint32_t i = b0 + threadIdx.x;
    if (i >= n) return;
    link_at(i, n, icap, h, kv, sidx, ref, int_depth, int_node, body_node,
            int_local, spanning, spanning_cap, int_first, kComBlock, kComSuper);
}

// ---- 7. centre of mass --------------------------------------------------------
// Sum of the 8 children of internal cell pk in digit order 0..7 from 0.0
// (BarnesHutOctree.cpp:299-311): a body child adds (x m, y m, z m, m), a cell
// child its sums.  Empty children add +0.0, which changes no running sum that
// starts at +0.0, so they are skipped.  All eight children are loaded first,
// so their loads are in flight together; the additions keep digit order.
__device__ inline void add_children(const int32_t (&r)[8], const double4 (&v)[8],
                                    const uint32_t (&c)[8], InternalSums &out, uint32_t &cnt) {
    double sx = 0, sy = 0, sz = 0, sm = 0;
    cnt = 0;
#pragma unroll
    for (int d = 0; d < 8; ++d) {
        if (r[d] != kRefEmpty) {
            sx += v[d].x;
            sy += v[d].y;
            sz += v[d].z;
            sm += v[d].w;
            cnt += c[d];
        }
    }
    out = InternalSums{sx, sy, sz, sm};
}

// the term of a body child: (x m, y m, z m, m)
__device__ inline double4 body_term(const double4 p) {
    return make_double4(p.x * p.w, p.y * p.w, p.z * p.w, p.w);
}

// Traversal records and groups, written by the centre-of-mass kernels: a cell,
// once summed, writes the records of its 8 child slots (their data is at
// hand) and, if it holds more than rule.group_max bodies, marks the traversal
// groups among its children (a child cell with at most rule.group_max
// bodies, or a body).  The kernel that sums the root writes the root's
// record, and its group if the root holds at most rule.group_max bodies.
struct RecOut {
    double G;
    int f64, f32;  // FP64 records (cm); FP32 records and traversal groups
    double4 *cm;
    NodeF32 *rec;
    uint32_t *group_size;
    uint32_t *group_slot;  // 1 where a group starts, for a later scan; null: not kept
    GroupRule rule;  // group size and packing limit
};

// Record centre of a child from its term: a cell's sums, or a body's
// (x m, y m, z m, m).  The reference divides numerator by mass at every visit
// (BarnesHutAlgorithm.cpp:351-353); the quotient is the same.
__device__ inline double4 term_com(const double4 v) {
    return make_double4(v.x / v.w, v.y / v.w, v.z / v.w, v.w);
}

__device__ inline void put_record(const RecOut &o, uint64_t j, int32_t r, const double4 c) {
    if (o.f64) o.cm[j] = c;
    if (o.f32) {
        NodeF32 q;
        q.x = (float)c.x;
        q.y = (float)c.y;
        q.z = (float)c.z;
        q.gm = (float)(o.G * c.w);
        q.ref = r;
        q.lx = (float)(c.x - (double)q.x);
        q.ly = (float)(c.y - (double)q.y);
        q.lz = (float)(c.z - (double)q.z);
        o.rec[j] = q;
    }
}

// a traversal group of `size` bodies starts at sorted position p
__device__ inline void put_group(const RecOut &o, uint32_t p, uint32_t size) {
    if (o.f32) {
        o.group_size[p] = size;
        if (o.group_slot) o.group_slot[p] = 1u;
    }
}

// Traversal groups among the children of a cell that holds more than
// group_max bodies; first: the cell's first sorted position, m[d]: child d's
// body count (0 if empty).  Each child with at most group_max bodies is a
// group; in a cell of at most pack_max bodies, runs of such children are
// packed in digit order into groups of at most group_max bodies instead
// (siblings are consecutive in the sorted order; a child with more bodies
// ends a run).
__device__ inline void put_child_groups(const RecOut &o, uint32_t first, const uint32_t (&m)[8]) {
    const uint32_t gmax = o.rule.group_max;
    uint32_t total = 0;
#pragma unroll
    for (int d = 0; d < 8; ++d) total += m[d];
    const bool pack = total <= o.rule.pack_max;
    uint32_t pos = first, g0 = first, gs = 0;
#pragma unroll
    for (int d = 0; d < 8; ++d) {
        if (m[d] == 0) continue;
        if (gs && (!pack || m[d] > gmax || gs + m[d] > gmax)) {
            put_group(o, g0, gs);
            gs = 0;
        }
        if (m[d] <= gmax) {
            if (gs == 0) g0 = pos;
            gs += m[d];
        }
        pos += m[d];
    }
    if (gs) put_group(o, g0, gs);
}

// Records and groups of the children of cell pk (depth `depth`, first sorted
// position `first`), given their refs, terms and body counts; the root's own
// record and group when pk is the root.
__device__ inline void cell_outputs(const RecOut &o, uint32_t pk, uint32_t depth, uint32_t first,
                                    const int32_t (&r)[8], const double4 (&v)[8], const uint32_t (&c)[8],
                                    const double4 s, uint32_t cnt) {
    const uint64_t base = 1ull + 8ull * pk;
#pragma unroll
    for (int d = 0; d < 8; ++d) {
        if (r[d] == kRefEmpty)
            put_record(o, base + d, kRefEmpty, make_double4(0.0, 0.0, 0.0, 0.0));
        else
            put_record(o, base + d, r[d], term_com(v[d]));
    }
    if (cnt > o.rule.group_max) put_child_groups(o, first, c);
    if (depth == 0) {
        put_record(o, 0, (int32_t)pk, term_com(s));
        if (cnt <= o.rule.group_max) put_group(o, first, cnt);
    }
}

// The global-memory path: the cell's 8 children summed in digit order from 0.0,
// then the children's records and groups.
__device__ inline void sum_children_out(uint32_t pk, uint32_t depth, uint32_t first,
                                        const double4 *__restrict__ body4,
                                        const int32_t *__restrict__ ref, InternalSums *sums,
                                        uint32_t *counts, TreeHdr *h, const RecOut &o) {
    const uint64_t base = 1ull + 8ull * pk;
    int32_t r[8];
    double4 v[8];
    uint32_t c[8];
#pragma unroll
    for (int d = 0; d < 8; ++d) r[d] = ref[base + d];
#pragma unroll
    for (int d = 0; d < 8; ++d) {
        v[d] = make_double4(0.0, 0.0, 0.0, 0.0);
        c[d] = 0;
        if (r[d] >= 0) {
            const InternalSums q = sums[r[d]];
            v[d] = make_double4(q.x, q.y, q.z, q.m);
            c[d] = counts[r[d]];
        } else if (r[d] != kRefEmpty) {
            v[d] = body_term(body4[body_of_ref(r[d])]);
            c[d] = 1;
        }
    }
    InternalSums q;
    uint32_t cnt;
    add_children(r, v, c, q, cnt);
    sums[pk] = q;
    counts[pk] = cnt;
    if (q.m == 0) raise_flag(h, kFlagZeroMass);
    cell_outputs(o, pk, depth, first, r, v, c, make_double4(q.x, q.y, q.z, q.m), cnt);
}

// Centre of mass, level by level from the deepest cells up: a cell's sums
// (its children in digit order) need only deeper cells, so every cell of one
// depth can be summed at once, with a barrier between depths.
constexpr int kComThreads = 1024;

// Counts per depth, cnt[0, kMaxDepth), to first places (cnt, and a copy in cur;
// cnt[kMaxDepth] the total), by the first wave; bit d of *levels: depth d has
// cells.
static_assert(kMaxDepth < 64, "one lane per depth and the total");
__device__ inline void depth_starts(uint32_t *cnt, uint32_t *cur, unsigned long long *levels) {
    const uint32_t t = threadIdx.x;
    if (t >= 64) return;
    const uint32_t c = t < (uint32_t)kMaxDepth ? cnt[t] : 0u;
    uint32_t inc = c;
#pragma unroll
    for (int w = 1; w < 64; w <<= 1) {
        const uint32_t v = __shfl_up(inc, w, 64);
        if (t >= (uint32_t)w) inc += v;
    }
    if (t <= (uint32_t)kMaxDepth) cnt[t] = inc - c;
    if (t < (uint32_t)kMaxDepth) cur[t] = inc - c;
    const unsigned long long lv = __ballot(c != 0);
    if (t == 0) *levels = lv;
}

__device__ __forceinline__ unsigned long long uniform64(unsigned long long v) {
    return (unsigned long long)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v) |
           (unsigned long long)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32)) << 32;
}

// Cells [kb, ke) bucketed by depth into lvl[kb ..) (cells with keep(k) only),
// then sum(k) for each, deepest depth first.  cnt/cur: kMaxDepth + 1 and
// kMaxDepth LDS words.  Every thread of the workgroup calls it.
template <typename Keep, typename Sum>
__device__ inline void com_levels(uint32_t kb, uint32_t ke, Keep keep,
                                  const uint8_t *__restrict__ int_depth, uint32_t *lvl,
                                  uint32_t *cnt, uint32_t *cur, Sum sum) {
    __shared__ unsigned long long levels;
    const uint32_t t = threadIdx.x, nt = blockDim.x;
    for (uint32_t d = t; d <= (uint32_t)kMaxDepth; d += nt) cnt[d] = 0;
    __syncthreads();
    for (uint32_t k = kb + t; k < ke; k += nt)
        if (keep(k)) atomicAdd(&cnt[min((uint32_t)int_depth[k], (uint32_t)kMaxDepth - 1)], 1u);
    __syncthreads();
    depth_starts(cnt, cur, &levels);
    __syncthreads();
    for (uint32_t k = kb + t; k < ke; k += nt)
        if (keep(k))
            lvl[kb + atomicAdd(&cur[min((uint32_t)int_depth[k], (uint32_t)kMaxDepth - 1)], 1u)] = k;
    __syncthreads();
    for (unsigned long long lv = uniform64(levels); lv;) {
        const int d = 63 - __clzll((long long)lv);
        lv ^= 1ull << d;
        const uint32_t lb = cnt[d], le = cnt[d + 1];
        for (uint32_t j = lb + t; j < le; j += nt) sum(lvl[kb + j]);
        __syncthreads();
    }
}

// The levels in LDS, deepest first: cell c of order[cnt[d], cnt[d + 1]) gets
// term[kCell + c] = the sum of its eight children's terms, in digit order from
// 0.0 as sum_children_out, and m[kCell + c] = their bodies; at[8 c + digit] is
// the place of a child's term, which for an empty slot holds zeros.  Four lanes
// share a cell, one per component.  kThreads_ threads take part: a whole
// workgroup with a barrier between levels, or one wave, which needs none (its
// LDS accesses complete in order).  The chain from level to level is one read,
// the eight additions and one write: the next step's cell and places are read
// ahead of it, and the level bounds sit in the lanes of a register.
template <uint32_t kThreads_, uint32_t kCell>
__device__ __forceinline__ void sum_levels(uint32_t t, const uint32_t *cnt,
                                           unsigned long long lv, const uint16_t *order,
                                           const uint16_t *at_s, double4 *term4, uint32_t *m_s) {
    constexpr uint32_t step = kThreads_ / 4;
    const uint32_t comp = t & 3u;
    double *term = table_as<double>(term4) + comp;  // place p at term[4 p]
    const int starts = (int)cnt[min(t & 63u, (uint32_t)kMaxDepth)];
    uint32_t base = 0, end = 0;  // the next step's cells [base, min(base + step, end)): uniform
    bool fresh = false;          // the next step opens a level
    uint32_t nc = 0;
    uint4 nw = make_uint4(0, 0, 0, 0);
    bool has = false;
    auto next = [&]() {
        base += step;
        fresh = base >= end;
        if (fresh) {
            if (!lv) {
                end = 0;
                has = false;
                return;
            }
            const int d = 63 - __clzll((long long)lv);
            lv ^= 1ull << d;
            base = (uint32_t)__builtin_amdgcn_readlane(starts, d);
            end = (uint32_t)__builtin_amdgcn_readlane(starts, d + 1);
        }
        const uint32_t j = base + (t >> 2);
        has = j < end;
        if (has) {
            nc = order[j];
            nw = *reinterpret_cast<const uint4 *>(at_s + 8 * nc);
        }
    };
    next();
    while (end) {
        const uint32_t c = nc;
        const uint4 w = nw;
        const bool mine = has;
        next();
        if (mine) {
            const uint32_t at[8] = {w.x & 0xffffu, w.x >> 16, w.y & 0xffffu, w.y >> 16,
                                    w.z & 0xffffu, w.z >> 16, w.w & 0xffffu, w.w >> 16};
            double v[8];
            uint32_t m[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = term[4 * at[k]];
#pragma unroll
            for (int k = 0; k < 8; ++k) m[k] = m_s[at[k]];
            double sum = 0;
            uint32_t count = 0;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                sum += v[k];
                count += m[k];
            }
            term[4 * (kCell + c)] = sum;
            m_s[kCell + c] = count;  // the same from all four lanes
        }
        if (kThreads_ == 64)
            wave_lds_sync();
        else if (fresh)
            __syncthreads();
    }
}

// Pass 1: one workgroup per kComBlock consecutive (sorted) bodies sums the
// cells that lie inside its block.  Pair i owns cells [off[i], off[i+1]), so
// the block's cells are one contiguous range [kb, ke).  Up to kComLdsCells
// cells are summed entirely in LDS.  Staged once, two round trips to memory
// deep: the terms of the block's bodies and their input indices in sorted
// order; per child slot the place of the child's term, which bodies and cells
// write into the slot the topology pass gave them; and the cells bucketed by
// depth.  The levels touch LDS only (a barrier also waits for global stores).
// Then every body and every cell is divided once into its record centre, and a
// last pass writes the node records of the cells' child slots, consecutive
// threads on consecutive slots.  A larger block falls back to the same work in
// global memory.  The block also clears the group marks of its positions
// before any is set.
//
// What bounds it is the chain of levels (6 to 10 of them), each a barrier and
// three LDS round trips, not bytes.  So a level touches only its own cells;
// four lanes share a cell, one per component, and read all eight children
// together: body terms, cell sums and a zero for empty slots share one LDS
// table, so no child needs a branch.  An empty slot adds +0.0, which changes no
// running sum that starts at +0.0.
// (1024 bodies: 40 us with one lane per cell and a scan of all cells per level,
// 13.5 now; 100,003: 43 and 17; 1,048,576, disk: 107 and 58; 4,194,304: 366 and 243.)
constexpr uint32_t kComLdsCells = 576;   // about 490 per block; 537 the most seen (disk, Plummer)
constexpr int kComLocalThreads = 512;
constexpr int kComBodiesPerThread = kComBlock / kComLocalThreads;
constexpr int kComCellsPerThread = (kComLdsCells + kComLocalThreads - 1) / kComLocalThreads;
static_assert(kComBlock % kComLocalThreads == 0, "whole staging rounds");
// The LDS table of terms: the block's bodies, its cells, one zero.
constexpr uint32_t kTermCell = kComBlock, kTermZero = kTermCell + kComLdsCells;
static_assert(kTermZero < 0xffffu, "16-bit places");
// Block blk of one octree (the one-system kernel below, and the ensemble's,
// which runs the blocks of every system in one launch).
__device__ __forceinline__ void com_local_block(
    uint32_t blk, uint32_t n, uint32_t icap, TreeHdr *h, const double4 *__restrict__ body4,
    const uint32_t *__restrict__ sidx, const uint32_t *__restrict__ body_node,
    const int32_t *__restrict__ ref, const uint32_t *__restrict__ off,
    const uint8_t *__restrict__ int_depth, const uint8_t *__restrict__ int_local,
    const uint32_t *__restrict__ int_first, const uint32_t *__restrict__ int_node, uint32_t *lvl,
    InternalSums *sums, uint32_t *counts, const RecOut &o) {
    constexpr uint32_t nt = kComLocalThreads;
    __shared__ uint32_t cnt[kMaxDepth + 1], cur[kMaxDepth];
    __shared__ unsigned long long levels;        // bit d: a local cell of depth d
    __shared__ double4 term_s[kTermZero + 1];    // {x m, y m, z m, m}: bodies, cells, zero
    __shared__ uint32_t m_s[kTermZero + 1];      // bodies of a term: 1, a cell's count, 0
    __shared__ uint32_t i_s[kComBlock];          // input index of a body
    __shared__ alignas(16) uint16_t at_s[8 * kComLdsCells];  // child slot: place of its term
    __shared__ uint16_t order_s[kComLdsCells];  // local cells bucketed by depth
    __shared__ uint8_t depth_s[kComLdsCells];   // depth; kMaxDepth if not local
    const uint32_t t = threadIdx.x;
    const uint32_t s = blk * kComBlock;
    const uint32_t e = min(n, s + kComBlock);
    if (n < 2) {  // a lone body is the root leaf: no internal cell
        if (t == 0) {
            const uint32_t q = sidx[0];
            const double4 b = body4[q];
            if (b.w == 0) raise_flag(h, kFlagZeroMass);
            if (o.f32) {
                o.group_size[0] = 0;
                if (o.group_slot) o.group_slot[0] = 0;
            }
            put_record(o, 0, ref_of_body(q), term_com(body_term(b)));
            put_group(o, 0, 1);
        }
        return;
    }
    // first loads: body indices and leaf nodes, the cell range
    uint32_t bi[kComBodiesPerThread], bn[kComBodiesPerThread];
#pragma unroll
    for (int q = 0; q < kComBodiesPerThread; ++q) {
        const uint32_t i = s + t + q * nt;
        bi[q] = i < e ? sidx[i] : 0u;
        bn[q] = i < e ? body_node[i] : 0u;
    }
    const uint32_t I = min(h->internal_count, icap);
    const uint32_t kb = s < n - 1 ? min(off[s], I) : I;
    const uint32_t nc = (e < n - 1 ? min(off[e], I) : I) - kb;
    const bool fits = nc <= kComLdsCells;  // the same for the whole workgroup
    // the cells' data and the bodies
    uint32_t cf[kComCellsPerThread], cd[kComCellsPerThread], cn_[kComCellsPerThread];
    double4 b[kComBodiesPerThread];
#pragma unroll
    for (int q = 0; q < kComBodiesPerThread; ++q)
        if (s + t + q * nt < e) b[q] = body4[bi[q]];
#pragma unroll
    for (int q = 0; q < kComCellsPerThread; ++q) {
        const uint32_t c = t + q * nt;
        cd[q] = (uint32_t)kMaxDepth;
        if (!fits || c >= nc) continue;
        cf[q] = int_first[kb + c];
        cn_[q] = int_node[kb + c];
        const uint32_t d = min((uint32_t)int_depth[kb + c], (uint32_t)kMaxDepth - 1);
        cd[q] = int_local[kb + c] == 1 ? d : (uint32_t)kMaxDepth;
    }
    if (t <= (uint32_t)kMaxDepth) cnt[t] = 0;
    if (t < 4) table_as<double>(&term_s[kTermZero])[t] = 0.0;
    if (t == 4) m_s[kTermZero] = 0;
    if (fits) {
        constexpr uint32_t z2 = kTermZero | kTermZero << 16;
        for (uint32_t c = t; c < nc; c += nt)
            *reinterpret_cast<uint4 *>(&at_s[8 * c]) = make_uint4(z2, z2, z2, z2);
    }
    __syncthreads();
    // bodies and cells into the slots of their parents (slots of other blocks'
    // cells are left out; a cell that is not local is written and not used)
    const uint64_t slot0 = 1ull + 8ull * kb;
#pragma unroll
    for (int q = 0; q < kComBodiesPerThread; ++q) {
        const uint32_t p = t + q * nt;
        if (s + p >= e) continue;
        if (b[q].w == 0) raise_flag(h, kFlagZeroMass);
        term_s[p] = body_term(b[q]);
        m_s[p] = 1;
        i_s[p] = bi[q];
        const uint64_t j = (uint64_t)bn[q] - slot0;
        if (fits && j < 8ull * nc) at_s[j] = (uint16_t)p;
        if (o.f32) {
            o.group_size[s + p] = 0;
            if (o.group_slot) o.group_slot[s + p] = 0;
        }
    }
    if (!fits) {
        __syncthreads();
        com_levels(kb, kb + nc, [&](uint32_t k) { return int_local[k] == 1; }, int_depth, lvl, cnt,
                   cur, [&](uint32_t k) {
                       sum_children_out(k, int_depth[k], int_first[k], body4, ref,
                                        sums, counts, h, o);
                   });
        return;
    }
    uint32_t place[kComCellsPerThread];  // among the cells of its depth
#pragma unroll
    for (int q = 0; q < kComCellsPerThread; ++q) {
        const uint32_t c = t + q * nt;
        const bool has = c < nc;
        if (has) {
            const uint64_t j = (uint64_t)cn_[q] - slot0;
            if (j < 8ull * nc) at_s[j] = (uint16_t)(kTermCell + c);
            depth_s[c] = (uint8_t)cd[q];
        }
        // one LDS atomic per wave and depth: the lanes of one depth by ballots
        uint64_t peers = __ballot(has && cd[q] < (uint32_t)kMaxDepth);
#pragma unroll
        for (int w = 0; w < 6; ++w) {
            const bool bit = (cd[q] >> w) & 1u;
            const uint64_t bal = __ballot(bit);
            peers &= bit ? bal : ~bal;
        }
        const uint32_t lane = t & 63u;
        const uint32_t rank = (uint32_t)__popcll(peers & ((1ull << lane) - 1));
        uint32_t base = 0;
        if (((peers >> lane) & 1ull) && rank == 0)
            base = atomicAdd(&cnt[cd[q]], (uint32_t)__popcll(peers));
        place[q] = (uint32_t)__shfl((int)base, peers ? __ffsll((unsigned long long)peers) - 1 : 0, 64) + rank;
    }
    __syncthreads();
    depth_starts(cnt, cur, &levels);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kComCellsPerThread; ++q)
        if (cd[q] < (uint32_t)kMaxDepth) order_s[cnt[cd[q]] + place[q]] = (uint16_t)(t + q * nt);
    __syncthreads();
    sum_levels<kComLocalThreads, kTermCell>(t, cnt, uniform64(levels), order_s, at_s, term_s, m_s);
    // sums and group marks of the local cells; then bodies and cells to their
    // record centres, in place
#pragma unroll
    for (int q = 0; q < kComCellsPerThread; ++q) {
        const uint32_t c = t + q * nt;
        if (cd[q] >= (uint32_t)kMaxDepth) continue;
        const double4 g = term_s[kTermCell + c];
        const uint32_t count = m_s[kTermCell + c];
        if (g.w == 0) raise_flag(h, kFlagZeroMass);
        sums[kb + c] = InternalSums{g.x, g.y, g.z, g.w};
        counts[kb + c] = count;
        const double4 com = term_com(g);
        if (count > o.rule.group_max) {
            uint32_t m[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) m[k] = m_s[at_s[8 * c + k]];
            put_child_groups(o, cf[q], m);
        }
        if (cd[q] == 0) {  // the root (the block holds every body)
            put_record(o, 0, (int32_t)(kb + c), com);
            if (count <= o.rule.group_max) put_group(o, cf[q], count);
        }
        term_s[kTermCell + c] = com;
    }
#pragma unroll
    for (int q = 0; q < kComBodiesPerThread; ++q) {
        double4 *v = &term_s[t + q * nt];
        if (s + t + q * nt < e) *v = term_com(*v);
    }
    __syncthreads();
    // three slots per thread at a time, so that their LDS round trips overlap
    constexpr int kAhead = 3;
    for (uint32_t j0 = t; j0 < 8 * nc; j0 += kAhead * nt) {
        uint32_t at[kAhead], bi2[kAhead];
        double4 v[kAhead];
        bool live[kAhead];
#pragma unroll
        for (int q = 0; q < kAhead; ++q) {
            const uint32_t j = min(j0 + q * nt, 8 * nc - 1);
            live[q] = j0 + q * nt < 8 * nc && depth_s[j >> 3] < kMaxDepth;
            at[q] = at_s[j];
        }
#pragma unroll
        for (int q = 0; q < kAhead; ++q) {
            v[q] = term_s[at[q]];
            bi2[q] = i_s[min(at[q], kComBlock - 1)];
        }
#pragma unroll
        for (int q = 0; q < kAhead; ++q) {
            if (!live[q]) continue;
            const int32_t r = at[q] < kTermCell   ? ref_of_body(bi2[q])
                              : at[q] < kTermZero ? (int32_t)(kb + at[q] - kTermCell)
                                                  : kRefEmpty;
            put_record(o, slot0 + j0 + q * nt, r, v[q]);
        }
    }
}

__global__ void __launch_bounds__(kComLocalThreads) k_com_local(
    uint32_t n, uint32_t icap, TreeHdr *h, const double4 *__restrict__ body4,
    const uint32_t *__restrict__ sidx, const uint32_t *__restrict__ body_node,
    const int32_t *__restrict__ ref, const uint32_t *__restrict__ off,
    const uint8_t *__restrict__ int_depth, const uint8_t *__restrict__ int_local,
    const uint32_t *__restrict__ int_first, const uint32_t *__restrict__ int_node, uint32_t *lvl,
    InternalSums *sums, uint32_t *counts, RecOut o) {
    com_local_block(blockIdx.x, n, icap, h, body4, sidx, body_node, ref, off, int_depth, int_local,
                    int_first, int_node, lvl, sums, counts, o);
}

// Pass 2: the cells crossing block boundaries (the table
// spanning[block * kMaxDepth + depth]), in two launches.  want = 0: one
// workgroup per super-block of kComSuperBlocks blocks sums the cells that
// cross block boundaries inside it and lists those crossing its end (at most
// one per depth) in `cross`; want = 2: one workgroup sums the listed cells,
// which cross super-block boundaries.  A workgroup stages up to kSpanCells cells
// in LDS: the term of every child (a body, or a cell summed by an earlier
// pass) is loaded once, all loads in flight together, and its record is
// written then; a child summed by this workgroup is named by its LDS id
// (cid[k], written first).  The levels, deepest first, then read LDS only.
// More cells fall back to the same sums in global memory.
// One wave runs the levels (sum_levels: few cells a level, no barrier) while
// the others divide and write the records of the children it does not sum.
// (100,003 bodies: 25.6 us a launch with one lane per cell, a branch per child
// and a workgroup barrier per level, 13.8 now.)
constexpr uint32_t kSpanCells = 448;
constexpr uint32_t kSpanRowsAhead = 3;        // table entries per thread in flight
constexpr int kSpanSlots = (8 * (int)kSpanCells + kComThreads - 1) / kComThreads;  // per thread
constexpr uint32_t kSpanSum = 8 * kSpanCells;  // LDS terms: child slots, then sums
static_assert(kSpanCells <= (uint32_t)kComThreads - 64, "a cell per thread");
static_assert(9 * kSpanCells < 0x10000u, "16-bit places");
// Super-block (want 0) or cross list (want 2) sb of one octree.
__device__ __forceinline__ void com_span_block(
    uint32_t sb, uint32_t nblocks, uint32_t rows, uint32_t want, TreeHdr *h,
    const double4 *__restrict__ body4, const int32_t *__restrict__ ref,
    const uint32_t *__restrict__ spanning, const uint8_t *__restrict__ int_local,
    const uint32_t *__restrict__ int_first, const uint32_t *__restrict__ int_node, uint32_t *cid, InternalSums *sums, uint32_t *counts,
    uint32_t *cross, uint32_t cross_cap, const RecOut &o) {
    __shared__ uint32_t ncell, cnt[kMaxDepth + 1], cur[kMaxDepth];
    __shared__ unsigned long long levels;
    __shared__ uint32_t nx, xbase, xl[kMaxDepth];  // want 0: this super-block's crossing cells
    __shared__ uint32_t list[kSpanCells];  // cell index by LDS id
    __shared__ uint8_t ldep[kSpanCells];
    __shared__ uint16_t order[kSpanCells];  // LDS ids bucketed by depth
    __shared__ double4 term[9 * kSpanCells];  // terms of child slots (0 if empty), sums
    __shared__ uint32_t m_s[9 * kSpanCells];    // their bodies
    __shared__ alignas(16) uint16_t at_s[8 * kSpanCells];  // child slot: place of its term
    const uint32_t t = threadIdx.x;
    const uint32_t r0 = sb * rows;
    const uint32_t r1 = min(nblocks, r0 + rows);
    const uint64_t slot0 = (uint64_t)r0 * kMaxDepth, slot1 = (uint64_t)r1 * kMaxDepth;
    if (t == 0) {
        ncell = 0;
        nx = 0;
    }
    for (uint32_t d = t; d <= (uint32_t)kMaxDepth; d += kComThreads) cnt[d] = 0;
    __syncthreads();
    auto take = [&](uint32_t k, uint32_t d) {
        const uint32_t id = atomicAdd(&ncell, 1u);
        if (id < kSpanCells) {
            list[id] = k;
            ldep[id] = (uint8_t)d;
            cid[k] = id;
            atomicAdd(&cnt[d], 1u);
        }
    };
    // want 0 scans this super-block's table rows and keeps its crossing cells
    // (they all hold the super-block's end: at most one per depth); want 2
    // reads the list of those cells
    const uint32_t ncross = want == 2 ? min(h->cross_count, cross_cap) : 0u;
    if (want == 2) {
        for (uint32_t i = t; i < ncross; i += kComThreads) take(cross[i] >> 6, cross[i] & 63u);
    } else {
        for (uint64_t j0 = slot0; j0 < slot1; j0 += (uint64_t)kSpanRowsAhead * kComThreads) {
            uint32_t ks[kSpanRowsAhead];
#pragma unroll
            for (uint32_t q = 0; q < kSpanRowsAhead; ++q) {
                const uint64_t j = j0 + q * kComThreads + t;
                ks[q] = j < slot1 ? spanning[j] : kNoCell;
            }
#pragma unroll
            for (uint32_t q = 0; q < kSpanRowsAhead; ++q) {
                if (ks[q] == kNoCell) continue;
                const uint32_t d = (uint32_t)((j0 + q * kComThreads + t) % kMaxDepth);
                if (ks[q] & kSpanCross) {
                    const uint32_t x = atomicAdd(&nx, 1u);
                    if (x < (uint32_t)kMaxDepth) xl[x] = ((ks[q] & ~kSpanCross) << 6) | d;
                } else {
                    take(ks[q], d);
                }
            }
        }
    }
    __syncthreads();
    if (want != 2) {
        const uint32_t m = min(nx, (uint32_t)kMaxDepth);
        if (t == 0) xbase = m ? atomicAdd(&h->cross_count, m) : 0u;
        __syncthreads();
        if (t < m) {
            if (xbase + t < cross_cap) cross[xbase + t] = xl[t];
            else raise_flag(h, kFlagNodeOverflow);
        }
        if (t == 0 && nx > (uint32_t)kMaxDepth) raise_flag(h, kFlagNodeOverflow);
    }
    const uint32_t nk = ncell;  // the same for every thread
    if (nk > kSpanCells) {
        for (int d = kMaxDepth - 1; d >= 0; --d) {
            if (want == 2) {
                for (uint32_t i = t; i < ncross; i += kComThreads)
                    if ((cross[i] & 63u) == (uint32_t)d) {
                        const uint32_t k = cross[i] >> 6;
                        sum_children_out(k, (uint32_t)d, int_first[k], body4, ref,
                                         sums, counts, h, o);
                    }
            } else {
                for (uint64_t j = slot0 + (uint32_t)d + (uint64_t)t * kMaxDepth; j < slot1;
                     j += (uint64_t)kComThreads * kMaxDepth) {
                    const uint32_t k = spanning[j];
                    if (!(k & kSpanCross))  // neither empty nor crossing
                        sum_children_out(k, (uint32_t)d, int_first[k], body4, ref,
                                         sums, counts, h, o);
                }
            }
            __syncthreads();
        }
        return;
    }
    if (nk == 0) return;
    depth_starts(cnt, cur, &levels);
    __syncthreads();
    uint32_t node = 0, first = 0;  // of cell t
    if (t < nk) {
        order[atomicAdd(&cur[ldep[t]], 1u)] = (uint16_t)t;
        node = int_node[list[t]];
        first = int_first[list[t]];
    }
    // the child slots, all of a thread's loads in flight together.  A cell's
    // sums and count mean something only if an earlier pass summed it, its id
    // only if this workgroup does
    int32_t r[kSpanSlots];
    double4 v[kSpanSlots];
    bool put[kSpanSlots];  // the record is written from here
    uint32_t kind[kSpanSlots], here[kSpanSlots], count[kSpanSlots];
#pragma unroll
    for (int q = 0; q < kSpanSlots; ++q) {
        const uint32_t p = t + q * kComThreads;
        put[q] = p < 8 * nk;
        r[q] = put[q] ? ref[1ull + 8ull * list[p >> 3] + (p & 7u)] : kRefEmpty;
    }
#pragma unroll
    for (int q = 0; q < kSpanSlots; ++q) {
        v[q] = make_double4(0.0, 0.0, 0.0, 0.0);
        kind[q] = ~want;
        here[q] = 0;
        count[q] = 0;
        if (r[q] >= 0) {
            kind[q] = int_local[r[q]];
            here[q] = cid[r[q]];
            count[q] = counts[r[q]];
            v[q] = *table_as<const double4>(&sums[r[q]]);
        } else if (r[q] != kRefEmpty) {
            v[q] = body4[body_of_ref(r[q])];
        }
    }
#pragma unroll
    for (int q = 0; q < kSpanSlots; ++q) {
        const uint32_t p = t + q * kComThreads;
        if (!put[q]) continue;
        uint32_t at = p;
        if (kind[q] == want) {  // summed by this workgroup, one level deeper
            at = kSpanSum + min(here[q], kSpanCells - 1);
            put[q] = false;
        } else {
            if (r[q] < 0 && r[q] != kRefEmpty) {
                v[q] = body_term(v[q]);
                count[q] = 1;
            }
            term[p] = v[q];
            m_s[p] = count[q];
        }
        at_s[p] = (uint16_t)at;
    }
    __syncthreads();
    if (t < 64) sum_levels<64, kSpanSum>(t, cnt, uniform64(levels), order, at_s, term, m_s);
#pragma unroll
    for (int q = 0; q < kSpanSlots; ++q) {
        const uint32_t p = t + q * kComThreads;
        if (put[q])
            put_record(o, 1ull + 8ull * list[p >> 3] + (p & 7u), r[q],
                       r[q] == kRefEmpty ? v[q] : term_com(v[q]));
    }
    __syncthreads();
    // the cells summed here: sums, record (the root's is node 0), group marks
    if (t < nk) {
        const uint32_t k = list[t], bodies = m_s[kSpanSum + t];
        const double4 g = term[kSpanSum + t];
        if (g.w == 0) raise_flag(h, kFlagZeroMass);
        sums[k] = InternalSums{g.x, g.y, g.z, g.w};
        counts[k] = bodies;
        put_record(o, node, (int32_t)k, term_com(g));
        if (bodies > o.rule.group_max) {
            uint32_t m[8];
#pragma unroll
            for (int d = 0; d < 8; ++d) m[d] = m_s[at_s[8 * t + d]];
            put_child_groups(o, first, m);
        } else if (ldep[t] == 0) {
            put_group(o, first, bodies);
        }
    }
}

__global__ void __launch_bounds__(kComThreads) k_com_span(
    uint32_t nblocks, uint32_t rows, uint32_t want, TreeHdr *h, const double4 *__restrict__ body4,
    const int32_t *__restrict__ ref, const uint32_t *__restrict__ spanning,
    const uint8_t *__restrict__ int_local, const uint32_t *__restrict__ int_first,
    const uint32_t *__restrict__ int_node, uint32_t *cid, InternalSums *sums, uint32_t *counts,
    uint32_t *cross, uint32_t cross_cap, RecOut o) {
    com_span_block(blockIdx.x, nblocks, rows, want, h, body4, ref, spanning, int_local, int_first,
                   int_node, cid, sums, counts, cross, cross_cap, o);
}

// ---- traversal groups -------------------------------------------------------------
// A group is a cell with at most group_max bodies whose parent holds more, or
// a lone body whose parent holds more.  Groups partition the bodies into
// spatially compact runs of the octree order.  Every sorted position starts
// at most one group: the starts of each scan tile are counted, and a second
// launch writes them to their places -- the group list comes out in octree
// order, so neighbouring groups share most of their walk.
__global__ void __launch_bounds__(kScanThreads) k_group_count(
    const uint32_t *__restrict__ group_size, uint32_t n, uint32_t *part) {
    __shared__ uint32_t sh[2 * kScanThreads / 64];
    const uint64_t i0 = (uint64_t)blockIdx.x * kScanTile + threadIdx.x;
    uint32_t c = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const uint64_t i = i0 + (uint64_t)k * kScanThreads;
        if (i < n) c += group_size[i] != 0;
    }
    const ScanPlace pl = scan_place(c, nullptr, 0, true, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = pl.total;
}

__global__ void __launch_bounds__(kScanThreads) k_group_list(
    const uint32_t *__restrict__ group_size, uint32_t n, const uint32_t *__restrict__ part,
    uint32_t nparts, bool scanned, TreeHdr *h, uint2 *groups) {
    __shared__ uint32_t sh[2 * kScanThreads / 64];
    const uint64_t i0 = (uint64_t)blockIdx.x * kScanTile + (uint64_t)threadIdx.x * kScanItems;
    uint32_t v[kScanItems], c = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        v[k] = i0 + k < n ? group_size[i0 + k] : 0u;
        c += v[k] != 0;
    }
    const ScanPlace pl = scan_place(c, part, nparts, scanned, sh);
    uint32_t g = pl.first + pl.before;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k)
        if (v[k]) groups[g++] = make_uint2((uint32_t)i0 + k, v[k]);
    if (blockIdx.x + 1 == gridDim.x && threadIdx.x == 0) h->group_count = pl.first + pl.total;
}

// ---- ensemble: the octrees of many systems ------------------------------------------
constexpr int kForestThreads = 1024;
constexpr int kForestWaves = kForestThreads / 64;
// Per-wave contiguous range [*b, *e) of m items: 16 ranges of whole 64-item
// groups, so a wave reads 64 consecutive items at a time (coalesced) and the
// ranges keep the item order wave by wave.
__device__ inline void wave_range(uint32_t m, uint32_t *b, uint32_t *e) {
    const uint32_t chunk = ((m + kForestWaves - 1) / kForestWaves + 63u) & ~63u;
    const uint32_t w = threadIdx.x >> 6;
    *b = min(m, w * chunk);
    *e = min(m, *b + chunk);
}

// Exclusive scan in place of a[0..m) (global memory, this workgroup only):
// wave totals, their scan, then a running wave scan over each wave's range.
__device__ inline uint32_t wg_scan_array(uint32_t *a, uint32_t m, uint32_t *wsum) {
    const uint32_t t = threadIdx.x, lane = t & 63u, w = t >> 6;
    uint32_t b, e;
    wave_range(m, &b, &e);
    uint32_t s = 0;
#pragma unroll 8
    for (uint32_t i = b + lane; i < e; i += 64) s += a[i];
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off, 64);
    if (lane == 0) wsum[w] = s;
    __syncthreads();
    if (t == 0) {
        uint32_t run = 0;
        for (int k = 0; k < kForestWaves; ++k) {
            const uint32_t c = wsum[k];
            wsum[k] = run;
            run += c;
        }
        wsum[kForestWaves] = run;
    }
    __syncthreads();
    uint32_t carry = wsum[w];
    const uint32_t total = wsum[kForestWaves];
    constexpr uint32_t kAhead = 8;  // loads and wave scans in flight
    for (uint32_t g = b; g < e; g += 64 * kAhead) {
        uint32_t v[kAhead], inc[kAhead];
#pragma unroll
        for (uint32_t u = 0; u < kAhead; ++u) {
            const uint32_t i = g + 64 * u + lane;
            v[u] = i < e ? a[i] : 0u;
            inc[u] = v[u];
        }
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
#pragma unroll
            for (uint32_t u = 0; u < kAhead; ++u) {
                const uint32_t o = __shfl_up(inc[u], off, 64);
                if (lane >= (uint32_t)off) inc[u] += o;
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < kAhead; ++u) {
            const uint32_t i = g + 64 * u + lane;
            if (i < e) a[i] = carry + inc[u] - v[u];
            carry += __shfl(inc[u], 63, 64);
        }
    }
    __syncthreads();
    return total;
}

// 1. Per Barnes-Hut system (one workgroup each): header reset, AABB including
// the origin (every partial starts at 0.0), then cubify into the header.
__global__ void __launch_bounds__(kForestThreads) k_forest_aabb(
    const EnsSystem *__restrict__ sys, const uint32_t *__restrict__ order,
    const double *__restrict__ gx, const double *__restrict__ gy, const double *__restrict__ gz,
    ForestBufs fb) {
    __shared__ double red[kForestWaves][6], ext[6];
    const uint32_t s = order[blockIdx.x];
    const EnsSystem S = sys[s];
    const uint32_t n = S.n, t = threadIdx.x;
    const double *x = gx + S.body_off, *y = gy + S.body_off, *z = gz + S.body_off;
    TreeHdr *h = fb.hdr + s;
    if (t == 0) {
        h->internal_count = 0;
        h->max_depth = 0;
        h->status = 0;
        h->deep_runs = 0;
        h->stack_peak = 0;
        h->group_count = 0;
        h->group_next = 0;
        h->cross_count = 0;
        h->corr_pairs = 0;
    }
    __syncthreads();  // the reset precedes every flag raised below
    Extents e;
#pragma unroll 8
    for (uint32_t i = t; i < n; i += kForestThreads) {
        const double p[3] = {x[i], y[i], z[i]};
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            e.bad |= !isfinite(p[c]);
            e.mn[c] = sycl_min(e.mn[c], p[c]);
            e.mx[c] = sycl_max(e.mx[c], p[c]);
        }
    }
    if (e.bad) raise_flag(h, kFlagAabb);
    wave_extents(e);
    if ((t & 63) == 0)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            red[t >> 6][c] = e.mn[c];
            red[t >> 6][3 + c] = e.mx[c];
        }
    __syncthreads();
    if (t < 6) {
        double v = red[0][t];
#pragma unroll
        for (int w = 1; w < kForestWaves; ++w)
            v = t < 3 ? sycl_min(v, red[w][t]) : sycl_max(v, red[w][t]);
        ext[t] = v;
    }
    __syncthreads();
    if (t == 0) {
        const RootCube r = cubify(ext);
        store_cube(h, r);
        if (!r.ok) raise_flag(h, kFlagAabb);
    }
}

// The largest 63-bit key: the padding between two systems' slots sorts after
// their bodies (ties keep slot order, and padding slots follow the bodies).
constexpr uint64_t kPadKey = ~0ull >> 1;

// 2. Keys of every slot j of the forest's body space (all systems at once):
// a Barnes-Hut system's body i = j - fb_off gets its key in the system's root
// cell and its packed record; padding and direct-sum slots get kPadKey.
__global__ void __launch_bounds__(kThreads) k_forest_keys(
    uint32_t slots, const uint16_t *__restrict__ fb_sys, const EnsSystem *__restrict__ sys,
    const double *__restrict__ gx, const double *__restrict__ gy, const double *__restrict__ gz,
    const double *__restrict__ gm, ForestBufs fb, uint64_t *key, uint32_t *val) {
    const uint32_t j = blockIdx.x * kThreads + threadIdx.x;
    if (j >= slots) return;
    const uint32_t s = fb_sys[j];
    const EnsSystem S = sys[s];
    const uint32_t i = j - S.fb_off;
    uint64_t k = kPadKey;
    if (S.bh && i < S.n) {
        TreeHdr *h = fb.hdr + s;
        Cell c{h->minx, h->miny, h->minz, h->edge};
        const uint32_t b = S.body_off + i;
        const double px = gx[b], py = gy[b], pz = gz[b], pm = gm[b];
        k = key_from(c, px, py, pz);
        fb.body4[j] = make_double4(px, py, pz, pm);
        fb.klo[j] = k;  // the full key by slot, for k_forest_rekey
        if (pm == 0) raise_flag(h, kFlagZeroMass);  // an error of the reference's centre of mass
    }
    key[j] = k;
    val[j] = j;
}

// Low key bits sorted by the first forest-wide sort; the second sorts the
// system above the remaining high bits.  Both sorts then take 4 passes of 9
// bits (for up to 512 systems), the minimum of a sort.
constexpr int kForestLowBits = 36;

// 3b. After the sort by the low key bits: each slot's key becomes (its system,
// its high key bits), for the stable sort that gathers every system's slots
// back into its own range, in key order.  A slot's system is the last whose
// first slot is at or before it: up to kSysrankLds systems the first slots sit
// in LDS and each slot's system is found by bisection there, instead of a
// gathered load of fb_sys at a scattered slot.
constexpr uint32_t kSysrankLds = 8192;
constexpr uint32_t kSysrankBlocks = 2048;
__global__ void __launch_bounds__(kThreads) k_forest_sysrank(uint32_t slots, uint32_t nsys,
                                                             const uint32_t *__restrict__ first,
                                                             const uint16_t *__restrict__ fb_sys,
                                                             uint64_t *key,
                                                             const uint32_t *__restrict__ val) {
    __shared__ uint32_t fl[kSysrankLds];
    const bool lds = nsys <= kSysrankLds;
    if (lds) {
        for (uint32_t k = threadIdx.x; k < nsys; k += kThreads) fl[k] = first[k];
        __syncthreads();
    }
    const uint32_t stride = gridDim.x * kThreads;
    for (uint32_t j = blockIdx.x * kThreads + threadIdx.x; j < slots; j += stride) {
        const uint32_t v = val[j];
        uint32_t sys;
        if (lds) {
            // fl[0] = 0 <= v: keep fl[lo] <= v while halving the range
            uint32_t lo = 0, len = nsys;
            while (len > 1) {
                const uint32_t half = len >> 1;
                if (fl[lo + half] <= v) lo += half;
                len -= half;
            }
            sys = lo;
        } else {
            sys = fb_sys[v];
        }
        key[j] = ((uint64_t)sys << (3 * kKeyLevels - kForestLowBits)) | (key[j] >> kForestLowBits);
    }
}

// After the forest-wide sort, the build alternates stages over every body
// slot of the forest (all systems at once, the whole GPU) with stages of one
// workgroup per system, which hold what needs a barrier across one system:
// the cell-numbering scan, the level-by-level centre of mass and the group
// scan.  Every stage is the one-system build's per-element step; the trees
// are bit-identical to a one-system build.

// A slot's system and its index inside that system's slots.
struct SlotSys {
    uint32_t s, li;
    EnsSystem S;
};
__device__ inline SlotSys slot_sys(uint32_t j, const uint16_t *__restrict__ fb_sys,
                                   const EnsSystem *__restrict__ sys) {
    SlotSys r;
    r.s = fb_sys[j];
    r.S = sys[r.s];
    r.li = j - r.S.fb_off;
    return r;
}

// 3. The full keys of the bodies in sorted order (the second sort kept only
// the high key bits; k_forest_keys left every slot's full key in klo, which
// holds nothing else until the deep runs' second key words), and the
// system-local body indices.  `sorted` may be fb.sidx itself: each slot is
// read, then rewritten, by one thread.
__global__ void __launch_bounds__(kThreads) k_forest_rekey(uint32_t slots,
                                                           const uint16_t *__restrict__ fb_sys,
                                                           const EnsSystem *__restrict__ sys,
                                                           ForestBufs fb, const uint32_t *sorted) {
    const uint32_t j = blockIdx.x * kThreads + threadIdx.x;
    if (j >= slots) return;
    const SlotSys ss = slot_sys(j, fb_sys, sys);
    if (!ss.S.bh || ss.li >= ss.S.n) return;
    TreeHdr *h = fb.hdr + ss.s;
    uint32_t q = sorted[j] - ss.S.fb_off;
    if (q >= ss.S.n) {  // only after a failed sort, which the flag reports
        raise_flag(h, kFlagSortWait);
        q = 0;
    }
    fb.skey[j] = fb.klo[ss.S.fb_off + q];  // one gathered 8-byte key per body
    fb.sidx[j] = q;
}

// 4. lcp of each adjacent pair of a system's sorted bodies; a run of bodies
// sharing all 21 digits is extended and sorted by its first pair's thread.
__global__ void __launch_bounds__(kThreads) k_forest_lcp(
    uint32_t slots, const uint16_t *__restrict__ fb_sys, const EnsSystem *__restrict__ sys,
    const double *__restrict__ gx, const double *__restrict__ gy, const double *__restrict__ gz,
    ForestBufs fb) {
    const uint32_t j = blockIdx.x * kThreads + threadIdx.x;
    if (j >= slots) return;
    const SlotSys ss = slot_sys(j, fb_sys, sys);
    if (!ss.S.bh || ss.li + 1 >= ss.S.n) return;
    TreeHdr *h = fb.hdr + ss.s;
    const Cell root{h->minx, h->miny, h->minz, h->edge};
    const uint32_t fo = ss.S.fb_off, bo = ss.S.body_off;
    lcp_at(ss.li, gx + bo, gy + bo, gz + bo, ss.S.n, root, h, fb.skey + fo, fb.sidx + fo,
           fb.klo + fo, fb.lcp + fo);
}

// 5. chain: the internal cells owned by each pair.  (A system's deepest leaf
// is not needed by the ensemble; the header's max_depth stays 0.)
__global__ void __launch_bounds__(kThreads) k_forest_chain(uint32_t slots,
                                                           const uint16_t *__restrict__ fb_sys,
                                                           const EnsSystem *__restrict__ sys,
                                                           ForestBufs fb) {
    const uint32_t j = blockIdx.x * kThreads + threadIdx.x;
    if (j >= slots) return;
    const SlotSys ss = slot_sys(j, fb_sys, sys);
    if (ss.S.bh && ss.li + 1 < ss.S.n) chain_at(ss.li, fb.lcp + ss.S.fb_off, fb.chain + ss.S.fb_off);
}

// 6. Per system: cell numbering (exclusive scan of the chain), the internal
// cell count, the empty node slots the topology fills in, and an empty table
// of block-crossing cells.
__global__ void __launch_bounds__(kForestThreads) k_forest_number(
    const EnsSystem *__restrict__ sys, const uint32_t *__restrict__ order, ForestBufs fb) {
    __shared__ uint32_t wsum[kForestWaves + 1];
    const uint32_t s = order[blockIdx.x];
    const EnsSystem S = sys[s];
    const uint32_t n = S.n;
    TreeHdr *h = fb.hdr + s;
    const uint32_t I_all = n > 1 ? wg_scan_array(fb.chain + S.fb_off, n - 1, wsum) : 0u;
    if (threadIdx.x == 0) h->internal_count = I_all;
    const uint32_t I = min(I_all, S.icap);
    int32_t *ref = fb.ref + S.node_off;
    for (uint64_t j = threadIdx.x; j < 1 + 8ull * I; j += kForestThreads) ref[j] = kRefEmpty;
    uint32_t *spanning = fb.spanning + S.span_off;
    const uint32_t span_cap = kMaxDepth * ((n + kComBlock - 1) / kComBlock);
    for (uint32_t j = threadIdx.x; j < span_cap; j += kForestThreads) spanning[j] = kNoCell;
}

// 7. Topology of every body of the forest, as k_link: a block stages the keys
// of its slots and kLinkBack before them (whatever systems they belong to;
// a search only reads keys of its own system).  Cells are local to, or cross,
// the system's kComBlock-body blocks as in the one-system build.
__global__ void __launch_bounds__(kThreads) k_forest_link(uint32_t slots,
                                                          const uint16_t *__restrict__ fb_sys,
                                                          const EnsSystem *__restrict__ sys,
                                                          ForestBufs fb) {
    const uint32_t b0 = blockIdx.x * kThreads;
    KeyView kv{fb.skey, fb.klo, fb.lcp, fb.chain};
    link_window(kv, b0, slots);
    const uint32_t j = b0 + threadIdx.x;
    if (j >= slots) return;
    const SlotSys ss = slot_sys(j, fb_sys, sys);
    const EnsSystem &S = ss.S;
    if (!S.bh || ss.li >= S.n) return;
    const uint32_t fo = S.fb_off, io = S.int_off;
    // arrays and window bounds relative to the system's first slot; the unsigned
    // differences in KeyView place a position in or out of the window correctly
    // also when the window starts before the system
    kv.skey += fo;
    kv.klo += fo;
    kv.lcp += fo;
    kv.off += fo;
    kv.w0 -= fo;
    kv.w1 -= fo;
    link_at(ss.li, S.n, S.icap, fb.hdr + ss.s, kv, fb.sidx + fo,
            fb.ref + S.node_off, fb.int_depth + io, fb.int_node + io,
            fb.body_node + fo, fb.int_local + io, fb.spanning + S.span_off,
            kMaxDepth * ((S.n + kComBlock - 1) / kComBlock), fb.int_first + io, kComBlock,
            kComSuper);
}

// The one-system build's view of system s, for the centre-of-mass passes.
struct ForestTree {
    EnsSystem S;
    TreeHdr *h;
    RecOut o;
};
__device__ inline ForestTree forest_tree(const EnsSystem *__restrict__ sys, uint32_t s,
                                         const ForestBufs &fb, double G, GroupRule rule) {
    ForestTree f;
    f.S = sys[s];
    f.h = fb.hdr + s;
    const uint32_t fo = f.S.fb_off;
    f.o = RecOut{G, 0, 1, nullptr, fb.rec + f.S.node_off, fb.group_size + fo,
                 fb.group_slot + fo, rule};
    return f;
}

// 8. Centre of mass, node records and group marks, as k_com_local and
// k_com_span, for the blocks of every system in one launch each: block
// (system, b) of fb.blk_tab; then (system, super-block) of fb.span_tab
// (want 0), then the systems of fb.big_tab (want 2: cells crossing
// super-block ends).
__global__ void __launch_bounds__(kComLocalThreads) k_forest_com_local(
    const EnsSystem *__restrict__ sys, ForestBufs fb, double G, GroupRule rule) {
    const uint2 e = fb.blk_tab[blockIdx.x];
    const ForestTree f = forest_tree(sys, e.x, fb, G, rule);
    const EnsSystem &S = f.S;
    const uint32_t fo = S.fb_off, io = S.int_off;
    com_local_block(e.y, S.n, S.icap, f.h, fb.body4 + fo, fb.sidx + fo, fb.body_node + fo,
                    fb.ref + S.node_off, fb.chain + fo, fb.int_depth + io, fb.int_local + io,
                    fb.int_first + io, fb.int_node + io, fb.int_lvl + io, fb.int_sums + io, fb.int_count + io, f.o);
}

__global__ void __launch_bounds__(kComThreads) k_forest_com_span(
    const EnsSystem *__restrict__ sys, const uint2 *__restrict__ tab, uint32_t want, ForestBufs fb,
    double G, GroupRule rule) {
    const uint2 e = tab[blockIdx.x];
    const ForestTree f = forest_tree(sys, e.x, fb, G, rule);
    const EnsSystem &S = f.S;
    const uint32_t fo = S.fb_off, io = S.int_off;
    const uint32_t nblocks = (S.n + kComBlock - 1) / kComBlock;
    com_span_block(e.y, nblocks, want == 2 ? nblocks : kComSuperBlocks, want, f.h,
                   fb.body4 + fo, fb.ref + S.node_off, fb.spanning + S.span_off,
                   fb.int_local + io, fb.int_first + io, fb.int_node + io, fb.int_lvl + io,
                   fb.int_sums + io, fb.int_count + io, fb.cross + S.cross_off,
                   kMaxDepth * ((S.n + kComSuper - 1) / kComSuper + 1), f.o);
}

// 9. The traversal groups of every system: after one exclusive scan of the
// group marks over all slots of the forest (padding included, whatever it
// holds: a system's group numbers are differences of the scan, exact modulo
// 2^32), each group start writes its group; a system's first slot writes its
// group count and merges its status flags into *status.
__global__ void __launch_bounds__(kThreads) k_forest_groups(uint32_t slots,
                                                            const uint16_t *__restrict__ fb_sys,
                                                            const EnsSystem *__restrict__ sys,
                                                            ForestBufs fb,
                                                            const uint32_t *__restrict__ total,
                                                            uint32_t *items, uint32_t *status) {
    const uint32_t j = blockIdx.x * kThreads + threadIdx.x;
    if (j >= slots) return;
    const SlotSys ss = slot_sys(j, fb_sys, sys);
    const EnsSystem &S = ss.S;
    if (!S.bh || ss.li >= S.n) return;
    const uint32_t fo = S.fb_off;
    const uint32_t base = fb.group_slot[fo];
    const uint32_t gs = fb.group_size[j];
    if (gs) fb.groups[fo + (fb.group_slot[j] - base)] = make_uint2(ss.li, gs);
    if (ss.li == 0) {
        const uint32_t end = fo + S.n < slots ? fb.group_slot[fo + S.n] : *total;
        const uint32_t ng = end - base;
        TreeHdr *h = fb.hdr + ss.s;
        h->group_count = ng;
        items[ss.s] = ng;
        // flags were raised with device-scope atomics: read the word the same way
        const uint32_t st = __hip_atomic_load(&h->status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (st) atomicOr(status, st);
    }
}

}  // namespace

void launch_forest_build(const EnsSystem *sys, const uint32_t *order, uint32_t nbh,
                         uint32_t nsys, const double *x, const double *y, const double *z,
                         const double *m, double G, const ForestBufs &fb, GroupRule rule,
                         uint32_t *items, uint32_t *status, hipStream_t s) {
    if (nbh == 0) return;
    hipLaunchKernelGGL(k_forest_aabb, dim3(nbh), dim3(kForestThreads), 0, s, sys, order, x, y, z,
                       fb);
    // LSD over (system, key): one radix sort of every system's slots by the
    // low key bits, then a stable one by (system, high key bits): each
    // system's bodies end in its own slot range, in key order with ties in
    // index order (the order of a sort of that system alone)
    const uint32_t slots = fb.slots, blocks = ceil_div(slots, kThreads);
    uint64_t *k = fb.skey, *ka = fb.skey_alt;
    uint32_t *v = fb.sidx, *va = fb.sidx_alt;
    hipLaunchKernelGGL(k_forest_keys, dim3(blocks), dim3(kThreads), 0, s, slots,
                       (const uint16_t *)fb.fb_sys, sys, x, y, z, m, fb, k, v);
    SortEnd end = radix_sort_u64_u32(k, v, ka, va, slots, kForestLowBits, fb.radix_ctl, status,
                                     false, s);
    if (end == SortEnd::kRejected) return;  // reported in *status
    if (end == SortEnd::kInAlt) {
        std::swap(k, ka);
        std::swap(v, va);
    }
    hipLaunchKernelGGL(k_forest_sysrank, dim3(std::min(blocks, kSysrankBlocks)), dim3(kThreads), 0,
                       s, slots, nsys, (const uint32_t *)fb.sys_first, (const uint16_t *)fb.fb_sys,
                       k, (const uint32_t *)v);
    int sys_bits = 1;
    while (sys_bits < 16 && (1u << sys_bits) < nsys) ++sys_bits;
    // its own control words: a control buffer must always see the same pass count
    end = radix_sort_u64_u32(k, v, ka, va, slots, 3 * kKeyLevels - kForestLowBits + sys_bits,
                             fb.radix_ctl_sys, status, false, s);
    if (end == SortEnd::kRejected) return;
    if (end == SortEnd::kInAlt) {
        std::swap(k, ka);
        std::swap(v, va);
    }
    const uint16_t *fs = fb.fb_sys;
    hipLaunchKernelGGL(k_forest_rekey, dim3(blocks), dim3(kThreads), 0, s, slots, fs, sys, fb,
                       (const uint32_t *)v);
    hipLaunchKernelGGL(k_forest_lcp, dim3(blocks), dim3(kThreads), 0, s, slots, fs, sys, x, y, z,
                       fb);
    hipLaunchKernelGGL(k_forest_chain, dim3(blocks), dim3(kThreads), 0, s, slots, fs, sys, fb);
    hipLaunchKernelGGL(k_forest_number, dim3(nbh), dim3(kForestThreads), 0, s, sys, order, fb);
    hipLaunchKernelGGL(k_forest_link, dim3(blocks), dim3(kThreads), 0, s, slots, fs, sys, fb);
    if (fb.nblk)
        hipLaunchKernelGGL(k_forest_com_local, dim3(fb.nblk), dim3(kComLocalThreads), 0, s, sys, fb,
                           G, rule);
    if (fb.nspan)
        hipLaunchKernelGGL(k_forest_com_span, dim3(fb.nspan), dim3(kComThreads), 0, s, sys,
                           (const uint2 *)fb.span_tab, 0u, fb, G, rule);
    if (fb.nbig)
        hipLaunchKernelGGL(k_forest_com_span, dim3(fb.nbig), dim3(kComThreads), 0, s, sys,
                           (const uint2 *)fb.big_tab, 2u, fb, G, rule);
    uint32_t *total = fb.scan_part + (fb.scan_cap - 1);
    scan_exclusive_u32(fb.group_slot, fb.group_slot, slots, total, fb.scan_part, fb.scan_cap - 1,
                       s);
    hipLaunchKernelGGL(k_forest_groups, dim3(blocks), dim3(kThreads), 0, s, slots, fs, sys, fb,
                       (const uint32_t *)total, items, status);
}

// workgroups of the AABB pass: 1024 bodies each, at most kAabbBlocks
uint32_t aabb_blocks(uint32_t n) {
    return std::min<uint32_t>(kAabbBlocks, ceil_div(n, 4 * kAabbThreads));
}

void launch_aabb(const TreeBufs &t, const double *x, const double *y, const double *z,
                 hipStream_t s) {
    hipLaunchKernelGGL(k_aabb_partial, dim3(aabb_blocks(t.n)), dim3(kAabbThreads), 0, s, x, y, z,
                       t.n, t.aabb_part);
}

void launch_keys(TreeBufs &t, const double *x, const double *y, const double *z,
                 const double *m, hipStream_t s) {
    hipLaunchKernelGGL(k_keys, dim3(std::min(kKeyBlocks, ceil_div(t.n, kKeyThreads))),
                       dim3(kKeyThreads), 0, s, x, y, z, m, t.n, (const double *)t.aabb_part,
                       aabb_blocks(t.n), t.hdr, t.skey, t.sidx, t.body4, t.scan_part,
                       ceil_div(t.n, kScanTile), radix_count_args(t.n, t.radix_ctl));
}

void launch_key_sort(TreeBufs &t, hipStream_t s) {
    // a rejected sort (2^30 bodies or more, which the context's capacity
    // check already excludes) raises kFlagSortSize; the build reports it
    if (radix_sort_u64_u32(t.skey, t.sidx, t.skey_alt, t.sidx_alt, t.n, 3 * kKeyLevels,
                           t.radix_ctl, &t.hdr->status, true, s) == SortEnd::kInAlt) {
        std::swap(t.skey, t.skey_alt);
        std::swap(t.sidx, t.sidx_alt);
    }
}

void launch_topology(const TreeBufs &t, const double *x, const double *y, const double *z,
                     hipStream_t s) {
    const uint32_t n = t.n;
    const dim3 grid(ceil_div(n, kThreads));
    if (n > 1) {
        hipLaunchKernelGGL(k_lcp, grid, dim3(kThreads), 0, s, x, y, z, n, t.hdr, t.skey, t.sidx,
                           t.klo, t.lcp, t.scan_part);
        const uint32_t nparts = ceil_div(n - 1, kScanTile);
        const bool scanned = scan_parts_if_many(t.scan_part, nparts, s);
        hipLaunchKernelGGL(k_number, dim3(nparts), dim3(kScanThreads), 0, s,
                           (const int32_t *)t.lcp, n - 1, t.chain, (const uint32_t *)t.scan_part,
                           nparts, scanned, t.hdr, t.icap, t.ref, t.spanning, t.spanning_cap);
    }
    KeyView kv{t.skey, t.klo, t.lcp, t.chain};
    hipLaunchKernelGGL(k_link, grid, dim3(kThreads), 0, s, n, t.icap, t.hdr, kv,
                       (const uint32_t *)t.sidx, t.ref, t.int_depth, t.int_node,
                       t.body_node, t.int_local, t.spanning, t.spanning_cap, t.int_first);
}

void launch_max_depth(const TreeBufs &t, hipStream_t s) {
    if (t.n < 2) return;
    const uint32_t blocks = std::min<uint32_t>(kDepthBlocks, ceil_div(t.n, kThreads));
    hipLaunchKernelGGL(k_max_depth, dim3(blocks), dim3(kThreads), 0, s, (const int32_t *)t.lcp,
                       t.n, t.hdr);
}

void launch_com(const TreeBufs &t, double G, bool f64, bool f32, GroupRule rule, hipStream_t s) {
    const uint32_t nblocks = ceil_div(t.n, kComBlock);
    const RecOut o{G,     (int)f64,     (int)f32,     t.cm,
                   t.rec, t.group_size, nullptr,     rule};
    hipLaunchKernelGGL(k_com_local, dim3(nblocks), dim3(kComLocalThreads), 0, s, t.n, t.icap, t.hdr,
                       (const double4 *)t.body4, (const uint32_t *)t.sidx, (const uint32_t *)t.body_node,
                       (const int32_t *)t.ref, (const uint32_t *)t.chain, (const uint8_t *)t.int_depth,
                       (const uint8_t *)t.int_local, (const uint32_t *)t.int_first,
                       (const uint32_t *)t.int_node, t.int_lvl, t.int_sums, t.int_count, o);
    if (nblocks >= 2) {
        hipLaunchKernelGGL(k_com_span, dim3(ceil_div(nblocks, kComSuperBlocks)), dim3(kComThreads),
                           0, s, nblocks, kComSuperBlocks, 0u, t.hdr, (const double4 *)t.body4,
                           (const int32_t *)t.ref, (const uint32_t *)t.spanning,
                           (const uint8_t *)t.int_local, (const uint32_t *)t.int_first,
                           (const uint32_t *)t.int_node, t.int_lvl, t.int_sums, t.int_count,
                           t.cross, t.cross_cap, o);
        if (nblocks > kComSuperBlocks)
            hipLaunchKernelGGL(k_com_span, dim3(1), dim3(kComThreads), 0, s, nblocks, nblocks, 2u,
                               t.hdr, (const double4 *)t.body4, (const int32_t *)t.ref,
                               (const uint32_t *)t.spanning, (const uint8_t *)t.int_local,
                               (const uint32_t *)t.int_first, (const uint32_t *)t.int_node, t.int_lvl,
                               t.int_sums, t.int_count, t.cross, t.cross_cap, o);
    }
    if (f32) {
        const uint32_t nparts = ceil_div(t.n, kScanTile);
        if (nparts > 1)  // one tile has none before it (a launch of 3.6 us)
            hipLaunchKernelGGL(k_group_count, dim3(nparts), dim3(kScanThreads), 0, s,
                               (const uint32_t *)t.group_size, t.n, t.scan_part);
        const bool scanned = scan_parts_if_many(t.scan_part, nparts, s);
        hipLaunchKernelGGL(k_group_list, dim3(nparts), dim3(kScanThreads), 0, s,
                           (const uint32_t *)t.group_size, t.n, (const uint32_t *)t.scan_part,
                           nparts, scanned, t.hdr, t.groups);
    }
}

}  // namespace nb
