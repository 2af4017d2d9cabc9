// nb_scan.hip -- device-wide exclusive scan and stable key sorts.
//
// All are written for 64-lane wavefronts: prefix sums use __shfl_up inside a
// wave and LDS across the 4 waves of a 256-thread block; the sorts rank keys
// stably with a 9-ballot "match any" on the 9-bit digit, so no per-thread
// histogram is needed.  Small and middling sorts take one launch of tiles sorted
// in LDS, then merges; large ones one launch per digit.  The ensemble uses the
// scan for its group lists, the octree builds the sorts for the octant keys
// (rocPRIM/hipCUB are not used).
#include "nb_internal.h"

namespace nb {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr int kItems = kScanTile / kThreads;
constexpr int kRadixTile = 4096;       // keys per radix tile
constexpr int kRadixTileBig = 8192;    // keys per tile from kRadixBigMin keys on
constexpr int kRadixTileWide = 10240;  // or, where fewer rounds of tiles result
constexpr uint32_t kRadixBigMin = 1u << 21;
constexpr uint32_t kCus = 256;
constexpr uint32_t kSortMergeMax = 1u << 18;  // k_sort_tiles and k_merge_runs; above, passes
constexpr int kPassThreads = 512;
constexpr int kPassWaves = kPassThreads / 64;

__device__ inline uint32_t lane_id() { return threadIdx.x & 63u; }

__device__ inline uint32_t wave_inclusive_scan(uint32_t v) {
    const uint32_t lane = lane_id();
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t t = __shfl_up(v, d, 64);
        if (lane >= (uint32_t)d) v += t;
    }
    return v;
}

// Exclusive prefix of v over the block's 256 threads; *total = block sum.
__device__ inline uint32_t block_exclusive_scan(uint32_t v, uint32_t *sh, uint32_t *total) {
    const uint32_t inc = wave_inclusive_scan(v);
    const uint32_t w = threadIdx.x >> 6;
    if (lane_id() == 63) sh[w] = inc;
    __syncthreads();
    uint32_t off = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < kWaves; ++i) {
        const uint32_t s = sh[i];
        off += (uint32_t)i < w ? s : 0u;
        tot += s;
    }
    __syncthreads();
    *total = tot;
    return off + inc - v;
}

__global__ void __launch_bounds__(kThreads) k_scan_reduce(const uint32_t *__restrict__ in,
                                                          uint32_t n, uint32_t *part) {
    __shared__ uint32_t sh[kWaves];
    const uint64_t base = (uint64_t)blockIdx.x * kScanTile;
    uint32_t s = 0;
#pragma unroll
    for (int k = 0; k < kItems; ++k) {
        const uint64_t i = base + (uint64_t)k * kThreads + threadIdx.x;
        if (i < n) s += in[i];
    }
    uint32_t tot;
    block_exclusive_scan(s, sh, &tot);
    if (threadIdx.x == 0) part[blockIdx.x] = tot;
}

// One block: exclusive scan of the nb tile sums in place; *total = grand total.
__global__ void __launch_bounds__(kThreads) k_scan_parts(uint32_t *part, uint32_t nb,
                                                         uint32_t *total) {
    __shared__ uint32_t sh[kWaves];
    const uint32_t per = (nb + kThreads - 1) / kThreads;
    const uint32_t b0 = threadIdx.x * per;
    uint32_t s = 0;
    for (uint32_t i = 0; i < per; ++i)
        if (b0 + i < nb) s += part[b0 + i];
    uint32_t tot;
    uint32_t off = block_exclusive_scan(s, sh, &tot);
    for (uint32_t i = 0; i < per; ++i) {
        if (b0 + i < nb) {
            const uint32_t v = part[b0 + i];
            part[b0 + i] = off;
            off += v;
        }
    }
    if (threadIdx.x == 0 && total) *total = tot;
}

// Each thread scans kItems consecutive values; out may alias in.
__global__ void __launch_bounds__(kThreads) k_scan_down(const uint32_t *in, uint32_t *out,
                                                        uint32_t n, const uint32_t *part) {
    __shared__ uint32_t sh[kWaves];
    const uint64_t base = (uint64_t)blockIdx.x * kScanTile + (uint64_t)threadIdx.x * kItems;
    uint32_t v[kItems];
    uint32_t s = 0;
#pragma unroll
    for (int k = 0; k < kItems; ++k) {
        const uint64_t i = base + k;
        v[k] = i < n ? in[i] : 0u;
        s += v[k];
    }
    uint32_t tot;
    uint32_t off = block_exclusive_scan(s, sh, &tot) + part[blockIdx.x];
#pragma unroll
    for (int k = 0; k < kItems; ++k) {
        const uint64_t i = base + k;
        if (i < n) out[i] = off;
        off += v[k];
    }
}

// ---- radix sort: one sweep per digit -----------------------------------------
//
// Each pass is one k_radix_pass launch: a block takes the next tile id from a
// counter, publishes its tile's per-digit counts, ranks its keys in LDS, and
// learns how many keys of each digit the earlier tiles hold from their
// published counts (decoupled look-back: a tile that has finished its
// look-back publishes an inclusive prefix, so later tiles stop there).  Tile
// ids are handed out in the order blocks start, so every tile a block waits on
// belongs to a block that is running and that publishes its counts before it
// waits on anything: every wait ends.  The digit totals (which do not depend
// on the order) come from
// k_radix_count (or the caller's own kernel, see RadixCount) for pass 0 and from pass p - 1 for
// pass p, which counts the next digit of the keys it has loaded anyway.
//
// Digits are 9 bits wide: 7 passes cover the 63-bit octree keys (an odd
// count, so the result lands in the scratch buffers and the caller swaps).
//
// Control words (u32):
//   [0, 7 * 512)           digit totals of pass p at p * kBins
//   kCtlTiles + p          tile counter of pass p
//   kCtlStatus + plane     two status planes of nb x kBins words, plane p & 1
//                          for pass p; pass p clears its tile's row of the
//                          other plane for pass p + 1, and k_radix_count
//                          clears plane 0 (an odd pass count leaves it used)
// Pass p > 0 zeroes the totals and the tile counter of pass p - 1 (that
// launch has ended), and pass 0 those of the last pass.  Between sorts every
// word is therefore zero except the last pass's totals and tile counter,
// which pass 0 clears before pass passes - 2 adds to them (allocation sets
// everything to zero).  A status word is 0 (not yet published),
// kStatAgg | tile count, or kStatPrefix | count in tiles [0, t].  Counts stay
// below 2^30: octree contexts hold fewer than 2^29 bodies.

constexpr int kDigitBits = 9;
constexpr uint32_t kBins = kRadixBins;
static_assert(kBins == 1u << kDigitBits, "digit width");
constexpr int kMaxPasses = 7;
static_assert(kMaxPasses * kDigitBits >= 63, "the passes cover the keys");
static_assert(kBins == (uint32_t)kPassThreads, "thread tid owns digit tid");
constexpr uint32_t kCtlTiles = kMaxPasses * kBins;
constexpr uint32_t kCtlStatus = kCtlTiles + 64;  // planes start 256-byte aligned
constexpr uint32_t kStatAgg = 1u << 30;
constexpr uint32_t kStatPrefix = 2u << 30;
constexpr uint32_t kStatCount = kStatAgg - 1;
constexpr int kLookWindow = 32;               // predecessor tiles read per look-back step
constexpr uint32_t kLookSpinLimit = 1u << 22; // a safety net: the waits end (see above)
constexpr int kMinPasses = 4;  // the control-word rotation above needs 3 or more
constexpr int kCountThreads = 1024;
constexpr uint32_t kCountBlocks = 256;

__device__ inline uint32_t status_load(const uint32_t *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void status_store(uint32_t *p, uint32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A sort that cannot run reports it in the caller's status word.
__global__ void k_raise_flag(uint32_t *flags, uint32_t f) {
    if (threadIdx.x == 0) atomicOr(flags, f);
}

// Totals of the lowest digit of the keys: total[digit].  Also clears the
// status plane of the first pass, plane0[0, plane_words): the previous sort's
// last pass used it when the pass count is odd.
__global__ void __launch_bounds__(kCountThreads) k_radix_count(const uint64_t *__restrict__ keys,
                                                               uint32_t n,
                                                               uint32_t *__restrict__ total,
                                                               uint32_t *__restrict__ plane0,
                                                               uint64_t plane_words) {
    __shared__ uint32_t h[kBins];
    if (threadIdx.x < kBins) h[threadIdx.x] = 0;
    __syncthreads();
    const uint64_t stride = (uint64_t)gridDim.x * kCountThreads;
    for (uint64_t i = (uint64_t)blockIdx.x * kCountThreads + threadIdx.x; i < plane_words; i += stride)
        plane0[i] = 0;
#pragma unroll 4
    for (uint64_t i = (uint64_t)blockIdx.x * kCountThreads + threadIdx.x; i < n; i += stride)
        atomicAdd(&h[(uint32_t)keys[i] & (kBins - 1)], 1u);
    __syncthreads();
    if (threadIdx.x < kBins && h[threadIdx.x]) atomicAdd(&total[threadIdx.x], h[threadIdx.x]);
}

// Exclusive prefix over the block's threads of one value per thread (thread
// tid owns digit tid); ws holds kPassWaves words and is not reused.
__device__ inline uint32_t digit_exclusive_scan(uint32_t c, uint32_t *ws) {
    const uint32_t inc = wave_inclusive_scan(c);
    const uint32_t w = threadIdx.x >> 6;
    if (lane_id() == 63) ws[w] = inc;
    __syncthreads();
    uint32_t ex = inc - c;
    for (uint32_t k = 0; k < w; ++k) ex += ws[k];
    return ex;
}

// Keys of digit d in tiles [0, t), t > 0: walk back from tile t - 1,
// kLookWindow tiles per step, adding published counts up to and including the
// first inclusive prefix.  False if a predecessor never published (cannot
// happen, see above; the caller then raises a flag instead of waiting forever).
__device__ inline bool look_back(const uint32_t *stat, uint32_t t, uint32_t d, uint32_t *excl) {
    uint32_t sum = 0, spins = 0;
    int64_t j = (int64_t)t - 1;
    for (;;) {
        uint32_t v[kLookWindow];
#pragma unroll
        for (int k = 0; k < kLookWindow; ++k)
            v[k] = j - k >= 0 ? status_load(stat + (uint64_t)(j - k) * kBins + d) : kStatPrefix;
        bool pending = false;
#pragma unroll
        for (int k = 0; k < kLookWindow; ++k) pending |= v[k] == 0;
        while (pending) {
            if (++spins > kLookSpinLimit) return false;
            __builtin_amdgcn_s_sleep(2);
            pending = false;
#pragma unroll
            for (int k = 0; k < kLookWindow; ++k) {
                if (v[k] == 0) v[k] = status_load(stat + (uint64_t)(j - k) * kBins + d);
                pending |= v[k] == 0;
            }
        }
        bool found = false;
#pragma unroll
        for (int k = 0; k < kLookWindow; ++k) {
            if (!found) {
                sum += v[k] & kStatCount;
                found = v[k] >= kStatPrefix;
            }
        }
        if (found) {
            *excl = sum;
            return true;
        }
        j -= kLookWindow;
    }
}

// Lanes of the wave whose digit equals the lane's own (valid lanes only): one
// ballot per digit bit.
__device__ __forceinline__ uint64_t digit_peers(uint32_t d, bool valid) {
    uint64_t peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < kDigitBits; ++b) {
        const bool bit = (d >> b) & 1u;
        const uint64_t bal = __ballot(bit);
        peers &= bit ? bal : ~bal;
    }
    return peers;
}
__device__ __forceinline__ uint64_t lanes_below() {
    const uint32_t lane = lane_id();
    return lane == 0 ? 0ull : (~0ull >> (64u - lane));
}

// One stable pass over digit (key >> 9 pass) & 511 of a tile of kTile
// keys.  Wave w holds the tile's keys [w * kTile / 8, (w + 1) * kTile / 8) and
// ranks them 64 at a time against its own digit counters, with no barrier between
// rounds: a key's place among its digit's keys in the tile is (same digit in
// earlier waves) + (in earlier rounds of its wave) + (in lower lanes of its
// round), so the order is stable.  The tile is reordered in LDS by digit and
// written out digit run by digit run, so consecutive threads write
// consecutive addresses.
template <int kTile>
__global__ void __launch_bounds__(kPassThreads) k_radix_pass(
    const uint64_t *__restrict__ keys, const uint32_t *__restrict__ vals,
    uint64_t *__restrict__ okeys, uint32_t *__restrict__ ovals, uint32_t n, int pass, int passes,
    uint32_t *__restrict__ ctl, uint32_t nb, uint32_t *__restrict__ flags) {
    __shared__ uint32_t wcnt[kPassWaves][kBins];  // digit-d keys of wave w, then their first place
    __shared__ uint32_t next_hist[kBins];          // tile histogram of the next pass's digit
    __shared__ uint32_t dbase[kBins];              // first tile position of digit d
    __shared__ uint32_t gbase[kBins];              // output position of the tile's first digit-d key
    __shared__ uint32_t wsum[2][kPassWaves];
    __shared__ uint64_t lk[kTile];
    __shared__ uint32_t lv[kTile];
    __shared__ uint32_t tile_id, stuck;
    const uint32_t tid = threadIdx.x, lane = lane_id(), w = tid >> 6;
    const bool owner = tid < kBins;  // thread tid owns digit tid
    const int shift = kDigitBits * pass;
    uint32_t *total = ctl + pass * kBins;
    uint32_t *stat = ctl + kCtlStatus + (uint64_t)(pass & 1) * kBins * nb;
    uint32_t *stat_next = ctl + kCtlStatus + (uint64_t)((pass + 1) & 1) * kBins * nb;
    const bool has_next = pass + 1 < passes;
    if (tid == 0) {
        tile_id = atomicAdd(ctl + kCtlTiles + pass, 1u);
        stuck = 0;
    }
    for (uint32_t i = tid; i < kPassWaves * kBins; i += kPassThreads) (&wcnt[0][0])[i] = 0;
    if (owner) next_hist[tid] = 0;
    __syncthreads();
    const uint32_t t = tile_id;
    if (t >= nb) {  // only with corrupt control words: report it and touch nothing
        if (tid == 0) atomicOr(flags, kFlagSortWait);
        return;  // block-uniform, before any further barrier
    }
    if (t == 0 && owner) {
        // the previous pass (or the last pass of the previous sort) has ended
        const int prev = pass > 0 ? pass - 1 : passes - 1;
        ctl[prev * kBins + tid] = 0;
        if (tid == 0) ctl[kCtlTiles + prev] = 0;
    }
    const uint64_t tile = (uint64_t)t * kTile;
    const uint64_t rest = (uint64_t)n - tile;  // > 0: one block per tile
    const uint32_t tn = rest < (uint64_t)kTile ? (uint32_t)rest : (uint32_t)kTile;
    constexpr int kPassItems = kTile / kPassThreads;  // keys per lane
    const uint32_t wbase = w * (kPassItems * 64u);
    uint64_t kk[kPassItems];
    uint32_t vv[kPassItems], dg[kPassItems], rk[kPassItems];
#pragma unroll
    for (int r = 0; r < kPassItems; ++r) {
        const uint32_t j = wbase + (uint32_t)r * 64u + lane;
        kk[r] = j < tn ? keys[tile + j] : ~0ull;
        vv[r] = j < tn ? vals[tile + j] : 0u;
    }
    const uint64_t lt_mask = lanes_below();
#pragma unroll
    for (int r = 0; r < kPassItems; ++r) {
        const bool valid = wbase + (uint32_t)r * 64u + lane < tn;
        const uint32_t d = (uint32_t)(kk[r] >> shift) & (kBins - 1);
        dg[r] = d;
        const uint64_t peers = digit_peers(d, valid);
        const uint32_t rank = (uint32_t)__popcll(peers & lt_mask);
        // a wave's LDS accesses complete in order: the next round reads this write
        const uint32_t before = wcnt[w][d];
        rk[r] = before + rank;
        if (valid && rank == 0) wcnt[w][d] = before + (uint32_t)__popcll(peers);
        if (valid && has_next)
            atomicAdd(&next_hist[(uint32_t)(kk[r] >> (shift + kDigitBits)) & (kBins - 1)], 1u);
    }
    __syncthreads();
    uint32_t c = 0, gtot = 0;
    if (owner) {
        // per-wave counts of digit tid become offsets among the tile's digit-tid keys
#pragma unroll
        for (int k = 0; k < kPassWaves; ++k) {
            const uint32_t cnt = wcnt[k][tid];
            wcnt[k][tid] = c;
            c += cnt;
        }
        status_store(stat + (uint64_t)t * kBins + tid, (t == 0 ? kStatPrefix : kStatAgg) | c);
        stat_next[(uint64_t)t * kBins + tid] = 0;
        if (has_next && next_hist[tid]) atomicAdd(total + kBins + tid, next_hist[tid]);
        gtot = total[tid];
    }
    const uint32_t ex = digit_exclusive_scan(c, wsum[0]);
    const uint32_t goff = digit_exclusive_scan(gtot, wsum[1]);
    if (owner) {
        dbase[tid] = ex;
#pragma unroll
        for (int k = 0; k < kPassWaves; ++k) wcnt[k][tid] += ex;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kPassItems; ++r) {
        if (wbase + (uint32_t)r * 64u + lane < tn) {
            const uint32_t p = wcnt[w][dg[r]] + rk[r];
            lk[p] = kk[r];
            lv[p] = vv[r];
        }
    }
    if (owner) {
        uint32_t excl = 0;
        if (t > 0) {
            if (!look_back(stat, t, tid, &excl)) stuck = 1;
            // published even when stuck, so that later tiles do not wait as well
            status_store(stat + (uint64_t)t * kBins + tid, kStatPrefix | (excl + c));
        }
        gbase[tid] = goff + excl;
    }
    __syncthreads();
    if (stuck) {
        if (tid == 0) atomicOr(flags, kFlagSortWait);
        return;
    }
    for (uint32_t j = tid; j < tn; j += kPassThreads) {
        const uint64_t key = lk[j];
        const uint32_t d = (uint32_t)(key >> shift) & (kBins - 1);
        const uint32_t pos = gbase[d] + (j - dbase[d]);
        if (pos < n) {
            okeys[pos] = key;
            ovals[pos] = lv[j];
        }
    }
}

// ---- small and middling sorts ---------------------------------------------------
// A pass over a few tiles is all latency: of 9.2 us in the kernel (100,003 keys,
// 25 tiles of 4096) ranking takes 2.6 us, the look-back 1.9, two scans behind a
// load 2.1, a tile id 0.7, and a launch comes on top, seven times.  So up to
// kSortMergeMax keys are sorted otherwise: one launch in which every workgroup
// sorts a tile of up to 2048 keys in LDS, all passes (k_sort_tiles), then one
// launch per factor of eight that merges eight runs into one (k_merge_runs).
//
// A merged key's place is its own index plus, for each of the other seven runs,
// the number of keys there that come before it.  Equal keys keep the order of
// their runs, so the sort is stable.
//
// Whole sorts: 1024 keys 51 us in passes, 13.4 here; 100,003: 84 and 50; 262,144:
// 27 us less here; 400,000 and 524,288: within 3 us of each other; 1,048,576: 80 us
// more (a merge reads every key eight times over), hence the limit.
template <int kItems_>
__global__ void __launch_bounds__(1024) k_sort_tiles(
    const uint64_t *__restrict__ keys, const uint32_t *__restrict__ vals,
    uint64_t *__restrict__ okeys, uint32_t *__restrict__ ovals, uint32_t total, int passes) {
    constexpr uint32_t waves = 16;
    __shared__ uint32_t wcnt[waves][kBins];  // digit-d keys of wave w, then those of earlier waves
    __shared__ uint32_t dbase[kBins];
    __shared__ uint32_t ws[kBins / 64];
    __shared__ uint64_t lk[1024 * kItems_];
    __shared__ uint32_t lv[1024 * kItems_];
    const uint32_t tid = threadIdx.x, w = tid >> 6;
    const uint32_t j0 = w * (64u * kItems_) + lane_id();
    const uint32_t tile = blockIdx.x * (1024u * kItems_);
    const uint32_t n = min(total - tile, 1024u * kItems_);  // keys of this tile
    keys += tile;
    vals += tile;
    okeys += tile;
    ovals += tile;
    uint64_t kk[kItems_];
    uint32_t vv[kItems_], dg[kItems_], rk[kItems_];
#pragma unroll
    for (int r = 0; r < kItems_; ++r) {
        const uint32_t j = j0 + 64u * r;
        kk[r] = j < n ? keys[j] : ~0ull;
        vv[r] = j < n ? vals[j] : 0u;
    }
    const uint64_t lt_mask = lanes_below();
    for (int pass = 0; pass < passes; ++pass) {
        const int shift = kDigitBits * pass;
        for (uint32_t i = tid; i < waves * kBins; i += 1024) (&wcnt[0][0])[i] = 0;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kItems_; ++r) {
            const bool valid = j0 + 64u * r < n;
            const uint32_t d = (uint32_t)(kk[r] >> shift) & (kBins - 1);
            const uint64_t peers = digit_peers(d, valid);
            const uint32_t rank = (uint32_t)__popcll(peers & lt_mask);
            // a wave's LDS accesses complete in order: the next round reads this write
            const uint32_t before = wcnt[w][d];
            dg[r] = d;
            rk[r] = before + rank;
            if (valid && rank == 0) wcnt[w][d] = before + (uint32_t)__popcll(peers);
        }
        __syncthreads();
        uint32_t c = 0, inc = 0;
        if (tid < kBins) {
            uint32_t cnt[waves];
#pragma unroll
            for (uint32_t k = 0; k < waves; ++k) cnt[k] = wcnt[k][tid];
#pragma unroll
            for (uint32_t k = 0; k < waves; ++k) {
                wcnt[k][tid] = c;
                c += cnt[k];
            }
            inc = wave_inclusive_scan(c);
            if (lane_id() == 63) ws[w] = inc;
        }
        __syncthreads();
        if (tid < kBins) {
            uint32_t ex = inc - c;
#pragma unroll
            for (uint32_t k = 0; k < kBins / 64; ++k) ex += k < w ? ws[k] : 0u;
            dbase[tid] = ex;
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kItems_; ++r) {
            if (j0 + 64u * r < n) {
                const uint32_t p = dbase[dg[r]] + wcnt[w][dg[r]] + rk[r];
                lk[p] = kk[r];
                lv[p] = vv[r];
            }
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kItems_; ++r) {
            const uint32_t j = j0 + 64u * r;
            if (j < n) {
                kk[r] = lk[j];
                vv[r] = lv[j];
            }
        }
    }
#pragma unroll
    for (int r = 0; r < kItems_; ++r) {
        const uint32_t j = j0 + 64u * r;
        if (j < n) {
            okeys[j] = kk[r];
            ovals[j] = vv[r];
        }
    }
}

constexpr int kMergeThreads = 256;
constexpr uint32_t kMergeRuns = 8;
constexpr uint32_t kMergeLds = 4096;  // keys of the other runs held in LDS
// Does a key of run q come before key (of run own)?  Equal keys keep the order
// of their runs.
__device__ __forceinline__ bool merge_before(uint64_t other, uint32_t q, uint64_t key, uint32_t own) {
    return q < own ? other <= key : other < key;
}

// A workgroup places kMergeThreads consecutive keys of one run.  Its first and
// last key bound the places of all of them in each other run: a wave finds the
// bounds with 64 probes at a time (two or three dependent loads instead of a
// dozen).  The keys between the bounds, about kMergeThreads per run, then go to
// LDS, where every thread bisects.  If they are more than kMergeLds (a short last
// run, or runs of unlike ranges), every 2nd, 4th, ... goes there instead, and the
// last steps of the bisection read global memory.
// run: keys per sorted run (a power of two, a multiple of kMergeThreads); mask: the
// key bits that the runs are sorted by.
__global__ void __launch_bounds__(kMergeThreads) k_merge_runs(
    const uint64_t *__restrict__ keys, const uint32_t *__restrict__ vals,
    uint64_t *__restrict__ okeys, uint32_t *__restrict__ ovals, uint32_t n, uint32_t run,
    uint64_t mask) {
    constexpr uint32_t waves = kMergeThreads / 64, per = kMergeRuns / waves;
    __shared__ uint64_t win[kMergeLds];
    __shared__ uint32_t bound[2][kMergeRuns];
    const uint32_t t = threadIdx.x, lane = lane_id(), w = t >> 6;
    const uint32_t i0 = blockIdx.x * kMergeThreads;
    const uint32_t i1 = min(n, i0 + kMergeThreads) - 1;    // last key
    const uint32_t own = i0 / run;                          // this workgroup's run
    const uint32_t first = own / kMergeRuns * kMergeRuns;   // first run of its eight
    const uint32_t i = min(i0 + t, i1);
    const uint64_t full = keys[i], key = full & mask;
    const uint32_t val = vals[i];
    const uint64_t end_key[2] = {keys[i0] & mask, keys[i1] & mask};
    // the wave's runs, both ends: lo keys are known to come before, the next rem
    // are open
    uint32_t lo[2 * per], rem[2 * per];
#pragma unroll
    for (uint32_t k = 0; k < 2 * per; ++k) {
        const uint32_t q = first + w * per + (k >> 1);
        const uint64_t begin = (uint64_t)q * run;
        lo[k] = 0;
        rem[k] = q == own || begin >= n ? 0u : (uint32_t)min((uint64_t)run, n - begin);
    }
    for (;;) {
        bool open = false;
        uint64_t probe[2 * per];
        uint32_t stride[2 * per];
#pragma unroll
        for (uint32_t k = 0; k < 2 * per; ++k) {
            const uint64_t begin = (uint64_t)(first + w * per + (k >> 1)) * run;
            stride[k] = (rem[k] + 63) / 64;
            open |= rem[k] != 0;
            const uint32_t p = (lane + 1) * stride[k] - 1;  // unused if rem is 0
            probe[k] = rem[k] && p < rem[k] ? keys[begin + lo[k] + p] & mask : ~0ull;
        }
        if (!open) break;  // the same for the whole wave
#pragma unroll
        for (uint32_t k = 0; k < 2 * per; ++k) {
            const uint32_t q = first + w * per + (k >> 1);
            const bool in = rem[k] && (lane + 1) * stride[k] - 1 < rem[k];
            const uint32_t c =
                (uint32_t)__popcll(__ballot(in && merge_before(probe[k], q, end_key[k & 1], own)));
            const uint32_t done = c * stride[k];
            lo[k] += done;
            rem[k] = rem[k] ? min(stride[k] - 1, rem[k] - done) : 0u;
        }
    }
#pragma unroll
    for (uint32_t k = 0; k < 2 * per; ++k)
        if (lane == 0) bound[k & 1][w * per + (k >> 1)] = lo[k];
    __syncthreads();
    uint32_t lower[kMergeRuns], cnt[kMergeRuns], at[kMergeRuns + 1], most = 0;
#pragma unroll
    for (uint32_t q = 0; q < kMergeRuns; ++q) {
        lower[q] = bound[0][q];
        cnt[q] = bound[1][q] - lower[q];
        most = max(most, cnt[q]);
    }
    uint32_t thin = 0;  // LDS holds the last of every 2^thin keys
    for (;; ++thin) {
        at[0] = 0;
#pragma unroll
        for (uint32_t q = 0; q < kMergeRuns; ++q) at[q + 1] = at[q] + (cnt[q] >> thin);
        if (at[kMergeRuns] <= kMergeLds) break;
    }
    // key p (from 0) between run q's bounds
    const auto key_at = [&](uint32_t q, uint32_t p) {
        const uint64_t src = (uint64_t)(first + q) * run + lower[q] + p;
        return src < n ? keys[src] & mask : ~0ull;
    };
    constexpr int kAhead = 8;  // loads in flight per thread
    for (uint32_t j0 = t; j0 < at[kMergeRuns]; j0 += kAhead * kMergeThreads) {
        uint64_t v[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const uint32_t j = min(j0 + u * kMergeThreads, at[kMergeRuns] - 1);
            uint64_t src = 0;
#pragma unroll
            for (uint32_t q = 0; q < kMergeRuns; ++q)
                if (j >= at[q])
                    src = (uint64_t)(first + q) * run + lower[q] + ((j - at[q] + 1) << thin) - 1;
            v[u] = keys[src] & mask;
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u)
            if (j0 + u * kMergeThreads < at[kMergeRuns]) win[j0 + u * kMergeThreads] = v[u];
    }
    __syncthreads();
    uint32_t before[kMergeRuns];
#pragma unroll
    for (uint32_t q = 0; q < kMergeRuns; ++q) before[q] = 0;
    const auto bisect = [&](uint32_t step, uint32_t stop, auto load) {
        for (; step >= stop; step >>= 1) {
            uint64_t v[kMergeRuns];
#pragma unroll
            for (uint32_t q = 0; q < kMergeRuns; ++q) v[q] = load(q, before[q] + step - 1);
#pragma unroll
            for (uint32_t q = 0; q < kMergeRuns; ++q)
                if (before[q] + step <= cnt[q] && merge_before(v[q], first + q, key, own))
                    before[q] += step;
        }
        return step;
    };
    uint32_t step = most ? 1u << (31 - __clz((int)most)) : 0u;
    if (step >> thin)
        step = bisect(step, 1u << thin, [&](uint32_t q, uint32_t p) {
            return win[min(at[q] + (p >> thin), kMergeLds - 1)];
        });
    if (thin) bisect(step, 1u, key_at);
    if (i0 + t > i1) return;
    uint32_t pos = first * run + (i - own * run);
#pragma unroll
    for (uint32_t q = 0; q < kMergeRuns; ++q) pos += lower[q] + before[q];
    okeys[pos] = full;
    ovals[pos] = val;
}

}  // namespace

uint32_t scan_scratch_words(uint32_t n) { return ceil_div(n ? n : 1, kScanTile) + 1; }

void scan_exclusive_u32(const uint32_t *in, uint32_t *out, uint32_t n, uint32_t *total_dev,
                        uint32_t *scratch, uint32_t scratch_cap, hipStream_t s) {
    if (n == 0) return;
    const uint32_t nb = ceil_div(n, kScanTile);
    if (nb > scratch_cap) return;  // caller sized the scratch with scan_scratch_words
    hipLaunchKernelGGL(k_scan_reduce, dim3(nb), dim3(kThreads), 0, s, in, n, scratch);
    hipLaunchKernelGGL(k_scan_parts, dim3(1), dim3(kThreads), 0, s, scratch, nb, total_dev);
    hipLaunchKernelGGL(k_scan_down, dim3(nb), dim3(kThreads), 0, s, in, out, n,
                       (const uint32_t *)scratch);
}

bool scan_parts_if_many(uint32_t *part, uint32_t nparts, hipStream_t s) {
    if (nparts <= kScanPartsInline) return false;
    hipLaunchKernelGGL(k_scan_parts, dim3(1), dim3(kThreads), 0, s, part, nparts,
                       (uint32_t *)nullptr);
    return true;
}

// tiles of a sort of n keys at the smaller tile size (the most control words)
uint32_t radix_blocks_for(uint32_t n) { return ceil_div(n ? n : 1, kRadixTile); }

uint32_t radix_ctl_words(uint32_t n) { return kCtlStatus + 2u * kBins * radix_blocks_for(n); }

// Keys per tile of a sort of n keys.  Larger tiles for large sorts: half the
// look-back chain and longer digit runs in the scatter, once there are enough
// tiles to fill the device.  A CU holds one tile of either larger size, so time
// goes with (rounds of tiles) x (keys per tile): 2,110,000 keys are 258 tiles of
// 8192, a second round for two of them (41 us a pass), and 207 of 10,240 (29 us);
// 4,194,304 are two rounds of either, and 8192 is the smaller.
static uint32_t radix_tile(uint32_t n) {
    if (n < kRadixBigMin) return kRadixTile;
    const auto cost = [&](uint32_t tile) {
        return (uint64_t)ceil_div(ceil_div(n, tile), kCus) * tile;
    };
    return cost(kRadixTileWide) < cost(kRadixTileBig) ? kRadixTileWide : kRadixTileBig;
}

RadixCount radix_count_args(uint32_t n, uint32_t *ctl) {
    if (n <= kSortMergeMax || n >= kStatAgg) return RadixCount{nullptr, nullptr, 0};
    return RadixCount{ctl, ctl + kCtlStatus, (uint64_t)kBins * ceil_div(n, radix_tile(n))};
}

SortEnd radix_sort_u64_u32(uint64_t *keys, uint32_t *vals, uint64_t *keys_alt,
                           uint32_t *vals_alt, uint32_t n, int bits, uint32_t *ctl,
                           uint32_t *flags, bool counted, hipStream_t s) {
    if (n >= kStatAgg || bits <= 0 || bits > kDigitBits * kMaxPasses) {
        // counts of 2^30 keys and more do not fit the status words: nothing
        // is sorted, and the caller's status word says so
        hipLaunchKernelGGL(k_raise_flag, dim3(1), dim3(64), 0, s, flags, kFlagSortSize);
        return SortEnd::kRejected;
    }
    if (n <= 1) return SortEnd::kInPlace;
    const int passes = std::max((bits + kDigitBits - 1) / kDigitBits, kMinPasses);
    uint64_t *ka = keys, *kb = keys_alt;
    uint32_t *va = vals, *vb = vals_alt;
    if (n <= kSortMergeMax) {
        const uint32_t tile = n <= 1024 ? 1024 : 2048;
        hipLaunchKernelGGL(n <= 1024 ? k_sort_tiles<1> : k_sort_tiles<2>, dim3(ceil_div(n, tile)),
                           dim3(1024), 0, s, (const uint64_t *)ka, (const uint32_t *)va, kb, vb, n,
                           passes);
        std::swap(ka, kb);
        std::swap(va, vb);
        const uint64_t mask = ~0ull >> (64 - std::min(64, kDigitBits * passes));
        for (uint32_t run = tile; run < n; run *= kMergeRuns) {
            hipLaunchKernelGGL(k_merge_runs, dim3(ceil_div(n, kMergeThreads)), dim3(kMergeThreads),
                               0, s, (const uint64_t *)ka, (const uint32_t *)va, kb, vb, n, run, mask);
            std::swap(ka, kb);
            std::swap(va, vb);
        }
        return ka == keys ? SortEnd::kInPlace : SortEnd::kInAlt;
    }
    const uint32_t tile = radix_tile(n), nb = ceil_div(n, tile);
    const auto pass = tile == (uint32_t)kRadixTile      ? k_radix_pass<kRadixTile>
                      : tile == (uint32_t)kRadixTileBig ? k_radix_pass<kRadixTileBig>
                                                        : k_radix_pass<kRadixTileWide>;
    if (!counted)
        hipLaunchKernelGGL(k_radix_count, dim3(std::min(nb, kCountBlocks)), dim3(kCountThreads), 0,
                           s, (const uint64_t *)keys, n, ctl, ctl + kCtlStatus,
                           (uint64_t)kBins * nb);
    for (int p = 0; p < passes; ++p) {
        hipLaunchKernelGGL(pass, dim3(nb), dim3(kPassThreads), 0, s, (const uint64_t *)ka,
                           (const uint32_t *)va, kb, vb, n, p, passes, ctl, nb, flags);
        std::swap(ka, kb);
        std::swap(va, vb);
    }
    // an odd count ends in the scratch buffers
    return (passes & 1) ? SortEnd::kInAlt : SortEnd::kInPlace;
}

}  // namespace nb
