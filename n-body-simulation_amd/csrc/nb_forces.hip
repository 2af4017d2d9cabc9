// nb_forces.hip -- direct-sum and Barnes-Hut force kernels for gfx950.
//
// FP64 kernels reproduce the reference's arithmetic operation for operation
// (this file is compiled with -ffp-contract=off, and sycl::rsqrt is evaluated
// as 1.0/sqrt(x), two correctly rounded IEEE operations):
//   k_direct_f64   NaiveAlgorithm.cpp:299-352 (sum over j in index order)
//   k_bh_exact_*   BarnesHutAlgorithm.cpp:319-393 (per-body traversal, same
//                  visit order, same opening test)
// FP32 kernels do the pair arithmetic in FP32 (fmaf, v_rsq_f32) and fold the
// FP32 partial of every tile into FP64 accumulators:
//   k_direct_f32c  sources staged in LDS per wave, two targets per lane, split j
//   k_bh_group     one wavefront per group (an octree cell of <= 64 bodies);
//                  a cell is opened if any body of the group needs it; lanes
//                  test 8 sibling sets at a time and accepted cells/bodies are
//                  batched in LDS and evaluated 64 at a time.
#include <algorithm>
#include <cmath>

#include "nb_mlp.h"

namespace nb {
namespace {

__device__ inline void raise_flag(TreeHdr *h, uint32_t f) { atomicOr(&h->status, f); }

constexpr uint32_t kXcds = 8;  // XCDs of an MI355X; workgroups are dealt round-robin
constexpr uint32_t kCus = 256;  // CUs of an MI355X

// A value every lane of the wave holds alike, made visibly uniform (SGPR).
// The walks below are wave-collective (ballots, shuffles, one LDS list per
// wave): every branch that steers them must be uniform to the compiler, or
// control-flow structurisation may let parts of the wave run different
// iterations with partial exec masks.
__device__ inline uint32_t wave_uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

// ---------------------------------------------------------------------------
// FP64 direct sum, reference order.  The sum over j = 0..n-1 of a target must
// run in that order to be bit-exact, but only its three additions per pair
// are sequential; the pair terms m_j (r_ij den_ij), with their IEEE division
// and square root, are not.  A workgroup of sixteen waves owns T targets; for
// each chunk of sources its waves compute the terms into one of two LDS tiles
// while the first 3 T threads (component d of target t in thread d T + t) add
// the previous tile in source order.
//  - T = 64: a wave computes the terms of one source at a time, which it reads
//    through the scalar cache (staging the sources in LDS loads it with two
//    more reads per term than the five that the terms need).
//  - T = 16, where 64 targets per workgroup leave CUs idle: four sources at a
//    time; wave 0 only adds, since the chain of additions bounds a workgroup.
// The additions stand before the terms in a chunk, ahead of the other waves on
// their SIMDs (s_setprio); a wave's terms are interleaved, with one test for
// all that the IEEE sequences need no range handling.  16,384 bodies: 0.52 ms
// with the additions last, sources staged in LDS and one term at a time; 0.45
// without; 0.42 now that the reciprocal needs no v_rcp_f64, 244 cycles at 2.4 GHz
// per 64 pairs where the 31 FP64 operations, the quarter-rate estimate and three
// additions of a pair issue in about 188.
// 700 bodies 0.026 -> 0.011, 5001 0.162 -> 0.082, 8192 0.262 -> 0.133, 20,001
// 1.26 -> 0.76 ms.  T = 32 (two sources at a time) was slower than the better
// of the two at every size.
constexpr int kF64Waves = 16;
constexpr int kF64Threads = 64 * kF64Waves;
template <int T>
struct DirectF64 {
    static constexpr int kSub = 64 / T;             // sources per wave and step
    static constexpr int kPer = T == 64 ? 3 : 1;    // steps per chunk: its terms interleave
    static constexpr int kFirst = T == 64 ? 0 : 1;  // first wave that computes terms
    static constexpr int kChunk = (kF64Waves - kFirst) * kSub * kPer;  // sources per tile
    static constexpr int kTile = kChunk * T + (T < 64 ? T : 0);        // rows in other banks
    static constexpr uint32_t kAdders = (3 * T + 63) / 64;  // waves
};
constexpr int kF64Ahead = 8;  // an adder's LDS reads in flight ahead of its ordered additions

// Returns, in thread d T + t (d < 3), component d of the sum over j in order
// of m_j (r_ij den_ij) for target t, whose position (px, py, pz) every thread
// with threadIdx.x % T == t passes.
template <int T>
__device__ __forceinline__ double direct_f64_body(uint32_t n, const double *__restrict__ x,
                                                  const double *__restrict__ y,
                                                  const double *__restrict__ z,
                                                  const double *__restrict__ m, double eps2,
                                                  double px, double py, double pz) {
    using K = DirectF64<T>;
    constexpr int P = K::kPer, C = K::kChunk;
    __shared__ double term[2][3][K::kTile];
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t t = lane % T, sub = lane / T;
    const bool adds = w < K::kAdders, computes = w >= (uint32_t)K::kFirst;
    const uint32_t comp = T == 64 ? min(w, 2u) : min(sub, 2u);
    double acc = 0;
    uint32_t pending = 0;  // sources in the tile the adders still have to add
    int buf = 0;
    auto add_tile = [&](int b, uint32_t cnt) {
        const double *own = &term[b][comp][t];
        if (cnt == (uint32_t)C) {
            double v[2][kF64Ahead];
#pragma unroll
            for (int u = 0; u < kF64Ahead; ++u) v[0][u] = own[u * T];
#pragma unroll
            for (int jj = 0; jj < C; jj += kF64Ahead) {
                const int c = (jj / kF64Ahead) & 1;
#pragma unroll
                for (int u = 0; u < kF64Ahead; ++u)
                    if (jj + kF64Ahead + u < C) v[c ^ 1][u] = own[(jj + kF64Ahead + u) * T];
#pragma unroll
                for (int u = 0; u < kF64Ahead; ++u)
                    if (jj + u < C) acc += v[c][u];
            }
        } else {
            for (uint32_t jj = 0; jj < cnt; ++jj) acc += own[jj * T];
        }
    };
    // a computing wave's sources of a chunk: (w - kFirst) kPer kSub + u kSub + sub
    const uint32_t own0 = (w - (uint32_t)K::kFirst) * (P * K::kSub) + sub;
    double sx[P], sy[P], sz[P], sm[P];
    auto load = [&](uint32_t c) {
#pragma unroll
        for (int u = 0; u < P; ++u) {
            const uint32_t j = min(c + own0 + u * K::kSub, n - 1);
            sx[u] = x[j];
            sy[u] = y[j];
            sz[u] = z[j];
            sm[u] = m[j];
        }
    };
    if (computes) load(0);
    for (uint32_t c = 0; c < n; c += C) {
        // the adders first, ahead of the terms of the other waves on their SIMDs
        if (adds && pending) {
            __builtin_amdgcn_s_setprio(3);
            add_tile(buf ^ 1, pending);
            __builtin_amdgcn_s_setprio(0);
        }
        if (computes) {
            double r_x[P], r_y[P], r_z[P], den[P], m_j[P];
            bool in_range = true;
            uint32_t low = 0;  // one test of the low words: a test each took 0.05 ms more
#pragma unroll
            for (int u = 0; u < P; ++u) {
                r_x[u] = sx[u] - px;
                r_y[u] = sy[u] - py;
                r_z[u] = sz[u] - pz;
                m_j[u] = sm[u];
                den[u] = (r_x[u] * r_x[u]) + (r_y[u] * r_y[u]) + (r_z[u] * r_z[u]) + eps2;
                den[u] = den[u] * den[u] * den[u];
                in_range = in_range && inv_sqrt_exponent_ok(den[u]);
                low = max(low, (uint32_t)__double2loint(den[u]));
            }
            load(c + C);  // back before the barrier waits for it
            if (in_range && low < kRootOfOnes) {
#pragma unroll
                for (int u = 0; u < P; ++u) den[u] = inv_sqrt_core(den[u]);
            } else {
                for (int u = 0; u < P; ++u) den[u] = 1.0 / sqrt(den[u]);
            }
#pragma unroll
            for (int u = 0; u < P; ++u) {
                const uint32_t k = (own0 + u * K::kSub) * T + t;
                term[buf][0][k] = m_j[u] * (r_x[u] * den[u]);
                term[buf][1][k] = m_j[u] * (r_y[u] * den[u]);
                term[buf][2][k] = m_j[u] * (r_z[u] * den[u]);
            }
        }
        __syncthreads();
        pending = min((uint32_t)C, n - c);
        buf ^= 1;
    }
    if (adds && pending) add_tile(buf ^ 1, pending);
    return acc;
}

// ids: the targets' body indices, or null for targets 0 .. nt - 1
template <int T>
__global__ void __launch_bounds__(kF64Threads) k_direct_f64(
    uint32_t n, const double *__restrict__ x, const double *__restrict__ y,
    const double *__restrict__ z, const double *__restrict__ m, double G, double eps2,
    uint32_t nt, const uint32_t *__restrict__ ids, double *ax, double *ay, double *az) {
    const uint32_t k = blockIdx.x * T + threadIdx.x % T;
    const bool valid = k < nt;
    const uint32_t i = !valid ? 0u : (ids ? ids[k] : k);
    const double acc = direct_f64_body<T>(n, x, y, z, m, eps2, x[i], y[i], z[i]);
    const uint32_t d = threadIdx.x / T;
    if (valid && d < 3) (d == 0 ? ax : (d == 1 ? ay : az))[k] = acc * G;
}

// ---------------------------------------------------------------------------
// Split direct sums: FP32 pairs with FP64 accumulation (k_direct_f32c), and
// FP64 pairs with a corrected v_rsq_f64 (k_direct_f64f).
//
// grid.x: tiles of 64 targets per lane's target (the same for all waves of a
// block); grid.y: source splits, each a contiguous source range.  A block's
// waves share the range: each stages kSplitTile sources of its own at a time in
// LDS, converted from the FP64 state arrays on the way, with the next stage's
// loads in flight, and no barrier until the waves' sums are added at the end.
// With one split a block writes its targets' sums; with more it stores partial
// sums and k_split_reduce adds them in split order 0, 1, ..., so results do not
// depend on block timing.
constexpr int kSplitWaves = 4;
constexpr int kSplitThreads = 64 * kSplitWaves;
constexpr uint32_t kSplitTile = 64;  // sources per stage of one wave
constexpr int kF32cRun = 4;          // stages per FP32 sum
constexpr int kF64fPerLane = 2;      // targets per lane: each LDS read feeds two pairs
// Partial sums of a launch, at most (3 * 8 bytes each: 24 MiB).  A SIMD serves
// its oldest waves first, so the waves resident at the end finish one after the
// other with ever fewer to overlap: more blocks than fit at once (8 per CU)
// keep it filled.
constexpr uint32_t kSplitPartials = 1u << 20;
// Pairs per interleaved step: FP32 four in 53 VGPRs, eight waves per SIMD (eight
// pairs: 70 VGPRs and within 2 %); FP64 eight in 124 VGPRs, four waves (four
// pairs within 1 %).
constexpr int kF32cPairs = 4;
constexpr int kF64fPairs = 8;

// v_rsq_f32 with an s_nop on each side.  With two or more waves on a SIMD, two
// waves' FP32 instructions issue at once (2.4 cycles at 2.4 GHz per wave
// instruction instead of 4.2), but a v_rsq_f32 next to other vector
// instructions ends that for the instructions around it as well: one pair (12
// instructions and the v_rsq_f32) takes 53-57 cycles per 64 pairs, and 36-38
// with the two wait states.  The same instruction, so the same bits.
__device__ __forceinline__ float rsq_f32(float v) {
    float y;
    asm("s_nop 0\n\tv_rsq_f32 %0, %1\n\ts_nop 0" : "=v"(y) : "v"(v));
    return y;
}

// Four independent ones, one pair of wait states around them all.
__device__ __forceinline__ void rsq4_f32(float (&v)[4]) {
    asm("s_nop 0\n\tv_rsq_f32 %0, %0\n\tv_rsq_f32 %1, %1\n\tv_rsq_f32 %2, %2\n\t"
        "v_rsq_f32 %3, %3\n\ts_nop 0"
        : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]));
}

__device__ inline void pair_f32(const float4 s, float px, float py, float pz, float eps2,
                                float &fx, float &fy, float &fz) {
    const float dx = s.x - px, dy = s.y - py, dz = s.z - pz;
    const float r2 = fmaf(dx, dx, fmaf(dy, dy, fmaf(dz, dz, eps2)));
    const float inv = __builtin_amdgcn_rsqf(r2);
    const float f = (s.w * inv) * (inv * inv);
    fx = fmaf(f, dx, fx);
    fy = fmaf(f, dy, fy);
    fz = fmaf(f, dz, fz);
}

// w v^(-3/2) in FP64 from the hardware estimate y = v_rsq_f64(v), whose
// relative error is near 1e-8 (single-precision accuracy): with y2 = y^2 and
// e = 1 - v y2 (one fused multiply-add, so e is exact to the last bits),
// v^(-3/2) = y^3 (1 - e)^(-3/2) = y^3 (1 + 3e/2 + 15e^2/8 + ...).  The
// correction to second order in e leaves a truncation error near
// 35e^3/16 ~ 1e-23, below FP64 rounding (a Newton step, first order in e,
// would leave ~1e-14).  The rounding of y2 enters the factor y2 and, with
// weight -3/2, e, so half of it remains.  Seven operations after the estimate.
// Checked against long-double closed forms in the GPU tests.
__device__ inline double rsqrt3_f64(double w, double v) {
    const double y = __builtin_amdgcn_rsq(v);
    const double y2 = y * y;
    const double e = fma(-v, y2, 1.0);
    const double t = (w * y) * y2;
    return fma(t * e, fma(e, 1.875, 1.5), t);
}

// The end of a split direct sum: adds the waves' sums in wave order; with one
// split the block writes scale * sums, with more it stores its partial sums at
// partial[split][3][n] for k_split_reduce.
template <int PL>
__device__ __forceinline__ void split_finish(uint32_t n, double scale, const double (&sx)[PL],
                                             const double (&sy)[PL], const double (&sz)[PL],
                                             double *comb, double *partial, double *out_x,
                                             double *out_y, double *out_z) {
    constexpr uint32_t kTargets = 64 * PL;
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
    __syncthreads();  // comb lies over the waves' stages
#pragma unroll
    for (int q = 0; q < PL; ++q) {
        double *c = comb + (w * 3) * kTargets + q * 64 + lane;
        c[0] = sx[q];
        c[kTargets] = sy[q];
        c[2 * kTargets] = sz[q];
    }
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < 3 * kTargets; k += kSplitThreads) {
        const uint32_t d = k / kTargets, t = k % kTargets;
        double v = comb[k];
#pragma unroll
        for (int o = 1; o < kSplitWaves; ++o) v += comb[(o * 3) * kTargets + k];
        const uint64_t i = (uint64_t)blockIdx.x * kTargets + t;
        if (i >= n) continue;
        if (gridDim.y == 1) (d == 0 ? out_x : (d == 1 ? out_y : out_z))[i] = v * scale;
        else partial[((uint64_t)blockIdx.y * 3ull + d) * n + i] = v;
    }
}

// out = scale * (sum over splits 0, 1, ... in that order) of the partial
// sums; blockIdx.y is the component.
__global__ void __launch_bounds__(kSplitThreads) k_split_reduce(uint32_t n, uint32_t splits,
                                                                double scale,
                                                                const double *__restrict__ partial,
                                                                double *out_x, double *out_y,
                                                                double *out_z) {
    const uint32_t i = blockIdx.x * kSplitThreads + threadIdx.x;
    if (i >= n) return;
    const double *__restrict__ p = partial + (uint64_t)blockIdx.y * n + i;
    const uint64_t stride = 3ull * n;
    double o = 0;
    // eight splits' loads in flight before their (ordered) additions
    constexpr uint32_t kAhead = 8;
    uint32_t sp = 0;
    for (; sp + kAhead <= splits; sp += kAhead) {
        double v[kAhead];
#pragma unroll
        for (uint32_t u = 0; u < kAhead; ++u) v[u] = p[(sp + u) * stride];
#pragma unroll
        for (uint32_t u = 0; u < kAhead; ++u) o += v[u];
    }
    for (; sp < splits; ++sp) o += p[sp * stride];
    (blockIdx.y == 0 ? out_x : (blockIdx.y == 1 ? out_y : out_z))[i] = o * scale;
}

// One wave's walk over its share of the block's sources [j0, j1): runs of kRun
// stages of kSplitTile sources, the first at j0 + w kRun kSplitTile and
// kSplitWaves runs apart.  use(cnt) gets a stage of cnt sources, padded to
// kSplitTile with sources of zero mass; end_run() follows a run's last stage;
// pack converts one source.
template <int kRun, typename T4, typename Pack, typename Use, typename EndRun>
__device__ __forceinline__ void split_stages(uint32_t j0, uint32_t j1,
                                             const double *__restrict__ x,
                                             const double *__restrict__ y,
                                             const double *__restrict__ z,
                                             const double *__restrict__ m, T4 *stage, T4 pad,
                                             Pack pack, Use use, EndRun end_run) {
    // uniform: the lanes of a wave hand each other their stage in these loops
    const uint32_t lane = threadIdx.x & 63u, w = wave_uniform(threadIdx.x >> 6);
    constexpr uint32_t run = kRun * kSplitTile;
    double sx = 0, sy = 0, sz = 0, sm = 0;
    auto load = [&](uint32_t j) {
        if (j < j1) {
            sx = x[j];
            sy = y[j];
            sz = z[j];
            sm = m[j];
        }
    };
    uint32_t k = j0 + w * run, end = k + run;
    load(k + lane);
    while (k < j1) {
        // by component: a select between two structures goes through scratch memory
        const T4 p = pack(sx, sy, sz, sm);
        const bool real = k + lane < j1;
        T4 s;
        s.x = real ? p.x : pad.x;
        s.y = real ? p.y : pad.y;
        s.z = real ? p.z : pad.z;
        s.w = real ? p.w : pad.w;
        stage[lane] = s;
        const uint32_t cnt = min(kSplitTile, j1 - k);
        k += kSplitTile;
        const bool last = k == end || k >= j1;
        if (k == end) {
            k += (kSplitWaves - 1) * run;
            end = k + run;
        }
        load(k + lane);  // the next stage's, while this one is used
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        use(cnt);
        if (last) end_run();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

// FP32 pairs on absolute FP32 positions with G*m as the source weight; the
// FP32 sums of every 256 sources (kF32cRun stages, from a multiple of 256) are
// folded into FP64.  Bound by vector issue: 50,021 bodies in 0.656 ms (0.773
// with 256-source stages shared by a block and no wait states around the
// v_rsq_f32), 41 cycles at 2.4 GHz per 64 pairs, where a loop of such pairs alone takes 36-38.
// PL: targets per lane, 1 for small sums (twice the waves).
template <int PL>
__global__ void __launch_bounds__(kSplitThreads) __attribute__((amdgpu_waves_per_eu(8)))
k_direct_f32c(uint32_t n, const double *__restrict__ x, const double *__restrict__ y,
              const double *__restrict__ z, const double *__restrict__ m, double G, float eps2,
              uint32_t chunk, double *partial, double *ax_out, double *ay_out, double *az_out) {
    __shared__ double4 lds[kSplitWaves * 3 * 16 * PL];  // the stages, then the waves' sums
    static_assert(sizeof(float4) * kSplitTile * kSplitWaves <= sizeof(lds), "stages fit");
    const uint32_t lane = threadIdx.x & 63u;
    float4 *stage = table_as<float4>(lds) + (threadIdx.x >> 6) * kSplitTile;
    asm("" : "+v"(eps2));  // a scalar operand would end the double issue
    float px[PL], py[PL], pz[PL], fx[PL], fy[PL], fz[PL];
    double ax[PL], ay[PL], az[PL];
#pragma unroll
    for (int q = 0; q < PL; ++q) {
        const uint32_t i = blockIdx.x * 64 * PL + q * 64 + lane;
        const uint32_t ii = i < n ? i : n - 1;
        px[q] = (float)x[ii];
        py[q] = (float)y[ii];
        pz[q] = (float)z[ii];
        ax[q] = ay[q] = az[q] = 0.0;
        fx[q] = fy[q] = fz[q] = 0.f;
    }
    const uint32_t j0 = blockIdx.y * chunk;
    const uint32_t j1 = min(n, j0 + chunk);
    split_stages<kF32cRun, float4>(
        j0, j1, x, y, z, m, stage, make_float4(1e30f, 0.f, 0.f, 0.f),
        [&](double sx, double sy, double sz, double sm) {
            return make_float4((float)sx, (float)sy, (float)sz, (float)(G * sm));
        },
        [&](uint32_t cnt) {
            // kF32cPairs pairs at a time, stage by stage across the pairs, so
            // that neighbouring instructions are independent; the same
            // operations per pair as pair_f32
            constexpr int kSources = kF32cPairs / PL;
            static_assert(kSplitTile % kSources == 0, "whole steps per stage");
            for (uint32_t jj = 0; jj < cnt; jj += kSources) {
                float dx[kF32cPairs], dy[kF32cPairs], dz[kF32cPairs], inv[kF32cPairs],
                    wt[kF32cPairs];
#pragma unroll
                for (int u = 0; u < kSources; ++u) {
                    const float4 sj = stage[jj + u];
#pragma unroll
                    for (int q = 0; q < PL; ++q) {
                        const int p = u * PL + q;
                        dx[p] = sj.x - px[q];
                        dy[p] = sj.y - py[q];
                        dz[p] = sj.z - pz[q];
                        wt[p] = sj.w;
                        inv[p] = fmaf(dx[p], dx[p], fmaf(dy[p], dy[p], fmaf(dz[p], dz[p], eps2)));
                    }
                }
#pragma unroll
                for (int p = 0; p < kF32cPairs; ++p) inv[p] = rsq_f32(inv[p]);
#pragma unroll
                for (int u = 0; u < kSources; ++u)
#pragma unroll
                    for (int q = 0; q < PL; ++q) {
                        const int p = u * PL + q;
                        const float f = (wt[p] * inv[p]) * (inv[p] * inv[p]);
                        fx[q] = fmaf(f, dx[p], fx[q]);
                        fy[q] = fmaf(f, dy[p], fy[q]);
                        fz[q] = fmaf(f, dz[p], fz[q]);
                    }
            }
        },
        [&] {
#pragma unroll
            for (int q = 0; q < PL; ++q) {
                ax[q] += (double)fx[q];
                ay[q] += (double)fy[q];
                az[q] += (double)fz[q];
                fx[q] = fy[q] = fz[q] = 0.f;
            }
        });
    split_finish<PL>(n, 1.0, ax, ay, az, table_as<double>(lds), partial, ax_out, ay_out, az_out);
}

// FP64 pairs (the reference's formula, NaiveAlgorithm.cpp:318-351, with
// m r^-3 from rsqrt3_f64 and fused multiply-adds); G is applied to the sum, as
// in the reference (:348-351).  Bound by vector issue: 16 full-rate FP64
// instructions, the quarter-rate estimate and two moves (the compiler puts the
// addend 1.5 where its fused multiply-add leaves the result), about 88 of the 96
// cycles per 64 pairs that 16,384 bodies take; those in 0.165 ms (0.172-0.176
// before), 3001 in 0.0145 ms (0.052).
__global__ void __launch_bounds__(kSplitThreads) k_direct_f64f(
    uint32_t n, const double *__restrict__ x, const double *__restrict__ y,
    const double *__restrict__ z, const double *__restrict__ m, double G, double eps2,
    uint32_t chunk, double *partial, double *ax_out, double *ay_out, double *az_out) {
    __shared__ double4 lds[kSplitWaves * 3 * 16 * kF64fPerLane];  // the stages, then the waves' sums
    static_assert(sizeof(double4) * kSplitTile * kSplitWaves <= sizeof(lds), "stages fit");
    const uint32_t lane = threadIdx.x & 63u;
    double4 *stage = lds + (threadIdx.x >> 6) * kSplitTile;
    double px[kF64fPerLane], py[kF64fPerLane], pz[kF64fPerLane];
    double ax[kF64fPerLane], ay[kF64fPerLane], az[kF64fPerLane];
#pragma unroll
    for (int q = 0; q < kF64fPerLane; ++q) {
        const uint32_t i = blockIdx.x * 64 * kF64fPerLane + q * 64 + lane;
        const uint32_t ii = i < n ? i : n - 1;
        px[q] = x[ii];
        py[q] = y[ii];
        pz[q] = z[ii];
        ax[q] = ay[q] = az[q] = 0.0;
    }
    const uint32_t j0 = blockIdx.y * chunk;
    const uint32_t j1 = min(n, j0 + chunk);
    split_stages<1, double4>(
        j0, j1, x, y, z, m, stage, make_double4(0x1.3p+400, 0.0, 0.0, 0.0),
        [&](double sx, double sy, double sz, double sm) { return make_double4(sx, sy, sz, sm); },
        [&](uint32_t cnt) {
            // stage by stage across the pairs: the compiler otherwise runs each
            // pair's chain (the estimate, its correction, the force) to the end
            // before the next pair starts
            constexpr int kSources = kF64fPairs / kF64fPerLane;
            static_assert(kSplitTile % kSources == 0, "whole steps per stage");
            for (uint32_t jj = 0; jj < cnt; jj += kSources) {
                double dx[kF64fPairs], dy[kF64fPairs], dz[kF64fPairs], r2[kF64fPairs], f[kF64fPairs];
#pragma unroll
                for (int u = 0; u < kSources; ++u) {
                    const double4 sj = stage[jj + u];
#pragma unroll
                    for (int q = 0; q < kF64fPerLane; ++q) {
                        const int p = u * kF64fPerLane + q;
                        dx[p] = sj.x - px[q];
                        dy[p] = sj.y - py[q];
                        dz[p] = sj.z - pz[q];
                        f[p] = sj.w;
                        r2[p] = fma(dx[p], dx[p], fma(dy[p], dy[p], fma(dz[p], dz[p], eps2)));
                    }
                }
#pragma unroll
                for (int p = 0; p < kF64fPairs; ++p) f[p] = rsqrt3_f64(f[p], r2[p]);
#pragma unroll
                for (int u = 0; u < kSources; ++u)
#pragma unroll
                    for (int q = 0; q < kF64fPerLane; ++q) {
                        const int p = u * kF64fPerLane + q;
                        ax[q] = fma(f[p], dx[p], ax[q]);
                        ay[q] = fma(f[p], dy[p], ay[q]);
                        az[q] = fma(f[p], dz[p], az[q]);
                    }
            }
        },
        [] {});
    split_finish<kF64fPerLane>(n, G, ax, ay, az, table_as<double>(lds), partial, ax_out, ay_out, az_out);
}

// ---------------------------------------------------------------------------
// Reference-semantics Barnes-Hut traversal (FP64).  The reference walks the tree
// per body with a stack: children are pushed in digit order 5,7,4,6,1,3,0,2
// (BarnesHutAlgorithm.cpp:370-385) and popped from the end, a depth-first
// pre-order with the siblings in the order 2,0,3,1,6,4,7,5.
// Two kernels walk it in that order, one for small systems and one for large
// ones (launch_bh_exact chooses).  A stack per lane, one body per lane, loaded
// each node's record from 64 places and ran the branch of the term for the few
// lanes that needed it: 1M-body disk at theta 0.5 10.4 ms, now 5.5 (waves); 1024
// bodies 0.52 ms, now 0.107; 30,001 (Plummer, theta 1.05) 0.47, now 0.174
// (teams).
//
// k_bh_exact_team: a team of eight lanes walks the tree for one body and opens a
// cell in one step: lane p loads and tests the child at visit position p.
// Accepted nodes go to the team's list in LDS in the reference's order (those
// behind an opened sibling wait on a stack, as a mask of the cell's children),
// and once a list is nearly full, the lanes compute the terms of eight list
// entries at a time and three lanes add them, one component each, in list order:
// the reference's sum, bit for bit.  A walk takes one round trip to memory per
// opened cell; what bounds it is that latency and, with more bodies than fit at
// once, the bookkeeping of a step.
constexpr int kExactWaves = 4;  // waves per workgroup
constexpr int kExactThreads = 64 * kExactWaves;
constexpr uint32_t kTeams = 8;  // bodies per wave
constexpr uint32_t kTeamList = 40;  // entries; flushed above kTeamList - 16: a step adds up to 16
constexpr uint32_t kTeamStack = kMaxDepth + 2;  // one entry per level

struct TeamLds {
    uint32_t cell[kTeamStack][kTeams];   // cell with children left
    uint32_t ref[kTeamStack][kTeams];    // its next child to open
    uint32_t masks[kTeamStack][kTeams];  // level << 16 | children to open << 8 | to add
    uint32_t list[kTeams][kTeamList];    // node ids
    double term[kTeams][3][8];
};

// the slot of a cell's child at visit position p
__device__ inline uint32_t visit_digit(uint32_t p) { return (0x57461302u >> (4u * p)) & 7u; }

// Workgroup b runs on XCD b mod 8: give each XCD a contiguous run of blocks, so
// that its L2 holds the records of one region of the tree.
__device__ inline uint32_t xcd_contiguous_block() {
    const uint32_t xcd = blockIdx.x % kXcds, per = gridDim.x / kXcds, extra = gridDim.x % kXcds;
    return xcd * per + min(xcd, extra) + blockIdx.x / kXcds;
}

// The reference's opening test edge * (1.0 / sqrt(d2)) < theta of a child of
// level l (edge = root edge 2^-l).  It is decided from d2 against edge^2 /
// theta^2 (1 +- 2^-29), within a few roundings of the exact bound, and only the
// squared distances between those two pay the IEEE square root and division
// (exact).  A theta or a root edge whose squares could leave the normal range
// turns the bounds into NaN: then every test is the exact one.
struct ExactTest {
    double edge, theta, bound;
    __device__ ExactTest(double root_edge, double theta_) : edge(root_edge), theta(theta_) {
        const double e2 = edge * edge;
        const bool squares = (theta == 0.0 || (theta >= 1e-100 && theta <= 1e100)) &&
                             e2 >= 1e-60 && e2 <= 1e60;
        bound = squares ? e2 / (theta * theta) : __builtin_nan("");
    }
    __device__ double far2(int level) const { return ldexp(bound * (1.0 + 0x1p-29), -2 * level); }
    __device__ double near2(int level) const { return ldexp(bound * (1.0 - 0x1p-29), -2 * level); }
    __device__ bool far(int level, double d2) const {
        const double scaled = ldexp(d2, 2 * level);  // against the root's bounds
        bool yes = scaled > bound * (1.0 + 0x1p-29);
        if (!yes && !(scaled < bound * (1.0 - 0x1p-29))) yes = exact(level, d2);
        return yes;
    }
    __device__ bool exact(int level, double d2) const {
        const double d = 1.0 / sqrt(d2);
        return ldexp(edge, -level) * d < theta;
    }
};

__global__ void __launch_bounds__(kExactThreads) __attribute__((amdgpu_waves_per_eu(5)))
k_bh_exact_team(uint32_t n, const uint32_t *__restrict__ order, const double *__restrict__ x,
           const double *__restrict__ y, const double *__restrict__ z,
           const double4 *__restrict__ cm, const int32_t *__restrict__ ref, double G, double eps2,
           double theta, uint32_t icap, double *ax, double *ay, double *az, uint32_t *inter,
           TreeHdr *h) {
    __shared__ TeamLds lds[kExactWaves];
    const uint32_t lb = xcd_contiguous_block();
    const uint32_t lane = threadIdx.x & 63u, p = lane & 7u, team = lane >> 3, base = lane & 56u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    TeamLds &L = lds[wave];
    const uint64_t id = (uint64_t)(lb * kExactWaves + wave) * kTeams + team;
    const bool valid = id < n;
    const uint32_t i = order[valid ? id : n - 1];
    const int32_t self_ref = ref_of_body(i);
    const double px = x[i], py = y[i], pz = z[i];
    const uint32_t digit = visit_digit(p), below = (1u << p) - 1u;
    const ExactTest test(h->edge, theta);
    double acc = 0.0;           // lane p < 3: component p of the body's sum
    uint32_t cnt = 0;           // accepted nodes
    uint32_t ln = 0, sp = 0;    // list and stack sizes
    uint32_t cell = 0;          // the cell to open, if there is one
    uint32_t level = 0;         // its children's level (the root is level 0)
    bool have = false;
    uint32_t late = kTeamStack;  // stack entry whose next child to open is being loaded
    int32_t late_ref = 0;
    uint32_t budget = icap + 16;  // a correct octree is entered once per cell

    // the terms of the lists' full batches of eight (all: of every entry)
    auto flush = [&](bool all) {
        const uint32_t nb = all ? (ln + 7) >> 3 : ln >> 3;
        for (uint32_t b = 0; __ballot(b < nb); ++b) {
            const uint32_t k = 8 * b + p;
            const bool use = b < nb && k < ln;
            double t_x = 0.0, t_y = 0.0, t_z = 0.0;
            if (use) {
                const double4 c = cm[L.list[team][k]];
                const double d_x = c.x - px;
                const double d_y = c.y - py;
                const double d_z = c.z - pz;
                double den = (d_x * d_x) + (d_y * d_y) + (d_z * d_z) + eps2;
                den = den * den * den;
                den = inv_sqrt_ieee(den);
                t_x = c.w * (d_x * den);
                t_y = c.w * (d_y * den);
                t_z = c.w * (d_z * den);
            }
            L.term[team][0][p] = t_x;
            L.term[team][1][p] = t_y;
            L.term[team][2][p] = t_z;
            wave_lds_sync();
            if (p < 3) {
                double v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = L.term[team][p][u];
#pragma unroll
                for (int u = 0; u < 8; ++u) acc += v[u];
            }
            wave_lds_sync();
        }
        const uint32_t done = 8 * nb;
        if (!all && done > 0 && p < ln - done) L.list[team][p] = L.list[team][done + p];
        ln = all ? 0u : ln - done;
        wave_lds_sync();
    };

    // this lane's byte of a ballot: its team's positions
    auto team_bits = [&](uint64_t m) {
        return (uint32_t)((lane < 32 ? (uint32_t)m : (uint32_t)(m >> 32)) >> (base & 31u)) & 0xffu;
    };
    {
        const double4 c = cm[0];
        const int32_t r = ref[0];
        const double d_x = c.x - px, d_y = c.y - py, d_z = c.z - pz;
        const double d2 = d_x * d_x + d_y * d_y + d_z * d_z;
        const bool real = valid && r != kRefEmpty && c.w != 0;
        const bool take = real && (r < 0 ? r != self_ref : test.far(0, d2));
        if (take) {
            if (p == 0) L.list[team][0] = 0;
            cnt = ln = 1;
        } else if (real && r >= 0) {
            have = true;
            cell = (uint32_t)r;
            level = 1;
        }
    }
    while (__ballot(have || sp > 0)) {
        if (__ballot(ln > kTeamList - 16)) flush(false);
        if (late < kTeamStack) {
            if (p == 0) L.ref[late][team] = (uint32_t)late_ref;
            late = kTeamStack;
        }
        wave_lds_sync();
        // Without a cell to open: back to the deepest cell with children left,
        // for its accepted children before its next one to open.  One entry per
        // step: the teams' pops then run side by side with each other and with
        // the openings below, instead of in a loop as long as the longest.
        if (!have && sp > 0) {
            const uint32_t pc = L.cell[sp - 1][team], m = L.masks[sp - 1][team];
            uint32_t et = m & 0xffu, eo = (m >> 8) & 0xffu;
            const uint32_t q = (uint32_t)__builtin_ctz(eo | 0x100u);
            const uint32_t before = (1u << q) - 1u, above = ~(2u * before + 1u);
            const uint32_t emit = et & before;
            if (emit >> p & 1u)
                L.list[team][ln + __popc(emit & below)] = (uint32_t)(8ull * pc + 1u + digit);
            ln += __popc(emit);
            et &= above;
            eo &= above;
            have = q < 8;
            level = (m >> 16) + 1;
            cell = L.ref[sp - 1][team];
            if (et | eo) {
                if (p == 0) L.masks[sp - 1][team] = (m & 0xffff0000u) | eo << 8 | et;
                if (eo) {
                    late = sp - 1;
                    late_ref = ref[8ull * pc + 1u + visit_digit((uint32_t)__builtin_ctz(eo))];
                }
            } else {
                --sp;
            }
        }
        bool take = false, open = false;
        int32_t r = 0;
        uint32_t node = 0;
        if (have) {
            node = 8u * cell + 1u + digit;
            const double4 c = cm[node];
            r = ref[node];
            const double d_x = c.x - px;
            const double d_y = c.y - py;
            const double d_z = c.z - pz;
            const double d2 = d_x * d_x + d_y * d_y + d_z * d_z;
            const bool real = r != kRefEmpty && c.w != 0;
            if (r < 0) {
                take = real && r != self_ref;
            } else {
                take = test.far((int)level, d2);
                open = real && !take;
                take = real && take;
            }
        }
        uint32_t mt = team_bits(__ballot(take)), mo = team_bits(__ballot(open));
        cnt += __popc(mt);
        // the accepted children before the first one to open
        const uint32_t q = (uint32_t)__builtin_ctz(mo | 0x100u);
        const uint32_t before = (1u << q) - 1u, above = ~(2u * before + 1u);
        if (take && p < q) L.list[team][ln + __popc(mt & below)] = node;
        ln += __popc(mt & before);
        mt &= above;
        mo &= above;
        const uint32_t q2 = (uint32_t)__builtin_ctz(mo | 0x100u);
        const uint32_t next = (uint32_t)__shfl(r, (int)(base + (q & 7u)), 64);
        const uint32_t next2 = (uint32_t)__shfl(r, (int)(base + (q2 & 7u)), 64);
        have = q < 8;
        if (have) {
            if (mt | mo) {
                if (p == 0) {
                    L.cell[sp][team] = cell;
                    L.ref[sp][team] = next2;
                    L.masks[sp][team] = level << 16 | mo << 8 | mt;
                }
                ++sp;
            }
            cell = next;
            ++level;
            if (level > kMaxDepth + 1 || budget-- == 0) {  // a corrupt octree
                if (p == 0) raise_flag(h, kFlagStack);
                have = false;
                sp = 0;
                late = kTeamStack;
            }
        }
    }
    flush(true);
    if (!valid) return;
    if (p < 3) (p == 0 ? ax : (p == 1 ? ay : az))[i] = acc * G;
    if (inter && p == 3) inter[i] = cnt;
}

// k_bh_exact_wave: a wave walks the tree once for 64 bodies in octree order.  It
// visits, in the reference's pre-order, every node that any of them visits, and
// each lane takes part in the subtrees of the cells that its own body opens, so a
// body's accepted nodes come by in its own visit order.  The node at hand is the
// same for the whole wave: its record is an LDS broadcast (through v_readlane or
// the scalar cache: 7.2 and 8.2 ms on the 1M-body disk), empty slots cost a bit
// of a mask.  Bound by FP64 issue: on that disk a wave visits 2826 nodes, of
// which a body accepts 1130, at about 290 cycles each.
constexpr uint32_t kFrames = 8;  // levels of a wave's path whose children are kept in LDS
struct WaveLds {
    double4 cm[kFrames][8];           // by visit position
    int32_t ref[kFrames][8];
    uint2 path[kTeamStack];           // per level with children left: cell, their positions
};

__global__ void __launch_bounds__(kExactThreads) __attribute__((amdgpu_waves_per_eu(8)))
k_bh_exact_wave(uint32_t n, const uint32_t *__restrict__ order, const double *__restrict__ x,
                const double *__restrict__ y, const double *__restrict__ z,
                const double4 *__restrict__ cm, const int32_t *__restrict__ ref, double G,
                double eps2, double theta, uint32_t icap, double *ax, double *ay, double *az,
                uint32_t *inter, TreeHdr *h) {
    __shared__ WaveLds lds[kExactWaves];
    const uint32_t lb = xcd_contiguous_block();
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    WaveLds &L = lds[w];
    const uint64_t first = (uint64_t)(lb * kExactWaves + w) * 64u;
    if (first >= n) return;
    const bool valid = first + lane < n;
    const uint32_t i = order[valid ? first + lane : first];
    const int32_t self_ref = ref_of_body(i);
    const double px = x[i], py = y[i], pz = z[i];
    double acc_x = 0, acc_y = 0, acc_z = 0;
    uint32_t cnt = 0;
    const ExactTest test(h->edge, theta);
    // Levels: the root's slot is the only child of level 0, the children of the
    // root cell are level 1, and so on.  A lane takes part in level l if its
    // body opened the cell above (opened >= l; -1: no body).
    int opened = valid ? 0 : -1;
    uint64_t frames = 1;  // the levels whose children are in their frame (level mod kFrames)
    uint64_t resume = 0;  // the levels with children left
    const uint32_t digit = visit_digit(lane & 7u);
    int level = 0;
    uint32_t cell = 0;  // above the level
    // the children of `cell` into the level's frame; returns the positions of
    // those with a mass
    auto load_frame = [&](bool root) {
        const uint64_t node = root ? 0ull : 8ull * cell + 1u + digit;
        const double4 c = cm[node];
        const int32_t r = ref[node];
        const uint32_t k = (uint32_t)level % kFrames;
        wave_lds_sync();
        if (lane < 8) {
            // by component: the compiler passes a whole structure through scratch memory
            double *to = table_as<double>(&L.cm[k][lane]);
            to[0] = c.x;
            to[1] = c.y;
            to[2] = c.z;
            to[3] = c.w;
            L.ref[k][lane] = r;
        }
        wave_lds_sync();
        frames &= ~(0x0101010101010101ull << k);
        frames |= 1ull << level;
        return (uint32_t)__ballot(r != kRefEmpty && c.w != 0) & (root ? 1u : 0xffu);
    };
    uint32_t left = load_frame(true);
    uint32_t budget = icap + 16;  // a correct octree enters a cell once
    for (;;) {
        const bool here = opened >= level;
        const double far2 = test.far2(level), near2 = test.near2(level);
        const uint32_t k = (uint32_t)level % kFrames;
        bool open = false;
        int32_t r = 0;
        while (left) {  // the level's children until one is opened
            const uint32_t p = (uint32_t)__builtin_ctz(left);
            left &= left - 1;
            const double4 c = L.cm[k][p];
            r = (int32_t)wave_uniform((uint32_t)L.ref[k][p]);
            const double d_x = c.x - px;
            const double d_y = c.y - py;
            const double d_z = c.z - pz;
            const double d2 = d_x * d_x + d_y * d_y + d_z * d_z;
            bool take;
            if (r < 0) {
                take = here && r != self_ref;
            } else {
                bool far = d2 > far2;
                if (here && !far && !(d2 < near2)) far = test.exact(level, d2);
                open = here && !far;
                take = here && far;
            }
            if (take) {
                double den = d2 + eps2;
                den = den * den * den;
                den = inv_sqrt_ieee(den);
                acc_x += c.w * (d_x * den);
                acc_y += c.w * (d_y * den);
                acc_z += c.w * (d_z * den);
                ++cnt;
            }
            if (__ballot(open)) break;
        }
        if (__ballot(open)) {
            if (left) {
                L.path[level] = make_uint2(cell, left);
                resume |= 1ull << level;
            }
            ++level;
            if (budget-- == 0 || level > kMaxDepth + 1) {  // a corrupt octree
                if (lane == 0) raise_flag(h, kFlagStack);
                break;
            }
            if (open) opened = level;
            cell = (uint32_t)r;
            left = load_frame(false);
        } else {
            if (resume == 0) break;
            level = 63 - __clzll((long long)resume);
            resume &= ~(1ull << level);
            wave_lds_sync();
            const uint2 at = L.path[level];
            cell = wave_uniform(at.x);
            if (!(frames >> level & 1ull)) (void)load_frame(false);
            left = wave_uniform(at.y);
            opened = min(opened, level);
        }
    }
    if (!valid) return;
    ax[i] = acc_x * G;
    ay[i] = acc_y * G;
    az[i] = acc_z * G;
    if (inter) inter[i] = cnt;
}

// ---------------------------------------------------------------------------
// Group traversal (FP32 pair maths, FP64 accumulation).
//
// One wavefront walks the octree for one group: an octree cell with at most
// 64 bodies (a contiguous run of the octree order).  A cell is accepted when
// its centre of mass is farther than edge/theta from the group's bounding box
// -- so from every body of the group: the reference's opening test
// (BarnesHutAlgorithm.cpp:355-359) taken over the group; bodies in leaves are
// always taken exactly.  Each iteration pops up to 8 cells whose children
// must be examined, and lane l examines child (l & 7) of cell l >> 3: one
// 32-byte record load per lane.  Accepted cells and bodies are appended to an
// LDS list; every 128 entries the list is evaluated against the group's bodies.
// A group of s bodies uses lpb = floor(64/s) lanes per body, each taking
// every lpb-th list entry, so s * lpb of the 64 lanes do useful pairs (51 for
// s = 17, where rounding s up to a power of two would leave 34).
// Positions are relative to the group centre; the records' hi/lo split keeps
// the FP32 differences exact to the last FP32 bit.  Waves take groups from an
// atomic work queue.
constexpr int kGroup = 64;          // lanes per wavefront (a group has up to 2 x kGroup bodies)
static_assert(kGroupMax <= 2 * kGroup, "a lane holds at most two bodies of its group");
static_assert(kGroupLimit <= kGroup, "the tunable groups fit one body per lane");
constexpr int kStackCap = 1024;     // cells waiting to be opened (entry = k << 6 | depth)
// Child records per lane and walk step (8 kPop cells).  More loads in flight
// per wave cost registers: on a 1M-body disk kPop 2 and 4 made the traversal
// 7 % and 17 % slower than 1 (occupancy 6 -> 4 waves per SIMD).
constexpr int kPop = 1;
// List entries evaluated per flush, at most.  Each flush folds its FP32 sums
// into the FP64 accumulators and moves the list's tail to the front: 128
// entries halve those costs against 64.
constexpr int kFlushSpan = 2 * kGroup;
constexpr int kListCap = kFlushSpan + kGroup * kPop;
constexpr int kGroupBlocks = 8192;  // persistent waves
constexpr uint32_t kQueueStride = 32;  // one 128-byte line per group-queue counter
static_assert(kXcds * kQueueStride <= TreeBufs::kGroupQueueWords, "queue counters fit TreeBufs::gq");

// Every traversal starts with fresh queue cursors (a kernel, not a memset,
// so the sequence can be captured in a graph).

// The device-scope maximum with a read first: the read-modify-write (which
// serialises at one memory channel when every wave does it) only when it
// raises the value.
__device__ inline void raise_max(uint32_t *p, uint32_t v) {
    if (v > __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(p, v);
}

// Set bits of a wave-uniform mask in the lanes below this one (v_mbcnt: two
// VALU instructions, where a per-lane mask and popcount take four).
__device__ inline uint32_t count_below(uint64_t mask) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                     __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// lane 0's value of v, uniform
__device__ inline uint32_t lane0_uniform(uint32_t v) { return wave_uniform(__shfl(v, 0, 64)); }

// With the learned correction (kCorr), accepted cells that are close enough
// (e^2 > tau2 * d_group^2) are also queued in a second LDS list; every 16 such
// cells, the wave evaluates the network for the 16 cells x each body of the
// group (one 16-sample matrix-core tile per body) and adds the corrections of
// a body in a fixed order.
constexpr int kCorrTile = 16;
constexpr int kCellCap = kCorrTile + kGroup * kPop;

// One octree as the group walk sees it (body indices of sidx and of the node
// references index x, y, z, m, ax, ay, az, inter).
struct GroupTree {
    uint32_t n;
    const uint32_t *sidx;
    const double *x, *y, *z, *m;
    const NodeF32 *rec;
    uint32_t icap;
    float ro2_root;  // (root edge / theta)^2
    float e2_root;   // root edge^2
    double *ax, *ay, *az;
    uint32_t *inter;
    const float4 *gquad;  // G*Q per internal cell (quadrupole walks)
};

// Four entries on NB points, in entry order, their v_rsq_f32 together.
template <int NB>
__device__ __forceinline__ void pairs4_f32(const float4 (&e)[4], const float (&rx)[NB],
                                           const float (&ry)[NB], const float (&rz)[NB], float eps2,
                                           float (&fx)[NB], float (&fy)[NB], float (&fz)[NB]) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        float dx[4], dy[4], dz[4], inv[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            dx[u] = e[u].x - rx[b];
            dy[u] = e[u].y - ry[b];
            dz[u] = e[u].z - rz[b];
            inv[u] = fmaf(dx[u], dx[u], fmaf(dy[u], dy[u], fmaf(dz[u], dz[u], eps2)));
        }
        rsq4_f32(inv);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const float f = (e[u].w * inv[u]) * (inv[u] * inv[u]);
            fx[b] = fmaf(f, dx[u], fx[b]);
            fy[b] = fmaf(f, dy[u], fy[b]);
            fz[b] = fmaf(f, dz[u], fz[b]);
        }
    }
}

// The same for a stride known only at run time (lanes per body not a power
// of two).
__device__ __forceinline__ void flush_share_rt(const float4 *p, uint32_t stride, uint32_t t,
                                               float rx, float ry, float rz, float eps2, float &fx,
                                               float &fy, float &fz) {
    uint32_t k = 0;
    for (; k + 4 <= t; k += 4) {
        const float4 e[4] = {p[(k + 0) * stride], p[(k + 1) * stride], p[(k + 2) * stride],
                             p[(k + 3) * stride]};
        const float px[1] = {rx}, py[1] = {ry}, pz[1] = {rz};
        float gx[1] = {fx}, gy[1] = {fy}, gz[1] = {fz};
        pairs4_f32<1>(e, px, py, pz, eps2, gx, gy, gz);
        fx = gx[0];
        fy = gy[0];
        fz = gz[0];
    }
    for (; k < t; ++k) pair_f32(p[k * stride], rx, ry, rz, eps2, fx, fy, fz);
}

// Pair forces of list entries p[0], p[LPB], p[2 LPB], ... (t entries, in that
// order) on the NB points (rx, ry, rz)[b].  LPB and the uniform trip count make
// the LDS offsets immediates and let four reads be in flight ahead of the
// maths; with NB = 2 every entry read feeds two pairs.
template <int LPB, int NB>
__device__ __forceinline__ void flush_share(const float4 *p, uint32_t t, const float (&rx)[NB],
                                            const float (&ry)[NB], const float (&rz)[NB],
                                            float eps2, float (&fx)[NB], float (&fy)[NB],
                                            float (&fz)[NB]) {
    uint32_t k = 0;
    for (; k + 4 <= t; k += 4) {
        const float4 e[4] = {p[(k + 0) * LPB], p[(k + 1) * LPB], p[(k + 2) * LPB],
                             p[(k + 3) * LPB]};
        pairs4_f32<NB>(e, rx, ry, rz, eps2, fx, fy, fz);
    }
    for (; k < t; ++k) {
        const float4 e = p[k * LPB];
#pragma unroll
        for (int b = 0; b < NB; ++b) pair_f32(e, rx[b], ry[b], rz[b], eps2, fx[b], fy[b], fz[b]);
    }
}

// A list entry that adds exactly zero for any eps^2: its distance squared
// overflows to +inf, so rsqrt gives 0 and the force 0 * offset = 0.
__device__ inline float4 far_entry() { return make_float4(1e30f, 0.f, 0.f, 0.f); }

// A cell's monopole and traceless quadrupole, G folded into e.w = G M and
// Q = G sum m (3 s s^T - |s|^2 I) about the cell's centre of mass, passed as
// qa = {xx, yy, zz, xy}, qb = {xz, yz, -, -}.  With R = com - body (the pair
// offset), the potential -G M / |R| - R.Q.R / (2 |R|^5) gives
//   a = R (G M + 5/2 R.Q.R / R^2) / R^3 - Q.R / R^5,
// with R^2 softened by eps^2 as in the monopole.  32 VALU instructions (the
// monopole pair takes 13); 49 flop by the direct sum's counting.
__device__ inline void pair_quad(const float4 e, const float4 qa, const float4 qb, float px,
                                 float py, float pz, float eps2, float &fx, float &fy, float &fz) {
    const float dx = e.x - px, dy = e.y - py, dz = e.z - pz;
    const float r2 = fmaf(dx, dx, fmaf(dy, dy, fmaf(dz, dz, eps2)));
    const float inv = __builtin_amdgcn_rsqf(r2);
    const float inv2 = inv * inv;
    const float inv3 = inv * inv2;
    const float qx = fmaf(qa.x, dx, fmaf(qa.w, dy, qb.x * dz));
    const float qy = fmaf(qa.w, dx, fmaf(qa.y, dy, qb.y * dz));
    const float qz = fmaf(qb.x, dx, fmaf(qb.y, dy, qa.z * dz));
    const float rqr = fmaf(dx, qx, fmaf(dy, qy, dz * qz));
    const float b = inv3 * inv2;                                // R^-5
    const float a = fmaf((2.5f * rqr) * inv2, b, e.w * inv3);  // GM R^-3 + 5/2 RQR R^-7
    fx = fmaf(a, dx, fx);
    fy = fmaf(a, dy, fy);
    fz = fmaf(a, dz, fz);
    fx = fmaf(-b, qx, fx);
    fy = fmaf(-b, qy, fy);
    fz = fmaf(-b, qz, fz);
}

// Quadrupole pairs of cell entries p[0], p[LPB], ... (t of them, cell indices
// k[0], k[LPB], ...; the cells' G*Q records in gq[2k], gq[2k+1]).  Four
// entries' records are loaded ahead of their arithmetic.
template <int LPB>
__device__ __forceinline__ void qflush_share(const float4 *p, const uint32_t *k, uint32_t stride,
                                             uint32_t t, const float4 *__restrict__ gq, float rx,
                                             float ry, float rz, float eps2, float &fx, float &fy,
                                             float &fz) {
    const uint32_t st = LPB > 0 ? (uint32_t)LPB : stride;
    uint32_t u = 0;
    for (; u + 4 <= t; u += 4) {
        float4 e[4], qa[4], qb[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            e[v] = p[(u + v) * st];
            const uint32_t c = k[(u + v) * st];
            qa[v] = gq[2ull * c];
            qb[v] = gq[2ull * c + 1];
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) pair_quad(e[v], qa[v], qb[v], rx, ry, rz, eps2, fx, fy, fz);
    }
    for (; u < t; ++u) {
        const uint32_t c = k[u * st];
        pair_quad(p[u * st], gq[2ull * c], gq[2ull * c + 1], rx, ry, rz, eps2, fx, fy, fz);
    }
}

// LDS of one wave's walk.
struct GroupLds {
    uint32_t *stk;
    float4 *lst;
    float4 *qlst;    // quadrupole: accepted cells' entries
    uint32_t *qk;    // quadrupole: their internal-cell indices
    float4 *cl_e;    // correction: accepted cell offset from the group centre, G*M
    uint32_t *cl_k;  // correction: accepted cell's internal index
    float4 *boff;    // correction: body offsets from the group centre
    float4 *bcorr;   // correction: learned correction per body
};

// Bodies of the first of two passes over each flushed list, for a group of
// s <= 64 bodies (s: one pass), and the list entries per flush.  A pass over
// sa bodies gives each 64 / sa lanes, so an entry costs 1 / (64 / sa) trips;
// the split minimising the trips of both passes is taken if it saves at least
// 12 % of the one-pass trips (a second pass has its own set-up, reduction and
// registers; 31 of the 64 sizes split).  26 bodies: 5 with 12 lanes, then 21
// with 3, 0.42 trips per entry instead of 0.5 with 2 lanes each (52 of 64
// lanes busy).  A flush takes a multiple
// of both passes' lanes per body (60 for 3 and 12), so that only a group's
// last flush has remainder trips.  Computed at compile time.
struct TwoPass {
    uint8_t first[kGroup + 1];
    uint8_t chunk[kGroup + 1];
};
static_assert(kFlushSpan <= 255, "flush spans fit TwoPass::chunk");
constexpr uint32_t gcd_u32(uint32_t a, uint32_t b) { return b ? gcd_u32(b, a % b) : a; }
constexpr TwoPass make_two_pass() {
    TwoPass t{};
    for (uint32_t s = 1; s <= (uint32_t)kGroup; ++s) {
        // compare sums of 1 / lanes-per-body exactly: a / b < c / d <=> a d < c b
        const uint32_t one = (uint32_t)kGroup / s;  // one pass: 1 / one trips per entry
        uint32_t best = s, bn = 1, bd = one;          // best cost bn / bd
        for (uint32_t a = 1; a < s; ++a) {
            const uint32_t l1 = (uint32_t)kGroup / a, l2 = (uint32_t)kGroup / (s - a);
            const uint32_t cn = l1 + l2, cd = l1 * l2;  // 1 / l1 + 1 / l2
            if (cn * bd < bn * cd && 100 * cn * one < 88 * cd) {
                best = a;
                bn = cn;
                bd = cd;
            }
        }
        t.first[s] = (uint8_t)best;
        const uint32_t l1 = (uint32_t)kGroup / best;
        const uint32_t l2 = best < s ? (uint32_t)kGroup / (s - best) : l1;
        const uint32_t lcm = l1 / gcd_u32(l1, l2) * l2;
        t.chunk[s] = (uint8_t)(lcm <= (uint32_t)kFlushSpan ? lcm * ((uint32_t)kFlushSpan / lcm)
                                                             : (uint32_t)kFlushSpan);
    }
    return t;
}
__constant__ constexpr TwoPass kTwoPassTable = make_two_pass();

// Forces on the s bodies of one group starting at sorted position g0 (both
// wave-uniform, checked by the caller).  NB = 1 (s <= 64): lane l holds body
// l % s and list share l / s; the lpb = 64 / s lanes of a body share its list,
// and the 64 - s * lpb lanes beyond repeat share 0 and their sums are dropped.
// NB = 2 (64 < s <= 128): a lane holds bodies lane and lane + 64 and takes
// the whole list for both.  Monopole walks of one body per lane split the
// group into two passes over every flushed list (kTwoPassTable): bodies
// [0, sa) as above with sa in place of s, then bodies [sa, s), lane l
// holding body sa + l % (s - sa) and share l / (s - sa).  *ncorr_out
// accumulates network evaluations.
template <bool kCorr, int NB, bool kQuad>
__device__ __forceinline__ void group_walk_n(const GroupTree &T, uint32_t g0, uint32_t s,
                                             float eps2, const CorrArgs &corr,
                                             const MlpForward &w, const GroupLds &L,
                                             uint32_t &peak, bool &overflow,
                                             uint32_t &ncorr_out, uint32_t &nquad_out) {
    static_assert(!kQuad || NB == 1, "quadrupole walks hold one body per lane");
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t *__restrict__ sidx = T.sidx;
    const double *__restrict__ x = T.x, *__restrict__ y = T.y, *__restrict__ z = T.z,
                 *__restrict__ m = T.m;
    const NodeF32 *__restrict__ rec = T.rec;
    const uint32_t icap = T.icap;
    const float ro2_root = T.ro2_root, e2_root = T.e2_root;
    double *ax = T.ax, *ay = T.ay, *az = T.az;
    uint32_t *inter = T.inter;
    uint32_t *stk = L.stk;
    float4 *lst = L.lst, *cl_e = L.cl_e, *boff = L.boff, *bcorr = L.bcorr;
    uint32_t *cl_k = L.cl_k;
    float4 *qlst = L.qlst;
    uint32_t *qk = L.qk;
    const float4 *__restrict__ gquad = T.gquad;
    {
        // (quadrupole walks keep one pass: their second list is shared out
        // by the first pass's mapping only)
        constexpr bool kTwoPass = !kQuad && NB == 1;
        // bodies of the first pass (all of them without a second one)
        const uint32_t sa = kTwoPass && NB == 1 ? (uint32_t)kTwoPassTable.first[s] : s;
        const uint32_t sb = s - sa;                             // second pass: 0 or more
        const uint32_t ss = NB == 2 ? (uint32_t)kGroup : sa;  // body slots of the first pass
        const uint32_t sub = NB == 2 ? lane : lane % ss;      // which body of the group
        const uint32_t q = NB == 2 ? 0u : lane / ss;          // which share of the list
        const uint32_t lpb = (uint32_t)kGroup / ss;           // lanes per body
        const uint32_t qs = q < lpb ? q : 0u;                 // the share this lane computes
        // the second pass: body sa + sub2 in share q2 of 64 / sb
        const uint32_t sub2 = sb ? lane % sb : 0u;
        const uint32_t q2 = sb ? lane / sb : 0u;
        const uint32_t lpb2 = sb ? (uint32_t)kGroup / sb : 1u;
        const uint32_t qs2 = q2 < lpb2 ? q2 : 0u;
        // list entries per flush: a multiple of lpb (124 to 128), so that only
        // the group's last flush has a remainder trip (of lpb2 too with two passes)
        const uint32_t chunk =
            sb ? (uint32_t)kTwoPassTable.chunk[s] : lpb * ((uint32_t)kFlushSpan / lpb);
        const bool pow2 = (ss & (ss - 1)) == 0;
        bool valid[NB];
        uint32_t bi[NB];
        double px[NB], py[NB], pz[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const uint32_t k = sub + (uint32_t)b * kGroup;
            valid[b] = k < (NB == 2 ? s : sa);
            // an unused slot repeats a body of the group (its box stays the group's)
            bi[b] = sidx[g0 + (valid[b] ? k : (b == 0 ? 0u : sub))];
            px[b] = x[bi[b]];
            py[b] = y[bi[b]];
            pz[b] = z[bi[b]];
        }
        // the second pass's body (every lane holds one of the sb bodies)
        uint32_t bi2 = bi[0];
        double px2 = px[0], py2 = py[0], pz2 = pz[0];
        if (sb) {
            bi2 = sidx[g0 + sa + sub2];
            px2 = x[bi2];
            py2 = y[bi2];
            pz2 = z[bi2];
        }

        // bounding box (FP64, exact min/max), centre and half extent
        double mnx = fmin(px[0], px2), mny = fmin(py[0], py2), mnz = fmin(pz[0], pz2);
        double mxx = fmax(px[0], px2), mxy = fmax(py[0], py2), mxz = fmax(pz[0], pz2);
#pragma unroll
        for (int b = 1; b < NB; ++b) {
            mnx = fmin(mnx, px[b]);
            mny = fmin(mny, py[b]);
            mnz = fmin(mnz, pz[b]);
            mxx = fmax(mxx, px[b]);
            mxy = fmax(mxy, py[b]);
            mxz = fmax(mxz, pz[b]);
        }
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) {
            mnx = fmin(mnx, __shfl_xor(mnx, off, 64));
            mny = fmin(mny, __shfl_xor(mny, off, 64));
            mnz = fmin(mnz, __shfl_xor(mnz, off, 64));
            mxx = fmax(mxx, __shfl_xor(mxx, off, 64));
            mxy = fmax(mxy, __shfl_xor(mxy, off, 64));
            mxz = fmax(mxz, __shfl_xor(mxz, off, 64));
        }
        const double cx = 0.5 * (mnx + mxx), cy = 0.5 * (mny + mxy), cz = 0.5 * (mnz + mxz);
        // half extents rounded up so that the FP32 box always contains the bodies
        const float hx = (float)(0.5 * (mxx - mnx)) * 1.000001f;
        const float hy = (float)(0.5 * (mxy - mny)) * 1.000001f;
        const float hz = (float)(0.5 * (mxz - mnz)) * 1.000001f;
        const float gxh = (float)cx, gyh = (float)cy, gzh = (float)cz;
        const float gxl = (float)(cx - (double)gxh), gyl = (float)(cy - (double)gyh),
                    gzl = (float)(cz - (double)gzh);
        // The body's own offset is computed with exactly the operations that
        // produce its leaf's list entry (record hi/lo of (x*m)/m, k_records),
        // so the self pair has a distance of exactly 0 and adds nothing; with
        // eps^2 = 1e-22 any rounding residual would be a huge spurious force.
        float rx[NB], ry[NB], rz[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const double mb = m[bi[b]];
            const double c3[3] = {(px[b] * mb) / mb, (py[b] * mb) / mb, (pz[b] * mb) / mb};
            const float gh[3] = {gxh, gyh, gzh}, gl[3] = {gxl, gyl, gzl};
            float r3[3];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const float hi = (float)c3[c];
                const float lo = (float)(c3[c] - (double)hi);
                r3[c] = (hi - gh[c]) + (lo - gl[c]);
            }
            rx[b] = r3[0];
            ry[b] = r3[1];
            rz[b] = r3[2];
        }
        float rx2 = rx[0], ry2 = ry[0], rz2 = rz[0];
        if (sb) {
            const double mb = m[bi2];
            const double c3[3] = {(px2 * mb) / mb, (py2 * mb) / mb, (pz2 * mb) / mb};
            const float gh[3] = {gxh, gyh, gzh}, gl[3] = {gxl, gyl, gzl};
            float r3[3];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const float hi = (float)c3[c];
                const float lo = (float)(c3[c] - (double)hi);
                r3[c] = (hi - gh[c]) + (lo - gl[c]);
            }
            rx2 = r3[0];
            ry2 = r3[1];
            rz2 = r3[2];
        }

        double acc_x[NB], acc_y[NB], acc_z[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) acc_x[b] = acc_y[b] = acc_z[b] = 0.0;
        double acc2_x = 0.0, acc2_y = 0.0, acc2_z = 0.0;  // the second pass's body
        uint32_t n_inter = 0;
        uint32_t sp = 0, ln = 0;  // wave-uniform stack and list sizes
        uint32_t cn = 0;          // wave-uniform size of the correction's cell list
        uint32_t ncorr = 0;       // network evaluations of this group
        uint32_t qn = 0;          // wave-uniform size of the quadrupole cell list
        uint32_t nquad = 0;       // quadrupole pairs of this group
        if constexpr (kCorr) {
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const uint32_t k = sub + (uint32_t)b * kGroup;
                if (valid[b] && q == 0) boff[k] = make_float4(rx[b], ry[b], rz[b], 0.f);
                bcorr[lane + (uint32_t)b * kGroup] = make_float4(0.f, 0.f, 0.f, 0.f);
            }
            if (kTwoPass && sb && q2 == 0) boff[sa + sub2] = make_float4(rx2, ry2, rz2, 0.f);
        }

        // Entries lst[base .. base + cnt) (cnt <= kFlushSpan): lane share qs takes
        // qs, qs + lpb, ...  Every share runs cnt / lpb trips; then shares
        // qs < cnt % lpb take one more entry and the others a zero-force
        // entry (a select, so the trip count stays uniform and nothing is
        // written to the list).  The reads stay below base + cnt + lpb, inside
        // the list.
        auto flush = [&](uint32_t base, uint32_t cnt) {
            const uint32_t full = cnt / lpb;
            const uint32_t rem = cnt - full * lpb;
            const float4 *p = lst + base + qs;
            float fx[NB], fy[NB], fz[NB];
#pragma unroll
            for (int b = 0; b < NB; ++b) fx[b] = fy[b] = fz[b] = 0.f;
            if constexpr (NB == 2) {
                flush_share<1, 2>(p, cnt, rx, ry, rz, eps2, fx, fy, fz);  // lpb = 1
            } else {
                switch (lpb) {
                case 1: flush_share<1, 1>(p, full, rx, ry, rz, eps2, fx, fy, fz); break;
                case 2: flush_share<2, 1>(p, full, rx, ry, rz, eps2, fx, fy, fz); break;
                case 3: flush_share<3, 1>(p, full, rx, ry, rz, eps2, fx, fy, fz); break;
                case 4: flush_share<4, 1>(p, full, rx, ry, rz, eps2, fx, fy, fz); break;
                case 8: flush_share<8, 1>(p, full, rx, ry, rz, eps2, fx, fy, fz); break;
                case 16: flush_share<16, 1>(p, full, rx, ry, rz, eps2, fx, fy, fz); break;
                case 32: flush_share<32, 1>(p, full, rx, ry, rz, eps2, fx, fy, fz); break;
                case 64: flush_share<64, 1>(p, full, rx, ry, rz, eps2, fx, fy, fz); break;
                default:
                    flush_share_rt(p, lpb, full, rx[0], ry[0], rz[0], eps2, fx[0], fy[0], fz[0]);
                    break;
                }
                if (rem) {
                    const float4 e = p[full * lpb];
                    pair_f32(qs < rem ? e : far_entry(), rx[0], ry[0], rz[0], eps2, fx[0], fy[0],
                             fz[0]);
                }
            }
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                acc_x[b] += (double)fx[b];
                acc_y[b] += (double)fy[b];
                acc_z[b] += (double)fz[b];
            }
            if (kTwoPass && sb) {  // the same entries for the second pass's bodies
                const uint32_t full2 = cnt / lpb2;
                const uint32_t rem2 = cnt - full2 * lpb2;
                const float4 *p2 = lst + base + qs2;
                float gx2[1] = {0.f}, gy2[1] = {0.f}, gz2[1] = {0.f};
                const float qx[1] = {rx2}, qy[1] = {ry2}, qz[1] = {rz2};
                switch (lpb2) {  // the second pass's common strides (32, 21 or 16 bodies)
                case 2: flush_share<2, 1>(p2, full2, qx, qy, qz, eps2, gx2, gy2, gz2); break;
                case 3: flush_share<3, 1>(p2, full2, qx, qy, qz, eps2, gx2, gy2, gz2); break;
                case 4: flush_share<4, 1>(p2, full2, qx, qy, qz, eps2, gx2, gy2, gz2); break;
                default:
                    flush_share_rt(p2, lpb2, full2, rx2, ry2, rz2, eps2, gx2[0], gy2[0], gz2[0]);
                    break;
                }
                if (rem2) {
                    const float4 e = p2[full2 * lpb2];
                    pair_f32(qs2 < rem2 ? e : far_entry(), rx2, ry2, rz2, eps2, gx2[0], gy2[0],
                             gz2[0]);
                }
                acc2_x += (double)gx2[0];
                acc2_y += (double)gy2[0];
                acc2_z += (double)gz2[0];
            }
            n_inter += cnt;
        };

        // Quadrupole cells qlst[base .. base + cnt), shared out over the lanes
        // of a body as in flush.
        auto qflush = [&](uint32_t base, uint32_t cnt) {
            const uint32_t full = cnt / lpb;
            const uint32_t rem = cnt - full * lpb;
            const float4 *p = qlst + base + qs;
            const uint32_t *pk = qk + base + qs;
            float fx = 0.f, fy = 0.f, fz = 0.f;
            switch (lpb) {
            case 1: qflush_share<1>(p, pk, 1, full, gquad, rx[0], ry[0], rz[0], eps2, fx, fy, fz); break;
            case 2: qflush_share<2>(p, pk, 2, full, gquad, rx[0], ry[0], rz[0], eps2, fx, fy, fz); break;
            case 4: qflush_share<4>(p, pk, 4, full, gquad, rx[0], ry[0], rz[0], eps2, fx, fy, fz); break;
            case 8: qflush_share<8>(p, pk, 8, full, gquad, rx[0], ry[0], rz[0], eps2, fx, fy, fz); break;
            case 16: qflush_share<16>(p, pk, 16, full, gquad, rx[0], ry[0], rz[0], eps2, fx, fy, fz); break;
            case 32: qflush_share<32>(p, pk, 32, full, gquad, rx[0], ry[0], rz[0], eps2, fx, fy, fz); break;
            case 64: qflush_share<64>(p, pk, 64, full, gquad, rx[0], ry[0], rz[0], eps2, fx, fy, fz); break;
            default: qflush_share<0>(p, pk, lpb, full, gquad, rx[0], ry[0], rz[0], eps2, fx, fy, fz); break;
            }
            if (rem) {
                // shares past the remainder take a zero-force entry with a zero
                // quadrupole (a far entry with a real Q would give inf * 0)
                const bool real = qs < rem;
                const uint32_t c = real ? pk[full * lpb] : 0u;
                const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
                const float4 qa = gquad[2ull * c], qb = gquad[2ull * c + 1];
                pair_quad(real ? p[full * lpb] : far_entry(), real ? qa : zero, real ? qb : zero,
                          rx[0], ry[0], rz[0], eps2, fx, fy, fz);
            }
            acc_x[0] += (double)fx;
            acc_y[0] += (double)fy;
            acc_z[0] += (double)fz;
            n_inter += cnt;
            nquad += cnt * s;
        };

        // learned correction of cells cl[base .. base+cnt) (cnt <= 16) for every body
        auto corr_flush = [&](uint32_t base, uint32_t cnt) {
            const int g = (int)(lane >> 4), p = (int)(lane & 15);
            const bool pv = (uint32_t)p < cnt;
            const float4 ce = cl_e[base + p];
            MlpCell mc{};
            if (pv) mc = corr.mcell[cl_k[base + p]];
            const float e2c = mc.c.z * mc.c.z;
            ncorr += cnt * s;
            bf16x4 zero4;
            for (int i = 0; i < 4; ++i) zero4[i] = (__bf16)0.f;
            for (uint32_t b = 0; b < s; ++b) {
                const float4 bo = boff[b];
                float inv_d;
                bf16x4 xin = mlp_features(ce.x - bo.x, ce.y - bo.y, ce.z - bo.z, mc, g, inv_d);
                if (!pv) xin = zero4;
                MlpActs act;
                const f32x4 yv = mlp_forward_tile(w, xin, act);
                const float inv2 = inv_d * inv_d;
                const float sc = (pv && g == 0) ? ce.w * e2c * (inv2 * inv2) : 0.f;
                float cx = yv[0] * sc, cy = yv[1] * sc, cz = yv[2] * sc;
                for (int off = 8; off >= 1; off >>= 1) {
                    cx += __shfl_xor(cx, off, 64);
                    cy += __shfl_xor(cy, off, 64);
                    cz += __shfl_xor(cz, off, 64);
                }
                if (lane == 0) {
                    float4 t = bcorr[b];
                    t.x += cx;
                    t.y += cy;
                    t.z += cz;
                    bcorr[b] = t;
                }
            }
        };

        // A node goes to the list (accepted cell, or body leaf: exact pair, the
        // self pair adds 0) or is opened (cell failing the MAC); an empty slot
        // does neither.  d2 = squared distance to the group box.  Computed for
        // every lane without branches: an empty slot's values are unused.
        auto classify = [&](const NodeF32 &r, int depth, float4 &entry, float &d2,
                            bool &to_list, bool &to_open) {
            const float dx = (r.x - gxh) + (r.lx - gxl);
            const float dy = (r.y - gyh) + (r.ly - gyl);
            const float dz = (r.z - gzh) + (r.lz - gzl);
            entry = make_float4(dx, dy, dz, r.gm);
            const float ex = fmaxf(fabsf(dx) - hx, 0.f);
            const float ey = fmaxf(fabsf(dy) - hy, 0.f);
            const float ez = fmaxf(fabsf(dz) - hz, 0.f);
            d2 = fmaf(ex, ex, fmaf(ey, ey, ez * ez));
            // (edge / theta)^2 = ro2_root 4^-depth, exact (a power-of-two
            // scaling); computed rather than read from an LDS table, which
            // put an LDS round trip on every walk step's chain of waits
            const bool far_enough = d2 > ldexpf(ro2_root, -2 * depth);
            const bool cell = r.ref >= 0;
            to_list = r.ref != kRefEmpty && (!cell || far_enough);
            to_open = cell && !far_enough;
        };

        {
            float4 e;
            float d2r;
            const NodeF32 root = rec[0];
            // every lane evaluates the root alike
            bool rl, ro;
            classify(root, 0, e, d2r, rl, ro);
            const int cls = (int)wave_uniform(rl ? 1u : (ro ? 2u : 0u));
            if (cls == 1) {
                if (lane == 0) lst[0] = e;
                ln = 1;
                if constexpr (kCorr) {
                    if (wave_uniform(root.ref >= 0 && e2_root > corr.tau2 * d2r)) {
                        if (lane == 0) {
                            cl_e[0] = e;
                            cl_k[0] = (uint32_t)root.ref;
                        }
                        cn = 1;
                    }
                }
            } else if (cls == 2) {
                if (lane == 0) stk[0] = ((uint32_t)root.ref << 6);
                sp = 1;
            }
            __syncthreads();
        }

        // Pop up to 8 kPop cells and load this lane's kPop child records
        // (child lane & 7 of the cells lane >> 3, + 8, + 16, ...): the kPop
        // loads of a lane are in flight together, so a walk waits on memory
        // once per kPop batches of cells instead of once per batch.  Every
        // lane loads (a lane without a cell reads a child of cell 0 and is
        // marked idle): a load under a branch would make the compiler wait
        // for it at the branch's end, before the list evaluation that is
        // meant to hide it.
        NodeF32 r[kPop];
        int depth[kPop];
        bool live[kPop];
        auto pop_and_load = [&]() -> uint32_t {
            const uint32_t take = sp < 8u * kPop ? sp : 8u * kPop;
            sp -= take;
#pragma unroll
            for (int k = 0; k < kPop; ++k) {
                const uint32_t c = (lane >> 3) + 8u * (uint32_t)k;
                live[k] = c < take;
                const uint32_t entry = live[k] ? stk[sp + c] : 0u;
                depth[k] = (int)(entry & 63u) + 1;
                r[k] = rec[1ull + 8ull * (entry >> 6) + (lane & 7u)];
            }
            __syncthreads();
            return take;
        };

        // A correct octree opens every internal cell at most once per group,
        // so icap iterations bound the walk; the cap turns a corrupt tree into
        // an error instead of an endless loop.
        uint32_t budget = icap + 16;
        uint32_t take = sp > 0 ? pop_and_load() : 0u;
        while (take > 0) {
            if (budget-- == 0) {
                overflow = true;
                break;
            }
#pragma unroll
            for (int k = 0; k < kPop; ++k) {
                float4 e;
                float d2;
                bool to_list, to_open;
                classify(r[k], depth[k], e, d2, to_list, to_open);
                to_list = to_list && live[k];
                to_open = to_open && live[k];
                if constexpr (kQuad) {
                    // accepted cells to the quadrupole list, body leaves stay
                    const bool tq = to_list && r[k].ref >= 0;
                    const uint64_t bq = __ballot(tq);
                    if (tq) {
                        const uint32_t p = qn + count_below(bq);
                        qlst[p] = e;
                        qk[p] = (uint32_t)r[k].ref;
                    }
                    qn += __popcll(bq);  // < chunk before: at most kListCap - 1 after
                    to_list = to_list && !tq;
                }
                const uint64_t bl = __ballot(to_list);
                const uint64_t bo = __ballot(to_open);
                if (to_list) lst[ln + count_below(bl)] = e;
                if (to_open) {
                    const uint32_t p = sp + count_below(bo);
                    if (p < kStackCap) stk[p] = ((uint32_t)r[k].ref << 6) | (uint32_t)depth[k];
                }
                if constexpr (kCorr) {
                    const bool cc = to_list && r[k].ref >= 0 &&
                                    ldexpf(e2_root, -2 * depth[k]) > corr.tau2 * d2;
                    const uint64_t bc = __ballot(cc);
                    if (cc) {
                        const uint32_t p = cn + count_below(bc);
                        cl_e[p] = e;
                        cl_k[p] = (uint32_t)r[k].ref;
                    }
                    cn += __popcll(bc);  // < kCorrTile before: at most kCellCap - 1 after
                }
                ln += __popcll(bl);  // < chunk <= kFlushSpan before: at most kListCap - 1 after
                sp += __popcll(bo);
            }
            peak = sp > peak ? sp : peak;
            if (sp > kStackCap) {
                overflow = true;
                break;
            }
            __syncthreads();
            // issue the next loads; the list evaluation below hides their latency
            take = sp > 0 ? pop_and_load() : 0u;
            if (ln >= chunk) {
                uint32_t done = 0;
                for (; ln - done >= chunk; done += chunk) flush(done, chunk);
                __syncthreads();
                const uint32_t rest = ln - done;  // < chunk <= done: no overlap
                for (uint32_t i = lane; i < rest; i += kGroup) lst[i] = lst[done + i];
                ln = rest;
                __syncthreads();
            }
            if constexpr (kQuad) {
                if (qn >= chunk) {
                    uint32_t done = 0;
                    for (; qn - done >= chunk; done += chunk) qflush(done, chunk);
                    __syncthreads();
                    const uint32_t rest = qn - done;  // < chunk <= done: no overlap
                    for (uint32_t i = lane; i < rest; i += kGroup) {
                        qlst[i] = qlst[done + i];
                        qk[i] = qk[done + i];
                    }
                    qn = rest;
                    __syncthreads();
                }
            }
            if constexpr (kCorr) {
                if (cn >= (uint32_t)kCorrTile) {
                    uint32_t base = 0;
                    for (; cn - base >= (uint32_t)kCorrTile; base += kCorrTile)
                        corr_flush(base, kCorrTile);
                    __syncthreads();
                    const uint32_t rest = cn - base;
                    if (lane < rest) {
                        cl_e[lane] = cl_e[base + lane];
                        cl_k[lane] = cl_k[base + lane];
                    }
                    cn = rest;
                    __syncthreads();
                }
            }
        }
        if (ln > 0) flush(0, ln);
        if constexpr (kQuad) {
            if (qn > 0) qflush(0, qn);
        }
        if constexpr (kCorr) {
            if (cn > 0) corr_flush(0, cn);
        }
        __syncthreads();
        // add up the list shares of each body (fixed order: deterministic)
        if (pow2) {
            for (uint32_t off = ss; off < (uint32_t)kGroup; off <<= 1) {
                acc_x[0] += __shfl_xor(acc_x[0], off, 64);
                acc_y[0] += __shfl_xor(acc_y[0], off, 64);
                acc_z[0] += __shfl_xor(acc_z[0], off, 64);
            }
        } else {
            // body sub's shares sit in lanes sub + j ss, j < lpb; lane sub adds them
            double tx = acc_x[0], ty = acc_y[0], tz = acc_z[0];
            for (uint32_t j = 1; j < lpb; ++j) {
                const int src = (int)(sub + j * ss);
                tx += __shfl(acc_x[0], src, 64);
                ty += __shfl(acc_y[0], src, 64);
                tz += __shfl(acc_z[0], src, 64);
            }
            acc_x[0] = tx;
            acc_y[0] = ty;
            acc_z[0] = tz;
        }
        if (kTwoPass && sb) {
            // body sa + sub2's shares sit in lanes sub2 + j sb, j < lpb2; lane sub2 adds them
            double tx = acc2_x, ty = acc2_y, tz = acc2_z;
            for (uint32_t j = 1; j < lpb2; ++j) {
                const int src = (int)(sub2 + j * sb);
                tx += __shfl(acc2_x, src, 64);
                ty += __shfl(acc2_y, src, 64);
                tz += __shfl(acc2_z, src, 64);
            }
            acc2_x = tx;
            acc2_y = ty;
            acc2_z = tz;
        }
        ncorr_out += ncorr;
        nquad_out += nquad;
        // Stored also after an overflow (the caller reports it and the values
        // are then undefined): a predicate holding `overflow` would let the
        // compiler route the storing lanes past the caller's exit test, a
        // per-lane split of the wave's loop.
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            if (valid[b] && q == 0) {
                if constexpr (kCorr) {
                    const float4 c = bcorr[sub + (uint32_t)b * kGroup];
                    acc_x[b] += (double)c.x;
                    acc_y[b] += (double)c.y;
                    acc_z[b] += (double)c.z;
                }
                ax[bi[b]] = acc_x[b];
                ay[bi[b]] = acc_y[b];
                az[bi[b]] = acc_z[b];
                if (inter) inter[bi[b]] = n_inter;
            }
        }
        if (kTwoPass && sb && q2 == 0) {  // lanes 0 .. sb - 1
            if constexpr (kCorr) {
                const float4 c = bcorr[sa + sub2];
                acc2_x += (double)c.x;
                acc2_y += (double)c.y;
                acc2_z += (double)c.z;
            }
            ax[bi2] = acc2_x;
            ay[bi2] = acc2_y;
            az[bi2] = acc2_z;
            if (inter) inter[bi2] = n_inter;
        }
    }
}

// Forces on the bodies of one group grp = {first sorted position, count}
// (checked by the caller): one body per lane up to 64 bodies, two beyond.
template <bool kCorr, bool kQuad = false>
__device__ __forceinline__ void group_walk(const GroupTree &T, uint2 grp, float eps2,
                                           const CorrArgs &corr, const MlpForward &w,
                                           const GroupLds &L, uint32_t &peak, bool &overflow,
                                           uint32_t &ncorr_out, uint32_t &nquad_out) {
    const uint32_t g0 = wave_uniform(grp.x);
    const uint32_t s = wave_uniform(grp.y);
    if constexpr (kGroupMax > (uint32_t)kGroup && !kQuad) {
        if (s > (uint32_t)kGroup) {
            group_walk_n<kCorr, 2, false>(T, g0, s, eps2, corr, w, L, peak, overflow, ncorr_out,
                                          nquad_out);
            return;
        }
    }
    group_walk_n<kCorr, 1, kQuad>(T, g0, s, eps2, corr, w, L, peak, overflow, ncorr_out,
                                  nquad_out);
}

// a group {first, count} that a walk may trust
__device__ inline bool group_ok(uint2 grp, uint32_t n) {
    return grp.y != 0 && grp.y <= kGroupLimit && grp.x < n && grp.y <= n - grp.x;
}

// Before a traversal: reset the group queue, and order the last groups of
// each XCD's chunk (kTailGroups, at most two thirds of the chunk: sorting all
// of it scatters the walks that share L2 lines) by decreasing estimated cost,
// a group's size times the list length the previous traversal recorded for
// its first body.  The walks that end the launch are then the shortest
// instead of whichever groups come last in octree order (on a 1M-body disk
// the slowest waves ended 200 us after the queue ran dry, a fifth of the
// launch).  A counting sort by cost class (8 classes per factor of two, 256
// in all) in LDS; within a class the order is that of the LDS atomics.  Only
// the order in which groups start changes: each group's forces are the same.
// Without recorded lengths (all zero) the order stays.  One workgroup per
// chunk.
constexpr uint32_t kTailGroups = 4096;
constexpr int kTailThreads = 1024;
constexpr uint32_t kCostClasses = 256;
__device__ inline uint32_t cost_class(uint32_t v) {  // decreasing in v; 0 -> last class
    if (v == 0) return kCostClasses - 1;
    const uint32_t e = 31u - (uint32_t)__clz(v);  // floor(log2 v)
    const uint32_t f = e >= 3 ? (v >> (e - 3)) & 7u : (v << (3 - e)) & 7u;
    return kCostClasses - 2 - min(8 * e + f, kCostClasses - 2);
}
__global__ void __launch_bounds__(kTailThreads) k_group_queue_prepare(
    TreeHdr *h, uint32_t *gq, uint32_t n, uint2 *groups, const uint32_t *__restrict__ sidx,
    const uint32_t *__restrict__ inter) {
    __shared__ uint2 grp[kTailGroups];
    __shared__ uint8_t cls[kTailGroups];
    __shared__ uint32_t hist[kCostClasses], fill[kCostClasses];
    const uint32_t t = threadIdx.x, c = blockIdx.x;  // c: chunk (and XCD) index
    if (c == 0 && t == 0) {
        h->group_next = 0;
        h->corr_pairs = 0;
        h->quad_pairs = 0;
    }
    if (t == 0) gq[c * kQueueStride] = 0;
    if (!inter) return;
    const uint32_t ngroups = min(h->group_count, n);  // the traversal's chunk bounds
    const uint32_t lo = (uint32_t)((uint64_t)ngroups * c / kXcds);
    const uint32_t hi = (uint32_t)((uint64_t)ngroups * (c + 1) / kXcds);
    const uint32_t m = min(2 * (hi - lo) / 3, kTailGroups);
    if (m < 2) return;  // the same for the whole workgroup
    const uint32_t base = hi - m;
    for (uint32_t b = t; b < kCostClasses; b += kTailThreads) hist[b] = fill[b] = 0;
    __syncthreads();
    for (uint32_t i = t; i < m; i += kTailThreads) {
        const uint2 g = groups[base + i];
        grp[i] = g;
        uint32_t cost = 0;  // a group the walk would reject keeps cost 0
        if (group_ok(g, n)) {
            const uint64_t v = (uint64_t)g.y * inter[sidx[g.x]];
            cost = v < 0xffffffffull ? (uint32_t)v : 0xffffffffu;
        }
        const uint32_t k = cost_class(cost);
        cls[i] = (uint8_t)k;
        atomicAdd(&hist[k], 1u);
    }
    __syncthreads();
    if (hist[kCostClasses - 1] == m) return;  // no recorded lengths: keep the order
    if (t == 0) {  // exclusive prefix of the classes
        uint32_t run = 0;
        for (uint32_t b = 0; b < kCostClasses; ++b) {
            const uint32_t v = hist[b];
            hist[b] = run;
            run += v;
        }
    }
    __syncthreads();
    for (uint32_t i = t; i < m; i += kTailThreads) {
        const uint32_t k = cls[i];
        groups[base + hist[k] + atomicAdd(&fill[k], 1u)] = grp[i];
    }
}

// At most 96 VGPRs, five waves per SIMD, for the monopole and quadrupole walks
// (their two-pass flushes would otherwise take 103 and leave four; measured:
// 3 % faster on the 4M Plummer sphere, a forced six waves spill and lose
// 10 %).  The learned correction's walks hold the network's weights in
// registers and stay at one wave: the compiler's note that it cannot meet the
// target there is expected.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Wpass-failed"
template <bool kCorr, bool kQuad>
__global__ void __launch_bounds__(kGroup) __attribute__((amdgpu_waves_per_eu(5))) k_bh_group(
    uint32_t n, const uint32_t *__restrict__ sidx, const double *__restrict__ x,
    const double *__restrict__ y, const double *__restrict__ z, const double *__restrict__ m,
    const NodeF32 *__restrict__ rec, const uint2 *__restrict__ groups, double theta,
    float eps2, uint32_t icap, double *ax, double *ay, double *az, uint32_t *inter,
    TreeHdr *h, uint32_t *gq, CorrArgs corr, const float4 *__restrict__ gquad) {
    __shared__ uint32_t stk[kStackCap];
    __shared__ float4 lst[kListCap];
    __shared__ float4 qlst[kQuad ? kListCap : 1];
    __shared__ uint32_t qk[kQuad ? kListCap : 1];
    __shared__ float4 cl_e[kCorr ? kCellCap : 1];
    __shared__ uint32_t cl_k[kCorr ? kCellCap : 1];
    // bcorr is cleared lane by lane (lane + 64 b): at least one wave of entries
    constexpr uint32_t kCorrSlots = kGroupMax > (uint32_t)kGroup ? kGroupMax : (uint32_t)kGroup;
    __shared__ float4 boff[kCorr ? kGroupLimit : 1];
    __shared__ float4 bcorr[kCorr ? kCorrSlots : 1];
    const GroupLds L{stk, lst, qlst, qk, cl_e, cl_k, boff, bcorr};
    const uint32_t lane = threadIdx.x;
    const uint32_t ngroups = min(h->group_count, n);
    // (edge/theta)^2 of the root; a child at depth d uses ro2_root * 4^-d
    const double ro_root = h->edge / theta;
    const GroupTree T{n, sidx, x, y, z, m, rec, icap, (float)(ro_root * ro_root),
                      (float)(h->edge * h->edge), ax, ay, az, inter, gquad};
    MlpForward w;
    if constexpr (kCorr) w.load(corr.pack, corr.master, (int)lane);
    uint32_t peak = 0, ncorr = 0, nquad = 0;
    bool overflow = false;

    // Groups come in octree order: waves running at the same time walk
    // neighbouring groups, whose interaction lists overlap, so the records
    // they read are shared in L2.
    //
    // The list is cut into kXcds contiguous chunks, one per XCD: workgroup b
    // runs on XCD b mod kXcds, so the waves of one XCD walk one region of the
    // tree and its records stay in that XCD's L2.  A wave whose chunk is empty
    // goes on with the next chunks, so the XCDs finish together.  The chunk
    // counters sit in separate cache lines.
    uint32_t c = blockIdx.x % kXcds, visited = 0;
    for (;;) {
        const uint32_t lo = (uint32_t)((uint64_t)ngroups * c / kXcds);
        const uint32_t hi = (uint32_t)((uint64_t)ngroups * (c + 1) / kXcds);
        uint32_t slot = 0;
        if (lane == 0) {
            uint32_t *q = gq + c * kQueueStride;
            slot = __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (slot < hi - lo)  // no read-modify-write once the chunk is done
                slot = __hip_atomic_fetch_add(q, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        const uint32_t k = lane0_uniform(slot);
        if (k >= hi - lo) {
            if (++visited == kXcds) break;
            c = c + 1 == kXcds ? 0u : c + 1;
            continue;
        }
        const uint2 grp = groups[lo + k];
        if (!group_ok(grp, n)) {
            overflow = true;  // corrupt group table: report instead of reading out of bounds
            break;
        }
        group_walk<kCorr, kQuad>(T, grp, eps2, corr, w, L, peak, overflow, ncorr, nquad);
        if (overflow) break;
    }
    if constexpr (kCorr) {
        if (lane == 0 && ncorr) atomicAdd(&h->corr_pairs, (unsigned long long)ncorr);
    }
    if constexpr (kQuad) {
        if (lane == 0 && nquad) atomicAdd(&h->quad_pairs, (unsigned long long)nquad);
    }
    if (overflow) raise_flag(h, kFlagStack);
    if (lane == 0) raise_max(&h->stack_peak, peak);
}
#pragma clang diagnostic pop

// ---- ensemble of independent systems -------------------------------------------
__global__ void __launch_bounds__(64) k_ens_items(uint32_t nq, const uint32_t *__restrict__ qorder,
                                                  const uint32_t *__restrict__ items,
                                                  uint32_t *item_off, uint32_t *cursor,
                                                  uint32_t *status) {
    const uint32_t lane = threadIdx.x;
    uint32_t run = 0;
    for (uint32_t q0 = 0; q0 < nq; q0 += 64) {
        const uint32_t q = q0 + lane;
        const uint32_t c = q < nq ? items[qorder[q]] : 0u;
        uint32_t inc = c;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t v = __shfl_up(inc, d, 64);
            if (lane >= (uint32_t)d) inc += v;
        }
        if (q < nq) item_off[q] = run + inc - c;
        run += __shfl(inc, 63, 64);
    }
    if (lane == 0) item_off[nq] = run;
    if (lane < kXcds) cursor[lane * kQueueStride] = 0;
    (void)status;
}

// Direct sum for targets [tile*64*TPL, (tile+1)*64*TPL) of one system, TPL
// per lane: FP32 pairs on offsets from the tile's first body (FP64
// subtraction, so nearby pairs keep their precision; a body's own offset
// equals its source offset, so the self pair adds exactly 0), FP64 sum of each
// 64-source chunk.  Two targets per lane halve the LDS reads per pair.
template <int TPL>
__device__ inline void direct_tile(const double *__restrict__ x, const double *__restrict__ y,
                                   const double *__restrict__ z, const double *__restrict__ m,
                                   uint32_t n, uint32_t tile, double G, float eps2, double *ax,
                                   double *ay, double *az, uint32_t *inter, float4 *stage) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t t0 = tile * kEnsTile * TPL;
    const double rx = x[t0], ry = y[t0], rz = z[t0];
    float px[TPL], py[TPL], pz[TPL];
    double acc_x[TPL], acc_y[TPL], acc_z[TPL];
#pragma unroll
    for (int q = 0; q < TPL; ++q) {
        const uint32_t i = t0 + lane + (uint32_t)q * kEnsTile;
        const uint32_t ii = i < n ? i : t0;
        px[q] = (float)(x[ii] - rx);
        py[q] = (float)(y[ii] - ry);
        pz[q] = (float)(z[ii] - rz);
        acc_x[q] = acc_y[q] = acc_z[q] = 0.0;
    }
    for (uint32_t c = 0; c < n; c += kEnsTile) {
        const uint32_t j = c + lane;
        float4 sv = make_float4(0.f, 0.f, 0.f, 0.f);
        if (j < n)
            sv = make_float4((float)(x[j] - rx), (float)(y[j] - ry), (float)(z[j] - rz),
                             (float)(G * m[j]));
        __syncthreads();
        stage[lane] = sv;
        __syncthreads();
        const uint32_t cnt = min(kEnsTile, n - c);
        float fx[TPL], fy[TPL], fz[TPL];
#pragma unroll
        for (int q = 0; q < TPL; ++q) fx[q] = fy[q] = fz[q] = 0.f;
        for (uint32_t k = 0; k < cnt; ++k) {
            const float4 e = stage[k];
#pragma unroll
            for (int q = 0; q < TPL; ++q) pair_f32(e, px[q], py[q], pz[q], eps2, fx[q], fy[q], fz[q]);
        }
#pragma unroll
        for (int q = 0; q < TPL; ++q) {
            acc_x[q] += (double)fx[q];
            acc_y[q] += (double)fy[q];
            acc_z[q] += (double)fz[q];
        }
    }
#pragma unroll
    for (int q = 0; q < TPL; ++q) {
        const uint32_t i = t0 + lane + (uint32_t)q * kEnsTile;
        if (i < n) {
            ax[i] = acc_x[q];
            ay[i] = acc_y[q];
            az[i] = acc_z[q];
            inter[i] = n;
        }
    }
}

// Persistent: every wave takes items from the queue until it is empty.  As in
// k_bh_group the queue is cut into one contiguous chunk per XCD (the items of a
// system follow each other, so its tree stays in one L2) and a wave goes on with
// the next chunk when its own is empty, and 96 VGPRs leave five waves per
// SIMD (the walk's constants of a system do not all fit: 6 VGPRs and 28 SGPRs are spilled,
// 28 bytes of scratch).  One queue, four waves per SIMD and no VGPR spilled before; forces
// of a step, ms, before and now: 24 systems (0.4 million bodies) 0.634 and 0.555, 128 (1.9
// million) 1.72 and 1.69, 512 (8.0 million) 6.75 and 6.66.
__global__ void __launch_bounds__(kGroup) __attribute__((amdgpu_waves_per_eu(5)))
k_ens_forces(EnsForceArgs a) {
    __shared__ uint32_t stk[kStackCap];
    __shared__ float4 lst[kListCap];
    const GroupLds L{stk, lst, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
    const uint32_t lane = threadIdx.x;
    const uint32_t total = a.item_off[a.nq];
    const MlpForward w{};
    const CorrArgs corr{};
    uint32_t peak = 0, ncorr = 0, nquad = 0;
    bool overflow = false;
    // the queue position of the last item: items of one system follow each other
    uint32_t lo = 0, pb = 0, pe = 0;
    uint32_t c = blockIdx.x % kXcds, visited = 0;
    for (;;) {
        const uint32_t clo = (uint32_t)((uint64_t)total * c / kXcds);
        const uint32_t chi = (uint32_t)((uint64_t)total * (c + 1) / kXcds);
        uint32_t slot = 0;
        if (lane == 0) {
            uint32_t *q = a.cursor + c * kQueueStride;
            slot = __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (slot < chi - clo)
                slot = __hip_atomic_fetch_add(q, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        const uint32_t k = lane0_uniform(slot);
        if (k >= chi - clo) {
            if (++visited == kXcds) break;
            c = c + 1 == kXcds ? 0u : c + 1;
            continue;
        }
        const uint32_t it = clo + k;
        if (it < pb || it >= pe) {
            // queue position q with item_off[q] <= it < item_off[q + 1]
            uint32_t hi = a.nq;
            lo = 0;
            while (hi - lo > 1) {
                const uint32_t mid = (lo + hi) >> 1;
                if (a.item_off[mid] <= it) lo = mid;
                else hi = mid;
            }
            pb = a.item_off[lo];
            pe = a.item_off[lo + 1];
        }
        const uint32_t s = a.qorder[lo];
        const EnsSystem S = a.sys[s];
        const uint32_t local = it - pb;
        const uint32_t bo = S.body_off;
        if (S.bh) {
            const double edge = a.fb.hdr[s].edge;
            const double ro = edge / a.theta;
            const GroupTree T{S.n, a.fb.sidx + S.fb_off, a.x + bo, a.y + bo, a.z + bo, a.m + bo,
                              a.fb.rec + S.node_off, S.icap, (float)(ro * ro),
                              (float)(edge * edge), a.ax + bo, a.ay + bo, a.az + bo,
                              a.inter + bo, nullptr};
            const uint2 grp = a.fb.groups[S.fb_off + local];
            if (!group_ok(grp, S.n)) {
                overflow = true;
                break;
            }
            group_walk<false>(T, grp, a.eps2, corr, w, L, peak, overflow, ncorr, nquad);
            if (overflow) break;
        } else if (a.direct_tpl == 2) {
            direct_tile<2>(a.x + bo, a.y + bo, a.z + bo, a.m + bo, S.n, local, a.G, a.eps2,
                           a.ax + bo, a.ay + bo, a.az + bo, a.inter + bo, lst);
        } else {
            direct_tile<1>(a.x + bo, a.y + bo, a.z + bo, a.m + bo, S.n, local, a.G, a.eps2,
                           a.ax + bo, a.ay + bo, a.az + bo, a.inter + bo, lst);
        }
    }
    if (overflow && lane == 0) atomicOr(a.status, kFlagStack);
}

}  // namespace

void launch_direct_targets_f64(uint32_t n, const double *x, const double *y, const double *z,
                               const double *m, double G, double eps2, uint32_t nt,
                               const uint32_t *targets, double *ax, double *ay, double *az,
                               hipStream_t s) {
    if (nt == 0) return;
    // A round of workgroups is one of 64 targets or two of 16 per CU (1024
    // threads each), and a round of 16-target ones takes 0.6 of the other's time
    // (0.139 ms for 8192 targets x sources against 0.223) and leaves a shorter
    // remainder.
    const uint32_t rounds = ceil_div(nt, 64 * kCus);
    const bool small = 0.6 * std::max(1.0, nt / (2.0 * 16 * kCus)) < rounds;
    const dim3 block(kF64Threads);
    if (small)
        hipLaunchKernelGGL(k_direct_f64<16>, dim3(ceil_div(nt, 16)), block, 0, s, n, x, y, z, m, G,
                           eps2, nt, targets, ax, ay, az);
    else
        hipLaunchKernelGGL(k_direct_f64<64>, dim3(ceil_div(nt, 64)), block, 0, s, n, x, y, z, m, G,
                           eps2, nt, targets, ax, ay, az);
}

void launch_direct_f64(uint32_t n, const double *x, const double *y, const double *z,
                       const double *m, double G, double eps2, double *ax, double *ay,
                       double *az, hipStream_t s) {
    launch_direct_targets_f64(n, x, y, z, m, G, eps2, n, nullptr, ax, ay, az, s);
}

namespace {
// How a split direct sum of n bodies is cut.
struct SplitPlan {
    uint32_t per_lane;  // targets per lane
    uint32_t tiles;     // blocks of 64 per_lane targets
    uint32_t splits;    // source ranges
    uint32_t chunk;     // sources per range
};
// Small sums are cut as finely as the kernels allow (one run or stage per wave
// and, FP32, one target per lane), to have as many waves as they can: FP32
// 0.013 ms for 1024 bodies, 0.0175 for 3001 and 0.051 for 12,001 with the reduction
// (two targets per lane 0.024, 0.027 and 0.059; blocks of 512 targets and 256
// sources 0.027, 0.050 and 0.081); at 16,384 both were alike, beyond, two targets per lane
// faster (50,021: 0.703 against 0.725).  Figures of the alternatives are those of
// stages that went through scratch memory, 3 to 7 % slower than now.
SplitPlan split_plan(bool fp64, uint32_t n) {
    SplitPlan p;
    p.per_lane = fp64 ? (uint32_t)kF64fPerLane : (n < 16384 ? 1u : 2u);
    p.tiles = ceil_div(n, 64 * p.per_lane);
    const uint32_t step = kSplitTile * kSplitWaves * (fp64 ? 1u : (uint32_t)kF32cRun);
    const uint32_t least = fp64 && n >= 8192 ? 2 * step : step;
    const uint32_t most = kSplitPartials / (p.tiles * 64 * p.per_lane);
    p.splits = std::max<uint32_t>(1, std::min(most, ceil_div(n, least)));
    p.chunk = ceil_div(ceil_div(n, p.splits), step) * step;
    p.splits = ceil_div(n, p.chunk);
    return p;
}
}  // namespace

// scratch: the partial sums [split][3][n] doubles (none with one split)
uint64_t direct_split_scratch_bytes(uint32_t n) {
    const uint32_t splits = std::max(split_plan(false, n).splits, split_plan(true, n).splits);
    return splits > 1 ? 3ull * n * splits * sizeof(double) : 0;
}

void launch_direct_split(bool fp64, uint32_t n, const double *x, const double *y,
                         const double *z, const double *m, double G, double eps2, double *ax,
                         double *ay, double *az, double *partial, hipStream_t s) {
    if (n == 0) return;
    const SplitPlan p = split_plan(fp64, n);
    const dim3 grid(p.tiles, p.splits), block(kSplitThreads);
    if (fp64)
        hipLaunchKernelGGL(k_direct_f64f, grid, block, 0, s, n, x, y, z, m, G, eps2, p.chunk,
                           partial, ax, ay, az);
    else if (p.per_lane == 1)
        hipLaunchKernelGGL(k_direct_f32c<1>, grid, block, 0, s, n, x, y, z, m, G, (float)eps2,
                           p.chunk, partial, ax, ay, az);
    else
        hipLaunchKernelGGL(k_direct_f32c<2>, grid, block, 0, s, n, x, y, z, m, G, (float)eps2,
                           p.chunk, partial, ax, ay, az);
    if (p.splits > 1)
        hipLaunchKernelGGL(k_split_reduce, dim3(ceil_div(n, kSplitThreads), 3), block, 0, s, n,
                           p.splits, fp64 ? G : 1.0, (const double *)partial, ax, ay, az);
}

void launch_bh_exact(const TreeBufs &t, const double *x, const double *y, const double *z,
                     double G, double eps2, double theta, double *ax, double *ay, double *az,
                     uint32_t *interactions, hipStream_t s) {
    // Waves of 64 bodies from 100,000 bodies at theta 0.5 and below, up to
    // 170,000 at theta 0.85 and above: they need fewer instructions per node but
    // leave one wave per 64 bodies, whose visits follow one another, and short
    // walks share less.  Traversal, ms (teams, waves, a stack per lane):
    //   80,001 disk, 0.5      0.80   1.19   1.43
    //   100,003 Plummer, 0.7  1.00   1.02   1.21
    //   100,003 Plummer, 1.05 0.48   0.54   0.55
    //   120,001 Plummer, 0.5  2.41   2.18   2.74
    //   150,001 disk, 1.05    0.35   0.44   0.37
    //   150,001 Plummer, 1.05 0.66   0.63   0.66
    //   180,001 disk, 0.85    0.61   0.64   0.57
    //   180,001 disk, 1.05    0.41   0.45   0.40
    //   180,001 Plummer, 1.05 0.78   0.64   0.68
    //   205,001 disk, 0.7     0.99   0.86   1.01
    //   205,001 disk, 1.05    0.46   0.48   0.43
    //   205,001 Plummer, 1.05 0.89   0.69   0.77
    //   262,144 disk, 0.85    0.86   0.75   0.68
    //   262,144 Plummer, 0.7  2.40   1.42   1.80
    //   300,001 disk, 0.85    0.98   0.82   0.80
    //   300,001 disk, 1.05    0.66   0.59   0.51
    //   400,001 disk, 1.05    0.87   0.68   0.64
    //   500,001 disk, 1.05    1.08   0.81   0.84
    //   600,001 Plummer, 1.05 2.49   1.35   1.54
    //   1,048,576 disk, 1.05  2.27   1.39   1.40
    // The line lies where the two lose as much on a disk as they gain on a Plummer
    // sphere (the sizes alone do not tell these apart).  A stack per lane, 1.2 KB of
    // memory per body, did better on short walks of 170,000 to 500,000 bodies of a disk,
    // whose neighbours share little of them: up to 16 % (300,001, 1.05), and worse
    // on the spheres of that range, by 2 to 17 %.
    const double from = 100e3 + 200e3 * std::min(std::max(theta - 0.5, 0.0), 0.35);
    if (t.n >= from)
        hipLaunchKernelGGL(k_bh_exact_wave, dim3(ceil_div(t.n, 64 * kExactWaves)),
                           dim3(kExactThreads), 0, s, t.n, (const uint32_t *)t.sidx, x, y, z,
                           (const double4 *)t.cm, (const int32_t *)t.ref, G, eps2, theta, t.icap,
                           ax, ay, az, interactions, t.hdr);
    else
        hipLaunchKernelGGL(k_bh_exact_team, dim3(ceil_div(t.n, kTeams * kExactWaves)),
                           dim3(kExactThreads), 0, s, t.n, (const uint32_t *)t.sidx, x, y, z,
                           (const double4 *)t.cm, (const int32_t *)t.ref, G, eps2, theta, t.icap,
                           ax, ay, az, interactions, t.hdr);
}

void launch_bh_group(const TreeBufs &t, const double *x, const double *y, const double *z,
                     const double *m, double eps2, double theta, const float4 *gquad, double *ax,
                     double *ay, double *az, uint32_t *interactions, hipStream_t s) {
    const uint32_t blocks = std::min<uint32_t>(kGroupBlocks, t.n);
    hipLaunchKernelGGL(k_group_queue_prepare, dim3(kXcds), dim3(kTailThreads), 0, s, t.hdr, t.gq,
                       t.n, t.groups, (const uint32_t *)t.sidx, (const uint32_t *)interactions);
    if (gquad)
        hipLaunchKernelGGL((k_bh_group<false, true>), dim3(blocks), dim3(kGroup), 0, s, t.n,
                           (const uint32_t *)t.sidx, x, y, z, m, (const NodeF32 *)t.rec,
                           (const uint2 *)t.groups, theta, (float)eps2, t.icap, ax, ay, az,
                           interactions, t.hdr, t.gq, CorrArgs{}, gquad);
    else
        hipLaunchKernelGGL((k_bh_group<false, false>), dim3(blocks), dim3(kGroup), 0, s, t.n,
                           (const uint32_t *)t.sidx, x, y, z, m, (const NodeF32 *)t.rec,
                           (const uint2 *)t.groups, theta, (float)eps2, t.icap, ax, ay, az,
                           interactions, t.hdr, t.gq, CorrArgs{}, (const float4 *)nullptr);
}

void launch_bh_group_corr(const TreeBufs &t, const double *x, const double *y, const double *z,
                          const double *m, double eps2, double theta, const CorrArgs &corr,
                          const float4 *gquad, double *ax, double *ay, double *az,
                          uint32_t *interactions, hipStream_t s) {
    const uint32_t blocks = std::min<uint32_t>(kGroupBlocks, t.n);
    hipLaunchKernelGGL(k_group_queue_prepare, dim3(kXcds), dim3(kTailThreads), 0, s, t.hdr, t.gq,
                       t.n, t.groups, (const uint32_t *)t.sidx, (const uint32_t *)interactions);
    if (gquad)
        hipLaunchKernelGGL((k_bh_group<true, true>), dim3(blocks), dim3(kGroup), 0, s, t.n,
                           (const uint32_t *)t.sidx, x, y, z, m, (const NodeF32 *)t.rec,
                           (const uint2 *)t.groups, theta, (float)eps2, t.icap, ax, ay, az,
                           interactions, t.hdr, t.gq, corr, gquad);
    else
        hipLaunchKernelGGL((k_bh_group<true, false>), dim3(blocks), dim3(kGroup), 0, s, t.n,
                           (const uint32_t *)t.sidx, x, y, z, m, (const NodeF32 *)t.rec,
                           (const uint2 *)t.groups, theta, (float)eps2, t.icap, ax, ay, az,
                           interactions, t.hdr, t.gq, corr, (const float4 *)nullptr);
}

void launch_ens_items(uint32_t nq, const uint32_t *qorder, const uint32_t *items,
                      uint32_t *item_off, uint32_t *cursor, uint32_t *status, hipStream_t s) {
    hipLaunchKernelGGL(k_ens_items, dim3(1), dim3(64), 0, s, nq, qorder, items, item_off, cursor,
                       status);
}

void launch_ens_forces(const EnsForceArgs &a, uint32_t waves, hipStream_t s) {
    hipLaunchKernelGGL(k_ens_forces, dim3(std::max<uint32_t>(1, waves)), dim3(kGroup), 0, s, a);
}

}  // namespace nb
