// nb_energy.hip -- per-body energy terms for the --energy diagnostics.
//
// Same arithmetic as nBodyAlgorithm.cpp:48-64 (FP64, no softening, i < j
// pairs in index order; compiled with -ffp-contract=off): body j gets
//   E_kin[j] = 0.5 * m_j * (vx^2 + vy^2 + vz^2)
//   E_pot[j] = sum_{i<j} G * m_i * m_j / |p_j - p_i|
// The host adds the terms in body order (nBodyAlgorithm.cpp:71-74).
// O(N^2/2) pair work; every body's sum runs over i = 0, 1, ..., j - 1 in
// order, so the terms are bit-identical to the reference's.
#include <type_traits>

#include "nb_internal.h"

namespace nb {
namespace {

// k_energy_terms: a workgroup of sixteen waves owns 64 bodies j (one per
// lane).  For each chunk of 48 sources the waves compute the terms (three
// sources per wave, read through the scalar cache, interleaved) into one of two
// LDS tiles, and wave 0 adds the previous tile in source order first.  Two
// workgroups per CU (64 VGPRs, 2 more of them spilled; with one workgroup, 131,071
// bodies take 14.4 ms instead of 11.1).
//
// k_energy_rows: a lane computes and adds its body's terms by itself, eight
// interleaved, without the workgroup's barriers and LDS tiles (about 165 cycles
// at 2.4 GHz per 64 pairs, near what the 26 FP64 operations and two
// quarter-rate estimates issue in, against 190-200), but only once there are
// rows enough to balance over the CUs.
//
// One row per lane and one term at a time, as before: 10,000 bodies 1.53 ms
// (bound by the latency of a single term on a few CUs), 131,071 19.6 ms, 300,001
// 59 ms, 1,048,576 560 ms.  Now 0.37, 10.8, 46 and 552 ms (rows at 131,071: 12.5;
// workgroups at 200,001 and 300,001: 25.9 and 57 against 25.0 and 49).
constexpr uint32_t kRowsFrom = 192 * 1024;  // bodies from which the rows are faster
constexpr uint32_t kCus = 256;              // CUs of an MI355X
constexpr int kWaves = 16;
constexpr int kThreads = 64 * kWaves;
constexpr int kTile = 64;             // bodies j per block
constexpr int kPer = 3;               // sources per wave and chunk
constexpr int kChunk = kWaves * kPer;
constexpr int kAhead = 8;             // the adder's LDS reads ahead of its additions
static_assert(kChunk % kAhead == 0, "whole batches per tile");

// |v| in [2^-e, 2^e), on the exponent
__device__ inline bool exponent_within(double v, uint32_t e) {
    return ((uint32_t)__double2hiint(v) & 0x7fffffffu) - ((1023u - e) << 20) < (2u * e << 20);
}

// Block b holds bodies j of tile nb - 1 - b: the triangle's longest sums
// (the last bodies, i < j over almost all of the system) start first, and the
// short ones fill in behind them, so the launch does not end on a few long
// blocks.
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(8)))
k_energy_terms(
    uint32_t n, const double *__restrict__ x, const double *__restrict__ y,
    const double *__restrict__ z, const double *__restrict__ vx, const double *__restrict__ vy,
    const double *__restrict__ vz, const double *__restrict__ m, double G, double *ekin,
    double *epot) {
    __shared__ double term[2][kChunk][kTile];
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t tile = gridDim.x - 1 - blockIdx.x;
    const uint32_t j = tile * kTile + lane;
    const bool valid = j < n;
    const uint32_t jj = valid ? j : 0;
    const double pxj = x[jj], pyj = y[jj], pzj = z[jj], mj = m[jj];
    if (valid && w == kWaves - 1) {
        const double v = vx[j] * vx[j] + vy[j] * vy[j] + vz[j] * vz[j];
        ekin[j] = 0.5 * mj * v;
    }
    double ep = 0;
    auto add_tile = [&](int b) {  // wave 0
        double v[2][kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) v[0][u] = term[b][u][lane];
#pragma unroll
        for (int k = 0; k < kChunk; k += kAhead) {
            const int c = (k / kAhead) & 1;
            if (k + kAhead < kChunk) {
#pragma unroll
                for (int u = 0; u < kAhead; ++u) v[c ^ 1][u] = term[b][k + kAhead + u][lane];
            }
#pragma unroll
            for (int u = 0; u < kAhead; ++u) ep += v[c][u];
        }
    };
    double sx[kPer], sy[kPer], sz[kPer], sm[kPer];
    auto load = [&](uint32_t c) {  // uniform: scalar loads
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            const uint32_t i = min(c + w * kPer + u, n - 1);
            sx[u] = x[i];
            sy[u] = y[i];
            sz[u] = z[i];
            sm[u] = m[i];
        }
    };
    // The numerator G m_i m_j is (G m_i) m_j.  When G m_i and m_j both lie in
    // [2^-150, 2^150), it lies in div_sqrt_core's range and only the squared
    // distance needs checking.
    const bool mj_ok = exponent_within(mj, 150);
    const uint32_t last = min(n, (tile + 1) * kTile);  // bodies i < j of this block
    load(0);
    int buf = 0;
    // kAll: every source of the chunk comes before every body of the block
    auto chunk = [&](uint32_t c, auto kAll) {
        constexpr bool all = decltype(kAll)::value;
        if (w == 0 && c > 0) {
            __builtin_amdgcn_s_setprio(3);
            add_tile(buf ^ 1);
            __builtin_amdgcn_s_setprio(0);
        }
        double a[kPer], v[kPer];
        bool core = mj_ok;
        uint32_t low = 0;
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            const double r_x = pxj - sx[u];
            const double r_y = pyj - sy[u];
            const double r_z = pzj - sz[u];
            const double gm = G * sm[u];
            a[u] = gm * mj;
            v[u] = r_x * r_x + r_y * r_y + r_z * r_z;
            const bool ok = exponent_within(gm, 150) && exponent_within(v[u], 600);
            low = max(low, (uint32_t)__double2loint(v[u]));
            core = core && (ok || (!all && c + w * kPer + u >= j));
        }
        load(c + kChunk);  // back before the barrier waits for it
        if (core && low < kRootOfOnes) {
#pragma unroll
            for (int u = 0; u < kPer; ++u) a[u] = div_sqrt_core(a[u], v[u]);
        } else {
            for (int u = 0; u < kPer; ++u) a[u] = a[u] / sqrt(v[u]);
        }
        // sources at or past j add +0, which changes no sum
#pragma unroll
        for (int u = 0; u < kPer; ++u)
            term[buf][w * kPer + u][lane] = all || c + w * kPer + u < j ? a[u] : 0.0;
        __syncthreads();
        buf ^= 1;
    };
    uint32_t c = 0;
    for (; c + kChunk <= tile * kTile; c += kChunk) chunk(c, std::true_type{});
    for (; c < last; c += kChunk) chunk(c, std::false_type{});
    if (w == 0) {
        add_tile(buf ^ 1);
        if (valid) epot[j] = ep;
    }
}


// A squared distance v lies in [2^-600, 2^600) if distance_off(v) < kDistanceOff:
// v is a sum of squares, so no sign needs masking, and the largest value of
// several terms tests them all (1,048,576 bodies 572 ms with a test per term, 560
// so; 400,000 89 and 83; the workgroup kernel was 3 % slower with it).
constexpr uint32_t kDistanceOff = 1200u << 20;
__device__ inline uint32_t distance_off(double v) {
    return (uint32_t)__double2hiint(v) - ((1023u - 600u) << 20);
}

constexpr int kRowThreads = 256;  // bodies j per block, and sources i per LDS stage
constexpr int kRowPer = 8;        // terms interleaved

// Up to 458,752 bodies all blocks are resident from the start (7 per CU with 68
// VGPRs), dealt round the CUs, so every second round of kCus blocks counts its
// tiles the other way: long and short rows sum up alike on each CU (300,001 bodies:
// 58.7 ms without).  Beyond, the rounds still go from the longest rows to the
// shortest, and blocks that start later fill in behind those that end.
__global__ void __launch_bounds__(kRowThreads) k_energy_rows(
    uint32_t n, const double *__restrict__ x, const double *__restrict__ y,
    const double *__restrict__ z, const double *__restrict__ vx, const double *__restrict__ vy,
    const double *__restrict__ vz, const double *__restrict__ m, double G, double *ekin,
    double *epot) {
    __shared__ double4 src[kRowThreads];
    const uint32_t r = blockIdx.x / kCus, q = blockIdx.x % kCus;
    const uint32_t width = min(kCus, gridDim.x - r * kCus);
    const uint32_t tile = gridDim.x - 1 - (r * kCus + ((r & 1u) ? width - 1u - q : q));
    const uint32_t j = tile * kRowThreads + threadIdx.x;
    const bool valid = j < n;
    const uint32_t jj = valid ? j : 0;
    const double pxj = x[jj], pyj = y[jj], pzj = z[jj], mj = m[jj];
    if (valid) {
        const double v = vx[j] * vx[j] + vy[j] * vy[j] + vz[j] * vz[j];
        ekin[j] = 0.5 * mj * v;
    }
    double ep = 0;
    const bool mj_ok = exponent_within(mj, 150);
    const uint32_t last = min(n, (tile + 1) * kRowThreads);
    for (uint32_t k = 0; k < last; k += kRowThreads) {
        const uint32_t i = k + threadIdx.x;
        bool gm_ok = true;
        if (i < n) {
            const double gm = G * m[i];
            gm_ok = exponent_within(gm, 150);
            src[threadIdx.x] = make_double4(x[i], y[i], z[i], gm);
        }
        const bool tile_ok = __syncthreads_and(gm_ok);
        if (valid && j > k) {
            const uint32_t cnt = min((uint32_t)kRowThreads, j - k);
            uint32_t ii = 0;
            for (; ii + kRowPer <= cnt; ii += kRowPer) {
                double a[kRowPer], v[kRowPer];
                uint32_t worst = 0, low = 0;
#pragma unroll
                for (int u = 0; u < kRowPer; ++u) {
                    const double4 si = src[ii + u];
                    const double r_x = pxj - si.x, r_y = pyj - si.y, r_z = pzj - si.z;
                    a[u] = si.w * mj;
                    v[u] = r_x * r_x + r_y * r_y + r_z * r_z;
                    worst = max(worst, distance_off(v[u]));
                    low = max(low, (uint32_t)__double2loint(v[u]));
                }
                if (tile_ok && mj_ok && worst < kDistanceOff && low < kRootOfOnes) {
#pragma unroll
                    for (int u = 0; u < kRowPer; ++u) a[u] = div_sqrt_core(a[u], v[u]);
                } else {
                    for (int u = 0; u < kRowPer; ++u) a[u] = a[u] / sqrt(v[u]);
                }
#pragma unroll
                for (int u = 0; u < kRowPer; ++u) ep += a[u];
            }
            for (; ii < cnt; ++ii) {
                const double4 si = src[ii];
                const double r_x = pxj - si.x, r_y = pyj - si.y, r_z = pzj - si.z;
                ep += (si.w * mj) / sqrt(r_x * r_x + r_y * r_y + r_z * r_z);
            }
        }
        __syncthreads();
    }
    if (valid) epot[j] = ep;
}

}  // namespace

void launch_energy_terms(uint32_t n, const double *x, const double *y, const double *z,
                         const double *vx, const double *vy, const double *vz, const double *m,
                         double G, double *ekin, double *epot, hipStream_t s) {
    if (n == 0) return;
    if (n >= kRowsFrom) {
        hipLaunchKernelGGL(k_energy_rows, dim3(ceil_div(n, kRowThreads)), dim3(kRowThreads), 0, s,
                           n, x, y, z, vx, vy, vz, m, G, ekin, epot);
        return;
    }
    hipLaunchKernelGGL(k_energy_terms, dim3(ceil_div(n, kTile)), dim3(kThreads), 0, s, n, x, y, z,
                       vx, vy, vz, m, G, ekin, epot);
}

}  // namespace nb
