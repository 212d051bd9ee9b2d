// nbx_direct.hip - all-pairs gravitational accelerations on gfx950.
//
// direct_fp64: bit-identical to the scalar reference kernel
//   (src/c/physics/gravity.c:37-67). Every pair term is formed with the
//   reference's operations in the reference's order (this file is compiled
//   with -ffp-contract=off; nbx_exact.h gives the correctly rounded square
//   root and reciprocal), and each target's three sums are accumulated in
//   ascending j with j == i skipped. Only the term formation is parallel:
//   several waves compute a tile of terms into LDS, one wave adds them in
//   order; with enough targets one lane does both for its own target.
//
// direct_fp32: FP32 pair arithmetic on FP32-rounded positions/masses. Each lane
//   owns one target. In large systems the source index is wave-uniform, so
//   every source is fetched once per wave by scalar loads and broadcast
//   through SGPR operands (no LDS traffic), and a target's sources are split
//   over the 16 waves of its workgroup; small systems spread a wave over 16
//   targets x 4 sources. Partial sums of a few dozen sources are folded into a
//   per-target compensated (Kahan-Babuska) accumulator, and the ranges'
//   accumulators are combined in LDS in range order. G multiplies each
//   target's sum once, in FP64, so a pair costs 12 full-rate VALU instructions
//   and one v_rsq_f32.
#include <mutex>
#include <utility>

#include "nbx_exact.h"
#include "nbx_internal.h"
#include "nbx_learned.h"

namespace nbx {
namespace {

__global__ void clock_kernel(unsigned long long* __restrict__ clock) {
    clock_in(clock);
}

// A launch of its own for the clock, in front of the kernels of large systems:
// with the clock's few instructions inside, direct_fp32_kernel was 1% slower at
// 262,144 targets (in turn with one other build, 1.022 to 1.034 times its speed,
// 1.040 without).
void launch_clock(hipStream_t st, unsigned long long* clock) {
    if (clock != nullptr) {
        clock_kernel<<<1, 1, 0, st>>>(clock);
    }
}

constexpr int kExactTargets = 16;   // targets of a tile kernel's workgroup

// The pair terms of K sources against one target per lane, with the
// reference's operations in its order (gravity.c:46-57).
template <int K>
__device__ inline void exact_terms(const double (&sx)[K], const double (&sy)[K],
                                   const double (&sz)[K], const double (&sm)[K], double xi,
                                   double yi, double zi, double G, double eps2, double (&tx)[K],
                                   double (&ty)[K], double (&tz)[K]) {
    double r2[K], inv[K];
    ExactGuard guard;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        tx[k] = sx[k] - xi;
        ty[k] = sy[k] - yi;
        tz[k] = sz[k] - zi;
        r2[k] = tx[k] * tx[k] + ty[k] * ty[k] + tz[k] * tz[k] + eps2;
        inv[k] = exact_inv_sqrt(r2[k], guard);
    }
    if (__builtin_amdgcn_ballot_w64(guard.odd()) != 0) {
        // (keeps the branch: flattened into selects, every term would pay
        // for both paths)
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("");
#pragma unroll
        for (int k = 0; k < K; ++k) {
            inv[k] = 1.0 / sqrt(r2[k]);
        }
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const double inv3 = inv[k] * inv[k] * inv[k];
        const double s = G * sm[k] * inv3;
        tx[k] = s * tx[k];
        ty[k] = s * ty[k];
        tz[k] = s * tz[k];
    }
}

// Adds COUNT terms, STRIDE doubles apart in LDS, in order; the loads of the
// coming chunk are in flight during the adds of the current one, so the chain
// is the adds alone.
template <int COUNT, int STRIDE>
__device__ inline double add_in_order(double acc, const double* row) {
    constexpr int kChunk = COUNT % 16 == 0 ? 16 : 8;
    static_assert(COUNT % kChunk == 0, "whole chunks");
    double v[kChunk], w[kChunk];
#pragma unroll
    for (int e = 0; e < kChunk; ++e) {
        v[e] = row[e * STRIDE];
    }
#pragma unroll
    for (int c = kChunk; c < COUNT; c += kChunk) {
#pragma unroll
        for (int e = 0; e < kChunk; ++e) {
            w[e] = row[(c + e) * STRIDE];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < kChunk; ++e) {
            acc += v[e];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < kChunk; ++e) {
            v[e] = w[e];
        }
    }
#pragma unroll
    for (int e = 0; e < kChunk; ++e) {
        acc += v[e];
    }
    return acc;
}

// Lane LANE of each row of 16, in all lanes of that row.
template <int LANE>
__device__ inline double row_broadcast(double v) {
    constexpr int kNewBcast = 0x150;   // row_newbcast:LANE
    return __hiloint2double(
        __builtin_amdgcn_update_dpp(0, __double2hiint(v), kNewBcast + LANE, 0xf, 0xf, true),
        __builtin_amdgcn_update_dpp(0, __double2loint(v), kNewBcast + LANE, 0xf, 0xf, true));
}

template <int A, int... E>
__device__ inline void row_fields(double v, double (&x)[A], double (&y)[A], double (&z)[A],
                                  double (&m)[A], std::integer_sequence<int, E...>) {
    ((x[E] = row_broadcast<E>(v), y[E] = row_broadcast<4 + E>(v), z[E] = row_broadcast<8 + E>(v),
      m[E] = row_broadcast<12 + E>(v)), ...);
}

// Tile kernel: 16 targets per workgroup. WAVES waves form the terms of a tile
// of 4 A WAVES sources (a wave's lanes are 16 targets x 4 sources, A
// independent steps in flight), one more wave adds the previous tile's terms
// in source order: lane = component * 16 + target, so one add serves all three
// components. Two term buffers alternate, one barrier per tile. The own term
// and the sources past n are written as +0.0, which leaves a sum bit for bit
// as skipping them would (it starts at +0.0 and +0.0 + -0.0 is +0.0, so it is
// never -0.0).
// SUBSET: the targets are targets[k], k < count, and the accelerations go to
// out[3k .. 3k+2].
template <bool SUBSET, int WAVES, int A>
__global__ __launch_bounds__((WAVES + 1) * 64) void direct_fp64_tile_kernel(
    const double* __restrict__ px, const double* __restrict__ py, const double* __restrict__ pz,
    const double* __restrict__ m, double* __restrict__ ax, double* __restrict__ ay,
    double* __restrict__ az, int n, double G, double eps2, const int64_t* __restrict__ targets,
    int count, double* __restrict__ out, unsigned long long* __restrict__ clock) {
    clock_in(clock);
    constexpr int kTile = 4 * A * WAVES;
    constexpr int kRow = 3 * kExactTargets;
    static_assert(A <= 4, "a row of lanes holds four sources' fields");
    __shared__ double terms[2][kTile][kRow];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
    const int t = lane % kExactTargets;
    const int q = lane / kExactTargets;   // source of a step, or component of the adder
    const int k = blockIdx.x * kExactTargets + t;
    const bool valid = SUBSET ? k < count : k < n;
    const int i = !valid ? -1 : (SUBSET ? static_cast<int>(targets[k]) : k);
    const int tiles = (n + kTile - 1) / kTile;
    if (wave < WAVES) {
        const int ic = valid ? i : n - 1;
        const double xi = px[ic], yi = py[ic], zi = pz[ic];
        const int s0 = wave * 4 * A + q;   // this lane's first source of a tile
        // One load per tile: lane (q, 4 f + a) holds field f of the wave's
        // source 4 a + q; a row broadcast then hands step a's four fields to
        // the row's 16 targets. (With each lane loading its own steps'
        // fields the vector memory path was the bound: N = 4096 64 us.)
        const int field = t / 4;
        const double* base = field == 0 ? px : (field == 1 ? py : (field == 2 ? pz : m));
        const int mine = s0 + 4 * (t % 4);
        auto load = [&](int j0) {
            const int j = j0 + mine;
            return base[j < n ? j : n - 1];
        };
        double next = load(0);
        for (int b = 0; b < tiles; ++b) {
            const int j0 = b * kTile;
            const double cur = next;
            if (b + 1 < tiles) {
                next = load(j0 + kTile);   // in flight while this tile's terms are formed
            }
            double sx[A], sy[A], sz[A], sm[A], tx[A], ty[A], tz[A];
            row_fields(cur, sx, sy, sz, sm, std::make_integer_sequence<int, A>{});
            exact_terms<A>(sx, sy, sz, sm, xi, yi, zi, G, eps2, tx, ty, tz);
            // the own source or the end of the sources within this wave's part
            const int jw = j0 + wave * 4 * A;
            const bool near = static_cast<unsigned>(i - jw) < 4u * A;
            if (jw + 4 * A > n || __builtin_amdgcn_ballot_w64(near) != 0) {
#pragma unroll
                for (int a = 0; a < A; ++a) {
                    const int j = j0 + s0 + 4 * a;
                    const bool none = j >= n || j == i;
                    tx[a] = none ? 0.0 : tx[a];
                    ty[a] = none ? 0.0 : ty[a];
                    tz[a] = none ? 0.0 : tz[a];
                }
            }
            double (*row)[kRow] = terms[b & 1];
#pragma unroll
            for (int a = 0; a < A; ++a) {
                row[s0 + 4 * a][t] = tx[a];
                row[s0 + 4 * a][kExactTargets + t] = ty[a];
                row[s0 + 4 * a][2 * kExactTargets + t] = tz[a];
            }
            __syncthreads();   // tile b written; the adder takes it
        }
    } else {
        __builtin_amdgcn_s_setprio(3);   // the serial chain issues first
        double acc = 0.0;
        const int col = lane < kRow ? lane : kRow - 1;
        for (int b = 0; b < tiles; ++b) {
            __syncthreads();   // tile b written
            acc = add_in_order<kTile, kRow>(acc, &terms[b & 1][0][col]);
        }
        if (valid && lane < kRow) {
            if (SUBSET) {
                out[3 * static_cast<size_t>(k) + q] = acc;
            } else {
                (q == 0 ? ax : (q == 1 ? ay : az))[i] = acc;
            }
        }
    }
}

// One target per lane, sources in order through scalar loads, four sources'
// terms formed side by side and added in order: no LDS, no barrier.
template <bool SUBSET>
__global__ __launch_bounds__(256) void direct_fp64_lane_kernel(
    const double* __restrict__ px, const double* __restrict__ py, const double* __restrict__ pz,
    const double* __restrict__ m, double* __restrict__ ax, double* __restrict__ ay,
    double* __restrict__ az, int n, double G, double eps2, const int64_t* __restrict__ targets,
    int count, double* __restrict__ out) {
    constexpr int K = 4;
    const int k = blockIdx.x * 256 + threadIdx.x;
    const bool valid = SUBSET ? k < count : k < n;
    const int i = !valid ? -1 : (SUBSET ? static_cast<int>(targets[k]) : k);
    const int ic = valid ? i : n - 1;
    const double xi = px[ic], yi = py[ic], zi = pz[ic];
    double acx = 0.0, acy = 0.0, acz = 0.0;
    // sources of the coming group; its scalar loads are in flight while the
    // current group's terms are formed
    double nx[K], ny[K], nz[K], nm[K];
    auto load = [&](int j0) {
#pragma unroll
        for (int e = 0; e < K; ++e) {
            nx[e] = px[j0 + e];
            ny[e] = py[j0 + e];
            nz[e] = pz[j0 + e];
            nm[e] = m[j0 + e];
        }
    };
    const int whole = n / K * K;
    if (whole > 0) {
        load(0);
    }
    for (int j0 = 0; j0 < whole; j0 += K) {
        double sx[K], sy[K], sz[K], sm[K], tx[K], ty[K], tz[K];
#pragma unroll
        for (int e = 0; e < K; ++e) {
            sx[e] = nx[e];
            sy[e] = ny[e];
            sz[e] = nz[e];
            sm[e] = nm[e];
        }
        load(j0 + K < whole ? j0 + K : 0);
        exact_terms<K>(sx, sy, sz, sm, xi, yi, zi, G, eps2, tx, ty, tz);
        // the own term adds +0.0
        const bool near = static_cast<unsigned>(i - j0) < static_cast<unsigned>(K);
        if (__builtin_amdgcn_ballot_w64(near) != 0) {
#pragma unroll
            for (int e = 0; e < K; ++e) {
                const bool own = j0 + e == i;
                tx[e] = own ? 0.0 : tx[e];
                ty[e] = own ? 0.0 : ty[e];
                tz[e] = own ? 0.0 : tz[e];
            }
        }
#pragma unroll
        for (int e = 0; e < K; ++e) {
            acx += tx[e];
            acy += ty[e];
            acz += tz[e];
        }
    }
    for (int j = whole; j < n; ++j) {
        const double sx[1] = {px[j]}, sy[1] = {py[j]}, sz[1] = {pz[j]}, sm[1] = {m[j]};
        double tx[1], ty[1], tz[1];
        exact_terms<1>(sx, sy, sz, sm, xi, yi, zi, G, eps2, tx, ty, tz);
        acx += j == i ? 0.0 : tx[0];
        acy += j == i ? 0.0 : ty[0];
        acz += j == i ? 0.0 : tz[0];
    }
    if (valid) {
        if (SUBSET) {
            double* o = out + 3 * static_cast<size_t>(k);
            o[0] = acx;
            o[1] = acy;
            o[2] = acz;
        } else {
            ax[i] = acx;
            ay[i] = acy;
            az[i] = acz;
        }
    }
}

// Launches the FP64 all-pairs kernel over `count` targets (all n particles,
// or the SUBSET `targets`) that suits the grid. A workgroup of the tile kernel
// takes 16 targets. Up to one per CU, eight waves form terms; up to three per
// CU, six; beyond, three, of which four workgroups fit a CU. From 1.6 waves of
// targets per SIMD on the lane kernel, which has no LDS traffic, fills the chip
// by itself: its time is that of the SIMDs with two waves. Measured on MI355X, ms per evaluation with 8 / 6 / 3 waves
// and the lane kernel (every result bit for bit the same):
//   N = 1000   0.0137 / 0.0147 / 0.0178 / 0.096    N = 4096  0.0445 / 0.0476 / 0.0623 / 0.375
//   N = 8192   0.163  / 0.147  / 0.164  / 0.75     N = 12288 0.353  / 0.314  / 0.320  / -
//   N = 16384  0.604  / 0.522  / 0.492  / 1.54     N = 40000 3.44   / -      / 2.56   / 4.0
//   3 waves / lane: N = 98304 14.9 / 15.7, 104448 17.0 / 17.1, 106496 17.4 / 17.4,
//   108544 18.5 / 17.8, 110592 18.8 / 17.9, 131072 25.4 / 22.9
// The kernel this replaced (64 targets per workgroup, IEEE sqrt and divide):
// 0.049 ms at 1000, 0.186 at 4096, 0.79 at 16384, 4.28 at 40000, 9.05 at 65536
// (now 6.9). The bound is FP64 issue: about 36 instructions and a v_rsq_f64 a
// pair, 84 ns per 64 pairs and SIMD, against 72 instructions and two
// transcendentals before; a tile kernel's adder and row broadcasts add 12.
template <bool SUBSET>
void launch_direct_fp64(hipStream_t st, int cu_count, const double* px, const double* py,
                        const double* pz, const double* m, double* ax, double* ay, double* az,
                        int n, double G, double eps2, const int64_t* targets, int count,
                        double* out, unsigned long long* clock = nullptr) {
    auto go = [&](auto kernel, unsigned grid, unsigned threads) {
        kernel<<<grid, threads, 0, st>>>(px, py, pz, m, ax, ay, az, n, G, eps2, targets, count,
                                         out, clock);
    };
    const unsigned blocks = grid_for(static_cast<size_t>(count), kExactTargets);
    const unsigned cus = static_cast<unsigned>(cu_count);
    if (blocks <= cus) {
        go(direct_fp64_tile_kernel<SUBSET, 8, 4>, blocks, 9 * kWave);
    } else if (blocks <= 3 * cus) {
        go(direct_fp64_tile_kernel<SUBSET, 6, 4>, blocks, 7 * kWave);
    } else if (blocks < 26 * cus) {
        go(direct_fp64_tile_kernel<SUBSET, 3, 4>, blocks, 4 * kWave);
    } else {
        launch_clock(st, clock);
        direct_fp64_lane_kernel<SUBSET>
            <<<grid_for(static_cast<size_t>(count), 256), 256, 0, st>>>(
                px, py, pz, m, ax, ay, az, n, G, eps2, targets, count, out);
    }
}

__device__ inline void two_sum_add(float& s, float& c, float v) {
    // Kahan-Babuska (Neumaier) step: exact error term of s + v goes to c.
    const float t = s + v;
    const float e = (fabsf(s) >= fabsf(v)) ? ((s - t) + v) : ((v - t) + s);
    s = t;
    c += e;
}

// One pair term m / r^3 d added to (ax, ay, az): 12 full-rate VALU instructions
// and one v_rsq_f32.
template <bool ZERO_EPS>
__device__ inline void fp32_pair(const float4& q, float xi, float yi, float zi, float eps2,
                                 float& ax, float& ay, float& az) {
    const float dx = q.x - xi;
    const float dy = q.y - yi;
    const float dz = q.z - zi;
    const float r2 = fmaf(dx, dx, fmaf(dy, dy, fmaf(dz, dz, eps2)));
    float inv = __builtin_amdgcn_rsqf(r2);
    if (ZERO_EPS) {
        inv = r2 > 0.f ? inv : 0.f;
    }
    const float inv2 = inv * inv;
    const float s = (q.w * inv) * inv2;
    ax = fmaf(s, dx, ax);
    ay = fmaf(s, dy, ay);
    az = fmaf(s, dz, az);
}

// One target per lane, 64 per workgroup. The targets' sources are split into S
// ranges of whole tiles, one per wave, and the partial sums meet in LDS in
// range order (deterministic).
template <int S, bool ZERO_EPS>
__global__ __launch_bounds__(S * kWave) void direct_fp32_kernel(const float4* __restrict__ pos,
                                                                double* __restrict__ ax,
                                                                double* __restrict__ ay,
                                                                double* __restrict__ az, int n,
                                                                double G, float eps2, int tile) {
    const int part = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
    const int lane = static_cast<int>(threadIdx.x) & (kWave - 1);
    const int i = blockIdx.x * kWave + lane;
    const float4 p = pos[i < n ? i : n - 1];
    const float xi = p.x, yi = p.y, zi = p.z;
    const int tiles = (n + tile - 1) / tile;
    const int per = (tiles + S - 1) / S;
    const int jb = min(n, part * per * tile);
    const int je = min(n, (part + 1) * per * tile);
    float sx = 0.f, sy = 0.f, sz = 0.f, cx = 0.f, cy = 0.f, cz = 0.f;
    for (int j0 = jb; j0 < je; j0 += tile) {
        const int j1 = (j0 + tile) < je ? (j0 + tile) : je;
        float px = 0.f, py = 0.f, pz = 0.f;
#pragma unroll 4
        for (int j = j0; j < j1; ++j) {
            fp32_pair<ZERO_EPS>(pos[j], xi, yi, zi, eps2, px, py, pz);
        }
        two_sum_add(sx, cx, px);
        two_sum_add(sy, cy, py);
        two_sum_add(sz, cz, pz);
    }
    __shared__ float part_sums[S - 1][6][kWave];
    if (part > 0) {
        float* r = &part_sums[part - 1][0][lane];
        r[0 * kWave] = sx;
        r[1 * kWave] = sy;
        r[2 * kWave] = sz;
        r[3 * kWave] = cx;
        r[4 * kWave] = cy;
        r[5 * kWave] = cz;
    }
    __syncthreads();
    if (part == 0) {
        for (int k = 0; k < S - 1; ++k) {
            two_sum_add(sx, cx, part_sums[k][0][lane]);
            two_sum_add(sy, cy, part_sums[k][1][lane]);
            two_sum_add(sz, cz, part_sums[k][2][lane]);
            cx += part_sums[k][3][lane];
            cy += part_sums[k][4][lane];
            cz += part_sums[k][5][lane];
        }
        if (i < n) {
            // G applied once per target, in FP64 (exact for G = 1)
            ax[i] = G * (static_cast<double>(sx) + static_cast<double>(cx));
            ay[i] = G * (static_cast<double>(sy) + static_cast<double>(cy));
            az[i] = G * (static_cast<double>(sz) + static_cast<double>(cz));
        }
    }
}

// Small systems: 16 targets per workgroup; a wave's lanes are 16 targets x 4
// sources, the 16 waves take every 16th group of four, and the 64 partial sums
// of a target (at most 192 plain terms each) meet by compensated adds, over the
// lanes and then over the waves in order. STAGE: one launch, every workgroup
// rounds all the sources to FP32 into LDS itself; otherwise they come from the
// staged positions `pos`.
constexpr int kStageN = 4096;
constexpr int kSmallN = 12288;
constexpr int kSmallTargets = 16;
constexpr int kSmallWaves = 16;
template <bool ZERO_EPS, bool STAGE>
__global__ __launch_bounds__(kSmallWaves * kWave) void direct_fp32_small_kernel(
    const double* __restrict__ px, const double* __restrict__ py, const double* __restrict__ pz,
    const double* __restrict__ m, const float4* __restrict__ pos, double* __restrict__ ax, double* __restrict__ ay,
    double* __restrict__ az, int n, double G, float eps2,
    unsigned long long* __restrict__ clock) {
    clock_in(clock);
    __shared__ float4 stage[STAGE ? kStageN : 1];
    __shared__ float part_sums[kSmallWaves][6][kSmallTargets];
    if (STAGE) {
        for (int j = threadIdx.x; j < n; j += kSmallWaves * kWave) {
            stage[j] = make_float4(static_cast<float>(px[j]), static_cast<float>(py[j]),
                                   static_cast<float>(pz[j]), static_cast<float>(m[j]));
        }
        __syncthreads();
    }
    const float4* src = STAGE ? stage : pos;
    const int wave = static_cast<int>(threadIdx.x) / kWave;
    const int lane = static_cast<int>(threadIdx.x) & (kWave - 1);
    const int t = lane % kSmallTargets;
    const int i = blockIdx.x * kSmallTargets + t;
    const float4 p = src[i < n ? i : n - 1];
    float s[3] = {0.f, 0.f, 0.f}, c[3] = {0.f, 0.f, 0.f};
#pragma unroll 4
    for (int j = wave * (kWave / kSmallTargets) + lane / kSmallTargets; j < n;
         j += kSmallWaves * (kWave / kSmallTargets)) {
        fp32_pair<ZERO_EPS>(src[j], p.x, p.y, p.z, eps2, s[0], s[1], s[2]);
    }
#pragma unroll
    for (int off = kSmallTargets; off < kWave; off <<= 1) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const float so = __shfl_xor(s[k], off), co = __shfl_xor(c[k], off);
            two_sum_add(s[k], c[k], so);
            c[k] += co;
        }
    }
    if (lane < kSmallTargets) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            part_sums[wave][k][t] = s[k];
            part_sums[wave][3 + k][t] = c[k];
        }
    }
    __syncthreads();
    // thread = component * 16 + target
    if (threadIdx.x < 3 * kSmallTargets) {
        const int k = threadIdx.x / kSmallTargets;
        float sum = 0.f, comp = 0.f;
#pragma unroll
        for (int w = 0; w < kSmallWaves; ++w) {
            two_sum_add(sum, comp, part_sums[w][k][t]);
            comp += part_sums[w][3 + k][t];
        }
        if (i < n) {
            // G applied once per target, in FP64 (exact for G = 1)
            (k == 0 ? ax : (k == 1 ? ay : az))[i] =
                G * (static_cast<double>(sum) + static_cast<double>(comp));
        }
    }
}

__global__ void refresh_pos4_kernel(const double* __restrict__ px, const double* __restrict__ py,
                                    const double* __restrict__ pz, const double* __restrict__ m,
                                    float4* __restrict__ out, int n,
                                    unsigned long long* __restrict__ clock) {
    clock_in(clock);
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        out[i] = make_float4(static_cast<float>(px[i]), static_cast<float>(py[i]),
                             static_cast<float>(pz[i]), static_cast<float>(m[i]));
    }
}

// Up to kStageN sources a workgroup stages all of them itself; up to kSmallN 16
// targets per workgroup give the chip more of them to run; beyond, 64 targets
// and 16 source ranges. Measured on MI355X, us per evaluation, against four
// ranges of 256-source tiles for all sizes (the kernel alone; in front of it a
// staging launch, which the first line no longer needs):
//   N = 1000 17.8 -> 6.8, 4096 58.8 -> 13.2  (all staged, 16 targets)
//   N = 5000 71.8 -> 23.7, 8192 113 -> 37.7, 12000 161 -> 75  (16 targets;
//     with 64 targets 36.7, 56.1, 83; at 16384 135 against 113)
//   N = 16384 221 -> 113, 32768 396 -> 363, 65536 1533 -> 1305,
//     131072 5668 -> 5064, 262144 20800 -> 19800  (8 ranges: 111, 387, 1363,
//     5151, 19965; 256-source tiles instead of 64: 262144 20046)
// At 262144 that is 3,470 G pairs/s, 44.7 cycles per wave of 64 pairs and SIMD at
// the 2.38 GHz that the chip ran at. The bound is issue: 12 instructions of 2
// cycles and a v_rsq_f32 of 8 are 32, and a loop of 12 v_fma_f32 and one v_rsq_f32
// alone measured 38.7.
template <bool ZERO_EPS>
void launch_direct_fp32(hipStream_t st, const double* px, const double* py, const double* pz,
                        const double* m, const float4* pos, double* ax, double* ay, double* az,
                        int n, double G, float eps2, bool staged, unsigned long long* clock) {
    if (n <= kSmallN) {
        const unsigned grid = grid_for(static_cast<size_t>(n), kSmallTargets);
        if (!staged) {
            direct_fp32_small_kernel<ZERO_EPS, true><<<grid, kSmallWaves * kWave, 0, st>>>(
                px, py, pz, m, pos, ax, ay, az, n, G, eps2, clock);
        } else {
            direct_fp32_small_kernel<ZERO_EPS, false><<<grid, kSmallWaves * kWave, 0, st>>>(
                px, py, pz, m, pos, ax, ay, az, n, G, eps2, clock);
        }
        return;
    }
    constexpr int kRanges = 16, kSourceTile = 64;
    launch_clock(st, clock);
    direct_fp32_kernel<kRanges, ZERO_EPS>
        <<<grid_for(static_cast<size_t>(n), kWave), kRanges * kWave, 0, st>>>(
            pos, ax, ay, az, n, G, eps2, kSourceTile);
}

// The FP32 all-pairs evaluation; staged: `pos` holds the positions (always
// beyond kStageN, where one workgroup's LDS does not).
void launch_direct_fp32(hipStream_t st, const double* px, const double* py, const double* pz,
                        const double* m, const float4* pos, double* ax, double* ay, double* az,
                        int n, const NBodySimProGravity* g, bool staged,
                        unsigned long long* clock = nullptr) {
    const double G = g->gravitational_constant;
    const float eps2 = static_cast<float>(g->softening_squared);
    if (eps2 > 0.f) {
        launch_direct_fp32<false>(st, px, py, pz, m, pos, ax, ay, az, n, G, eps2, staged, clock);
    } else {
        launch_direct_fp32<true>(st, px, py, pz, m, pos, ax, ay, az, n, G, eps2, staged, clock);
    }
}

}  // namespace

NBodySimProStatus refresh_pos4(Engine* e, NBodySimProError* error, unsigned long long* clock) {
    if (e->pos4_valid || e->n == 0) {
        return N_BODY_SIM_PRO_STATUS_OK;
    }
    const int n = static_cast<int>(e->n);
    refresh_pos4_kernel<<<grid_for(e->n, 256), 256, 0, e->stream>>>(e->px, e->py, e->pz, e->m,
                                                                     e->pos4, n, clock);
    NBX_HIP(error, hipGetLastError());
    e->pos4_valid = true;
    return N_BODY_SIM_PRO_STATUS_OK;
}

namespace {

// The clocks of an all-pairs evaluation in the engine's pinned memory: start
// of its first kernel, of the pair kernel, and of what follows it.
unsigned long long* clocks_of(Engine* e) {
    return reinterpret_cast<unsigned long long*>(static_cast<char*>(e->bh.report) + kClocksAt);
}

}  // namespace

NBodySimProStatus direct_fp64(Engine* e, const NBodySimProGravity* g, NBodySimProError* error) {
    const size_t n = e->n;
    e->pending = 0;
    if (n == 0) {
        return N_BODY_SIM_PRO_STATUS_OK;
    }
    launch_direct_fp64<false>(e->stream, e->cu_count, e->px, e->py, e->pz, e->m, e->ax, e->ay,
                              e->az, static_cast<int>(n), g->gravitational_constant,
                              g->softening_squared, nullptr, static_cast<int>(n), nullptr,
                              e->timed ? clocks_of(e) + 1 : nullptr);
    NBX_HIP(error, hipGetLastError());
    e->pending = e->timed ? 2 : 0;
    return N_BODY_SIM_PRO_STATUS_OK;
}

NBodySimProStatus direct_fp32(Engine* e, const NBodySimProGravity* g, NBodySimProError* error) {
    const size_t n = e->n;
    e->pending = 0;
    if (n == 0) {
        return N_BODY_SIM_PRO_STATUS_OK;
    }
    const bool stages = n > static_cast<size_t>(kStageN) && !e->pos4_valid;
    if (stages) {
        NBX_TRY(refresh_pos4(e, error, e->timed ? clocks_of(e) : nullptr));
    }
    launch_direct_fp32(e->stream, e->px, e->py, e->pz, e->m, e->pos4, e->ax, e->ay, e->az,
                       static_cast<int>(n), g, n > static_cast<size_t>(kStageN),
                       e->timed ? clocks_of(e) + 1 : nullptr);
    NBX_HIP(error, hipGetLastError());
    e->pending = e->timed ? (stages ? 4 : 3) : 0;
    return N_BODY_SIM_PRO_STATUS_OK;
}

unsigned long long* direct_end(Engine* e) {
    if (e->pending == 0) {
        return nullptr;
    }
    e->ended = true;
    return clocks_of(e) + 2;
}

// (Events around the kernel instead left the stream idle for 5.8 us each:
// FP64 drop-in call at 1,000 particles 37.4 us, 29.7 with the clocks. Events that
// the dispatch itself carries: 51.9.)
NBodySimProStatus direct_timings(Engine* e, NBodySimProError* error) {
    const int pending = e->pending;
    if (pending == 0) {
        return N_BODY_SIM_PRO_STATUS_OK;
    }
    if (!e->ended) {
        launch_clock(e->stream, direct_end(e));
        NBX_HIP(error, hipGetLastError());
        NBX_HIP(error, hipStreamSynchronize(e->stream));
    }
    e->pending = 0;
    e->ended = false;
    const unsigned long long* at = clocks_of(e);
    auto ms = [&](int from) {
        return at[2] > at[from] ? static_cast<double>(at[2] - at[from]) / e->clock_khz : 0.0;
    };
    const bool fp64 = pending == 2;
    const double kernel = ms(1), total = pending == 4 ? ms(0) : kernel;
    const double n = static_cast<double>(e->n);
    e->timings = NBXTimings{};
    e->timings.force_ms = total;
    e->timings.kernel_ms = kernel;
    e->timings.kernel_flops = 20.0 * n * (n - 1.0);
    // FP64: x, y, z, m of each; FP32: one float4; three doubles out
    e->timings.kernel_bytes = ((fp64 ? 4.0 * 8.0 : 16.0) + 3.0 * 8.0) * n;
    return N_BODY_SIM_PRO_STATUS_OK;
}

}  // namespace nbx

extern "C" NBodySimProStatus nbx_engine_direct_fp64_targets(NBXEngine* engine,
                                                            const NBodySimProGravity* gravity,
                                                            const int64_t* targets, size_t count,
                                                            double* out, NBodySimProError* error) {
    if (engine == nullptr || gravity == nullptr || (count > 0 && (targets == nullptr || out == nullptr))) {
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_ARGUMENT,
                 "engine, gravity, targets and out are required");
    }
    nbx::Engine* e = &engine->e;
    if (count == 0) {
        return N_BODY_SIM_PRO_STATUS_OK;
    }
    if (count > 0x7FFFFFFFull) {
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_ARGUMENT, "too many targets");
    }
    for (size_t k = 0; k < count; ++k) {
        if (targets[k] < 0 || static_cast<size_t>(targets[k]) >= e->n) {
            NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_ARGUMENT, "target index out of range");
        }
    }
    NBX_HIP(error, hipSetDevice(e->device));
    const size_t tbytes = (count * sizeof(int64_t) + 255) / 256 * 256;
    NBX_TRY(e->scratch.need<unsigned char>(tbytes + 3 * count * sizeof(double), error));
    int64_t* dt = e->scratch.as<int64_t>();
    double* dout = reinterpret_cast<double*>(e->scratch.as<unsigned char>() + tbytes);
    NBX_HIP(error, hipMemcpyAsync(dt, targets, count * sizeof(int64_t), hipMemcpyHostToDevice,
                                  e->stream));
    nbx::launch_direct_fp64<true>(e->stream, e->cu_count, e->px, e->py, e->pz, e->m, nullptr,
                                  nullptr, nullptr, static_cast<int>(e->n),
                                  gravity->gravitational_constant, gravity->softening_squared, dt,
                                  static_cast<int>(count), dout);
    NBX_HIP(error, hipGetLastError());
    NBX_HIP(error, hipMemcpyAsync(out, dout, 3 * count * sizeof(double), hipMemcpyDeviceToHost,
                                  e->stream));
    NBX_HIP(error, hipStreamSynchronize(e->stream));
    return N_BODY_SIM_PRO_STATUS_OK;
}

// ---- FP32 all-pairs without allocation (nbx_direct_fp32_noalloc) ----
//
// The FP32 (x, y, z, m) staging that nbx_hip_direct_fp32 keeps in its engine
// lives here in a fixed device array instead: each GPU the library runs on
// holds its own copy (16 MiB) until the process ends. Every call on a GPU
// shares that GPU's copy, so calls that overlap on one GPU (on different
// streams, or from different host threads) race. The staging is fully
// rewritten for [0, n) by each call, so nothing needs clearing.
namespace nbx {
namespace {
constexpr size_t kNoAllocMaxParticles = size_t(1) << 20;
constexpr int kNoAllocMaxDevices = 64;
std::mutex g_noalloc_mutex;
void* g_noalloc_staging[kNoAllocMaxDevices] = {};

// Whether any of the outputs (n doubles each) covers part of an input.
bool outputs_over_inputs(const double* const (&in)[4], double* const (&out)[3], size_t n) {
    const uintptr_t bytes = n * sizeof(double);
    for (const double* i : in) {
        for (const double* o : out) {
            const uintptr_t a = reinterpret_cast<uintptr_t>(i), b = reinterpret_cast<uintptr_t>(o);
            if (a < b + bytes && b < a + bytes) {
                return true;
            }
        }
    }
    return false;
}
}  // namespace
}  // namespace nbx

static __device__ __align__(256) float4 scratch[nbx::kNoAllocMaxParticles];

extern "C" NBodySimProStatus nbx_direct_fp32_noalloc(
    const double* positions_x, const double* positions_y, const double* positions_z,
    const double* masses, double* accelerations_x, double* accelerations_y,
    double* accelerations_z, size_t count, const NBodySimProGravity* gravity, void* stream,
    NBodySimProError* error) {
    if (gravity == nullptr) {
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_ARGUMENT, "gravity is required");
    }
    if (count == 0) {
        return N_BODY_SIM_PRO_STATUS_OK;
    }
    if (positions_x == nullptr || positions_y == nullptr || positions_z == nullptr ||
        masses == nullptr || accelerations_x == nullptr || accelerations_y == nullptr ||
        accelerations_z == nullptr) {
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_ARGUMENT,
                 "positions, masses and accelerations must be device pointers, not null");
    }
    if (count > nbx::kNoAllocMaxParticles) {
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_ARGUMENT,
                 "nbx_direct_fp32_noalloc takes at most 1048576 particles");
    }
    int device = -1;
    NBX_HIP(error, hipGetDevice(&device));
    if (device < 0 || device >= nbx::kNoAllocMaxDevices) {
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_UNSUPPORTED_PLATFORM, "device ordinal above 63");
    }
    float4* staging = nullptr;
    {
        // first call on this device (current): the device address of its copy
        std::lock_guard<std::mutex> lock(nbx::g_noalloc_mutex);
        if (nbx::g_noalloc_staging[device] == nullptr) {
            void* p = nullptr;
            NBX_HIP(error, hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
            nbx::g_noalloc_staging[device] = p;
        }
        staging = static_cast<float4*>(nbx::g_noalloc_staging[device]);
    }
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int n = static_cast<int>(count);
    // Accelerations may take the place of the inputs: then every input is read
    // by a launch of its own, also where each workgroup would read them all
    // itself while others store.
    const bool staged =
        count > static_cast<size_t>(nbx::kStageN) ||
        nbx::outputs_over_inputs({positions_x, positions_y, positions_z, masses},
                                 {accelerations_x, accelerations_y, accelerations_z}, count);
    if (staged) {
        nbx::refresh_pos4_kernel<<<nbx::grid_for(count, 256), 256, 0, st>>>(
            positions_x, positions_y, positions_z, masses, staging, n, nullptr);
    }
    // the same kernels as nbx_hip_direct_fp32 (identical results)
    nbx::launch_direct_fp32(st, positions_x, positions_y, positions_z, masses, staging,
                            accelerations_x, accelerations_y, accelerations_z, n, gravity, staged);
    NBX_HIP(error, hipGetLastError());
    return N_BODY_SIM_PRO_STATUS_OK;
}
