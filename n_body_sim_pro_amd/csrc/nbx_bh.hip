// nbx_bh.hip - Barnes-Hut on gfx950: bounding cube, keys, sorts, octree,
// centre-of-mass pass and walk, reproducing src/c/barnes_hut/barnes_hut.c.
//
// Topology. The reference builds a point-region octree by inserting particles
// one at a time in Morton order (barnes_hut.c:503-520); the octant of a
// particle in a cell is decided by strict '>' tests against the FP64 cell
// centre, and child centres come from repeated c +/- h*0.5 (:129-142,
// :202-211). The resulting tree does not depend on insertion order: two
// particles share the depth-d cell iff their first d octant digits agree.
// Here every particle's first 21 octant digits are computed with exactly those
// FP64 operations ("true-path key", 63 bits, the Morton key's layout) and the
// particles are ordered by them; particles that share all 21 digits by up to
// six more 21-digit words (depth <= 147 >= the reference's 128-level limit).
// The Morton keys and order themselves, which can differ where a coordinate
// lies within rounding of a cell face, do not enter the tree: the probes that
// report them compute them on demand.
//
// Nodes are laid out in depth-first pre-order with children in DESCENDING
// octant order, built from the sorted keys with no per-level launches:
// delta[t] = common levels of neighbours t, t+1 (in descending key order);
// position t starts the cells of depths (delta[t-1], delta[t]] and ends those
// of depths (delta[t], delta[t-1]]. A scan of the start counts gives every
// node's pre-order index; cells are also numbered depth-major ("level
// index"), and the k-th start and k-th end of one depth belong to the same
// cell, which gives each cell's last position (its skip pointer) and parent
// without searching. That pre-order with children 7..0 is exactly the order in
// which the reference's LIFO walk pops nodes (children pushed 0..7,
// barnes_hut.c:617-634), so a walk that follows skip pointers visits, for
// every query, the same nodes in the same order.
//
// The whole evaluation is enqueued without a host read in between: buffers are
// sized for the usual number of cells, and what the host would have to decide
// (a key order the fast sort cannot finish, more cells than fit, a tree too
// deep) raises a flag that makes the later kernels do nothing. The host reads
// flags, counts and the walk's counters once, at the end.
//
// Centre of mass. Computed in FP64 from the children in octant order 0..7
// (barnes_hut.c:230-244), one thread per cell, deepest level first. A
// workgroup builds the cells that lie within its tile of 256 to 1,024 tree
// positions in LDS, child tables and centres of mass together (build_kernel); one
// or two more launches do those that span tiles (span_com_kernel). A cell reads its
// children through an 8-slot child table, so results are deterministic and
// bit-identical to the reference.
//
// Walks. The FP64 walk (and the FP32 walk with reference lists): one wave = 8 to
// 64 (128) consecutive queries in tree order; the node index is wave-uniform
// (node records come in through scalar loads). Each lane keeps "skip_until": it is
// active at node i iff i >= skip_until. Active lanes apply the reference's
// own test (d^2 > 0 and 4h^2 < theta^2 d^2, unsoftened) and either take the
// monopole/leaf term (then skip the subtree) or descend. The wave moves to i+1
// if any active lane descends, else to skip[i]. Every lane thus sees exactly
// its reference interaction set, in reference order, with no stack. The FP64
// variant uses the reference arithmetic and is bit-identical. The default FP32
// walk is a group walk over the level-indexed cells (group_walk_kernel).
#include "nbx_exact.h"
#include "nbx_internal.h"

#include <cstring>
#include <type_traits>
#include <vector>

namespace nbx {
namespace {

constexpr int kThreads = 256;
constexpr int kExtWords = 6;
constexpr int kMaxLevels = 129;  // a shared depth-129 cell means depth > 128 (barnes_hut.c:149-153)
// What the host has to handle before the tree is valid: particles that share a
// whole key (small systems), a tree deeper than the reference's limit, an order
// that order_kernel could not finish, more cells than there is room for.
enum { FLAG_TIE = 0, FLAG_OVERFLOW = 1, FLAG_LONG_RUN = 2, FLAG_CELLS = 3 };
// FLAG_LONG_RUN: a run too long; tied positions that found no slot for their
// extension words.
enum { ORDER_RUN = 1u, ORDER_SLOTS = 2u };
// Flag words, the number of tied positions, the per-depth cell counts and their
// total.
constexpr int kTiedCount = 4;
constexpr int kDCount = 8;
constexpr int kFlagWords = 160;
static_assert(kDCount + kMaxLevels + 1 <= kFlagWords, "depth counts and total");

__device__ inline uint64_t spread3(uint64_t a) {
    uint64_t x = a & 0x1FFFFFull;
    x = (x | (x << 32)) & 0x1F00000000FFFFull;
    x = (x | (x << 16)) & 0x1F0000FF0000FFull;
    x = (x | (x << 8)) & 0x100F00F00F00F00Full;
    x = (x | (x << 4)) & 0x10C30C30C30C30C3ull;
    x = (x | (x << 2)) & 0x1249249249249249ull;
    return x;
}

// barnes_hut.c:286-294
__device__ inline uint64_t axis_code(double v, double c, double h) {
    double u = (v - c) / (2.0 * h) + 0.5;
    if (u < 0.0) {
        u = 0.0;
    } else if (u >= 1.0) {
        u = 1.0 - 1.0e-15;
    }
    return static_cast<uint64_t>(u * 2097152.0);
}

// One 21-level word of octant digits starting at the given cell (advances it).
__device__ inline uint64_t path_word(double x, double y, double z, double& cx, double& cy,
                                     double& cz, double& h) {
    uint64_t key = 0;
    for (int d = 0; d < 21; ++d) {
        const int o = (x > cx ? 1 : 0) | (y > cy ? 2 : 0) | (z > cz ? 4 : 0);
        key |= static_cast<uint64_t>(o) << (60 - 3 * d);
        const double off = h * 0.5;
        cx = cx + ((o & 1) ? off : -off);
        cy = cy + ((o & 2) ? off : -off);
        cz = cz + ((o & 4) ? off : -off);
        h = 0.5 * h;
    }
    return key;
}

__device__ inline int word_levels(uint64_t x) {
    // x != 0, key bits 0..62: first differing bit 62-k lies in level k/3.
    return (__clzll(static_cast<long long>(x)) - 1) / 3;
}

// The extension words of tree positions, six each (words null: none are made).
// With `slot`, position t's are those of slot[t], which only positions that
// share their key with a neighbour have.
struct ExtTable {
    const uint64_t* words;
    const uint32_t* slot;
    __device__ const uint64_t* of(int t) const {
        return words + static_cast<size_t>(slot != nullptr ? slot[t] : t) * kExtWords;
    }
};

__device__ inline int common_levels(const uint64_t* __restrict__ w, const ExtTable& ext, int a,
                                    int b) {
    const uint64_t x = w[a] ^ w[b];
    if (x != 0) {
        return word_levels(x);
    }
    if (ext.words == nullptr) {
        return 21;
    }
    const uint64_t* ea = ext.of(a);
    const uint64_t* eb = ext.of(b);
    for (int k = 0; k < kExtWords; ++k) {
        const uint64_t y = ea[k] ^ eb[k];
        if (y != 0) {
            const int l = 21 * (k + 1) + word_levels(y);
            return l < kMaxLevels ? l : kMaxLevels;
        }
    }
    return kMaxLevels;
}

// Octant digit of tree position t at level `level` (the octant of its depth
// level+1 cell inside its depth `level` cell, which holds a neighbour too).
__device__ inline int digit_at(const uint64_t* __restrict__ w, const ExtTable& ext, int t,
                               int level) {
    const uint64_t word = level < 21 ? w[t] : ext.of(t)[level / 21 - 1];
    return static_cast<int>((word >> (60 - 3 * (level % 21))) & 7u);
}

// ---------------------------------------------------------------- inputs and bounding cube
// Build inputs as one (x, y, z, m) record per particle (type In): the
// FP32-rounded values as float4 (hip_barnes_hut; every FP64 operation of the
// build sees them widened back, exactly) or the FP64 values as double4 (the
// FP64 walk). Half the bytes for the FP32 build in every pass that moves them.
__device__ inline double4 widen(const double4& v) {
    return v;
}

__device__ inline double4 widen(const float4& v) {
    return make_double4(static_cast<double>(v.x), static_cast<double>(v.y),
                        static_cast<double>(v.z), static_cast<double>(v.w));
}

template <typename In>
__device__ inline In build_input(const double* __restrict__ px, const double* __restrict__ py,
                                 const double* __restrict__ pz, const double* __restrict__ m,
                                 int i) {
    if constexpr (std::is_same_v<In, float4>) {
        return make_float4(static_cast<float>(px[i]), static_cast<float>(py[i]),
                           static_cast<float>(pz[i]), static_cast<float>(m[i]));
    } else {
        return make_double4(px[i], py[i], pz[i], m[i]);
    }
}

// barnes_hut.c:453-483. min/max are exact, so the reduction order is free.
// The same grid-stride pass writes the build inputs.
constexpr int kBBoxBlocks = 512;

// The workgroup's bounds from every thread's, into s[0..2][0] and s[3..5][0].
template <int T>
__device__ inline void block_bounds(const double (&lo)[3], const double (&hi)[3],
                                    double (*s)[T]) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        s[a][threadIdx.x] = lo[a];
        s[3 + a][threadIdx.x] = hi[a];
    }
    __syncthreads();
    for (int off = T / 2; off > 0; off >>= 1) {
        if (threadIdx.x < static_cast<unsigned>(off)) {
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const double l = s[a][threadIdx.x + off];
                const double h = s[3 + a][threadIdx.x + off];
                if (l < s[a][threadIdx.x]) s[a][threadIdx.x] = l;
                if (h > s[3 + a][threadIdx.x]) s[3 + a][threadIdx.x] = h;
            }
        }
        __syncthreads();
    }
}

// The walk's counters: cell terms, leaf terms, deferred queries. Behind them the
// device clock at the start of each phase of an evaluation: its first
// kernel's first workgroup writes it, all on one XCD. (An event between two
// kernels kept the stream idle for 5.8 us: six of them were a sixth of an
// evaluation of 10,000 particles.)
constexpr int kCounters = 3;
enum { PHASE_KEYS, PHASE_SORT, PHASE_TREE, PHASE_COM, PHASE_WALK, PHASE_END, kPhases };

__device__ inline void phase_begins(unsigned long long* __restrict__ counters, int phase) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        counters[kCounters + phase] = static_cast<unsigned long long>(wall_clock64());
    }
}

// The first workgroup also clears the build's flag words and the walk's
// counters (interactions, deferred queries), which only later kernels touch.
template <typename In>
__global__ __launch_bounds__(kThreads) void bbox_partial_kernel(
    const double* __restrict__ px, const double* __restrict__ py, const double* __restrict__ pz,
    const double* __restrict__ m, In* __restrict__ b4, int n, double* __restrict__ partial,
    unsigned* __restrict__ flags, int flag_words, unsigned long long* __restrict__ counters) {
    __shared__ double s[6][kThreads];
    if (blockIdx.x == 0) {
        for (int k = threadIdx.x; k < flag_words; k += kThreads) {
            flags[k] = 0u;
        }
        if (threadIdx.x < kCounters) {
            counters[threadIdx.x] = 0ull;
        }
    }
    phase_begins(counters, PHASE_KEYS);
    const double4 p0 = widen(build_input<In>(px, py, pz, m, 0));
    double lo[3] = {p0.x, p0.y, p0.z};
    double hi[3] = {lo[0], lo[1], lo[2]};
    for (int i = blockIdx.x * kThreads + threadIdx.x; i < n; i += gridDim.x * kThreads) {
        const In v = build_input<In>(px, py, pz, m, i);
        b4[i] = v;
        const double4 q = widen(v);
        const double p[3] = {q.x, q.y, q.z};
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            if (p[a] < lo[a]) lo[a] = p[a];
            if (p[a] > hi[a]) hi[a] = p[a];
        }
    }
    block_bounds<kThreads>(lo, hi, s);
    if (threadIdx.x < 6) {
        partial[blockIdx.x * 6 + threadIdx.x] = s[threadIdx.x][0];
    }
}

// The cube of every block's partial bounds, into LDS `cube` (centre xyz, half),
// by a whole workgroup; barnes_hut.c:471-483.
template <int T>
__device__ inline void block_root(const double* __restrict__ partial, int blocks,
                                  double (*s)[T], double* cube) {
    double lo[3] = {partial[0], partial[1], partial[2]};
    double hi[3] = {partial[3], partial[4], partial[5]};
    for (int b = threadIdx.x; b < blocks; b += T) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const double l = partial[b * 6 + a], h = partial[b * 6 + 3 + a];
            if (l < lo[a]) lo[a] = l;
            if (h > hi[a]) hi[a] = h;
        }
    }
    block_bounds<T>(lo, hi, s);
    if (threadIdx.x == 0) {
        const double l[3] = {s[0][0], s[1][0], s[2][0]};
        const double h[3] = {s[3][0], s[4][0], s[5][0]};
        double half = 0.5 * (h[0] - l[0]);
        const double hy = 0.5 * (h[1] - l[1]);
        const double hz = 0.5 * (h[2] - l[2]);
        if (hy > half) half = hy;
        if (hz > half) half = hz;
        if (half == 0.0) half = 0.5;
        half *= 1.0 + 1.0e-9;
        cube[0] = 0.5 * (l[0] + h[0]);
        cube[1] = 0.5 * (l[1] + h[1]);
        cube[2] = 0.5 * (l[2] + h[2]);
        cube[3] = half;
    }
    __syncthreads();
}

// ---------------------------------------------------------------- keys
// True-path key of every particle. Every workgroup first reduces the block
// bounds to the root cube itself (a launch of its own took 4.4 us at 10,000
// particles and 4.8 us at 1M); the first writes it.
template <typename In>
__global__ __launch_bounds__(kThreads) void keys_kernel(const In* __restrict__ b4, int n,
                                                        const double* __restrict__ partial,
                                                        int bb_blocks, double* __restrict__ root,
                                                        uint64_t* __restrict__ key) {
    __shared__ double s[6][kThreads];
    __shared__ double cube[4];
    block_root<kThreads>(partial, bb_blocks, s, cube);
    if (blockIdx.x == 0 && threadIdx.x < 4) {
        root[threadIdx.x] = cube[threadIdx.x];
    }
    for (int i = blockIdx.x * kThreads + threadIdx.x; i < n; i += gridDim.x * kThreads) {
        const double4 p = widen(b4[i]);
        double cx = cube[0], cy = cube[1], cz = cube[2], h = cube[3];
        key[i] = path_word(p.x, p.y, p.z, cx, cy, cz, h);
    }
}

// Morton key (barnes_hut.c:286-305).
__device__ inline uint64_t morton_key(const double4& p, const double* __restrict__ root) {
    const double cx = root[0], cy = root[1], cz = root[2], h = root[3];
    return spread3(axis_code(p.x, cx, h)) | (spread3(axis_code(p.y, cy, h)) << 1) |
           (spread3(axis_code(p.z, cz, h)) << 2);
}

// Only the parity probes and the node export read the Morton order; they
// compute it from the last build's inputs.
template <typename In>
__global__ void morton_keys_kernel(const In* __restrict__ b4, int n,
                                   const double* __restrict__ root, uint64_t* __restrict__ mkey,
                                   uint64_t* __restrict__ sortkey, uint32_t* __restrict__ idx) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        const uint64_t k = morton_key(widen(b4[i]), root);
        mkey[i] = k;
        sortkey[i] = k;
        idx[i] = static_cast<uint32_t>(i);
    }
}

// Octant digit of the cell (cx, cy, cz, h) that holds p; moves to that child.
__device__ inline int path_step(const double4& p, double& cx, double& cy, double& cz, double& h) {
    const int o = (p.x > cx ? 1 : 0) | (p.y > cy ? 2 : 0) | (p.z > cz ? 4 : 0);
    const double off = h * 0.5;
    cx = cx + ((o & 1) ? off : -off);
    cy = cy + ((o & 2) ? off : -off);
    cz = cz + ((o & 4) ? off : -off);
    h = off;
    return o;
}

// Order of two particles that share all 21 digits of the key: the sign of the
// first difference further down (0: none within kMaxLevels levels).
__device__ inline int deep_order(const double4& a, const double4& b,
                                 const double* __restrict__ root) {
    double cx = root[0], cy = root[1], cz = root[2], h = root[3];
    for (int d = 0; d < kMaxLevels; ++d) {
        double ux = cx, uy = cy, uz = cz, uh = h;
        const int oa = path_step(a, cx, cy, cz, h);
        const int ob = path_step(b, ux, uy, uz, uh);
        if (oa != ob) {
            return oa < ob ? -1 : 1;
        }
    }
    return 0;
}

// ext[k] = octant digits of levels 21(k+1) .. 21(k+1)+20 of one particle.
__device__ inline void extension_words(const double4& p, const double* __restrict__ root,
                                       uint64_t* __restrict__ ext) {
    double cx = root[0], cy = root[1], cz = root[2], h = root[3];
    path_word(p.x, p.y, p.z, cx, cy, cz, h);
    for (int k = 0; k < kExtWords; ++k) {
        ext[k] = path_word(p.x, p.y, p.z, cx, cy, cz, h);
    }
}

// Tree position t: the tree is laid out in descending key order. The tree-order
// inputs: FP32 s4 always, FP64 sp4 for FP64 inputs only (an FP32 build widens
// s4 where it needs FP64).
template <typename In>
__device__ inline void place(int t, uint64_t key, uint32_t o, const In* __restrict__ b4,
                             uint32_t* __restrict__ tperm, uint64_t* __restrict__ tword,
                             double4* __restrict__ sp4, float4* __restrict__ s4) {
    tperm[t] = o;
    tword[t] = key;
    const In p = b4[o];
    if constexpr (std::is_same_v<In, float4>) {
        s4[t] = p;
    } else {
        sp4[t] = p;
        s4[t] = make_float4(static_cast<float>(p.x), static_cast<float>(p.y),
                            static_cast<float>(p.z), static_cast<float>(p.w));
    }
}

// Large systems: radix passes on the top kSortTopBits key bits (levels 0..11:
// four of the seven 9-bit passes); order_kernel then orders each run of equal
// top bits by the low kSortLowBits and puts every particle at its tree
// position. The runs are short (two-galaxy input: at most 10 particles at 1M,
// 53 at 10M). A run longer than kFinishRun raises FLAG_LONG_RUN: the host, after
// reading the flags, sorts on all 63 bits (an escaper far out is enough: a
// Plummer sphere of 100,000 and one particle at 600 scale radii), and only where
// more than kFinishRun particles share a whole key on the extension words too.
// (Measured on MI355X, that input: 0.49 ms an evaluation, 0.30 without the
// escaper; 1.25 with the extension words of every particle sorted at once.)
constexpr int kSortLowBits = 27;
constexpr int kSortTopBits = 63 - kSortLowBits;
constexpr int kFinishRun = 64;
static_assert(kSortTopBits % 9 == 0, "whole 9-bit radix passes");

// Input: sorted (stably, from index order) by key >> low_bits. Element p
// goes to its run's first position plus the number of run members before it
// in key order. Members that share the whole key are ordered by their deeper
// digits, and each takes one of `slots` slots of ext for its extension words
// (nobody reads a position's words unless it shares its key with a neighbour).
// (Two of 25 evaluations of the 10M two-galaxy input hold such a pair; sorting
// all extension words of all particles took 8 ms each time.) Too few slots, or
// a run longer than kFinishRun, whose elements stay where they are (the output
// is still a permutation), raise the flag.
template <typename In>
__global__ __launch_bounds__(kThreads) void order_kernel(
    const uint64_t* __restrict__ kin, const uint32_t* __restrict__ vin, int n,
    const In* __restrict__ b4, const double* __restrict__ root, uint32_t* __restrict__ tperm,
    uint64_t* __restrict__ tword, uint64_t* __restrict__ ext, uint32_t* __restrict__ slot,
    unsigned slots, double4* __restrict__ sp4, float4* __restrict__ s4,
    unsigned* __restrict__ flags, int low_bits) {
    const int p = blockIdx.x * kThreads + threadIdx.x;
    if (p >= n) {
        return;
    }
    const uint64_t key = kin[p];
    const uint64_t top = key >> low_bits;
    // the run's bounds, at most kFinishRun steps to each side
    int a = p;
    while (a > 0 && p - a < kFinishRun && (kin[a - 1] >> low_bits) == top) {
        --a;
    }
    int b = p;
    while (b < n - 1 && b - p < kFinishRun && (kin[b + 1] >> low_bits) == top) {
        ++b;
    }
    int dst = p;
    bool tied = false;
    const uint32_t o = vin[p];
    if (b - a + 1 > kFinishRun) {
        // every member of a run this long sees a window of more than
        // kFinishRun positions, so the whole run stays in place
        atomicOr(&flags[FLAG_LONG_RUN], ORDER_RUN);
    } else {
        int rank = 0;
        for (int q = a; q <= b; ++q) {
            const uint64_t kq = kin[q];
            bool before = kq < key;
            if (kq == key && q != p) {
                tied = true;
                const int c = deep_order(widen(b4[vin[q]]), widen(b4[o]), root);
                before = c < 0 || (c == 0 && q < p);
            }
            rank += before ? 1 : 0;
        }
        dst = a + rank;
    }
    const int t = n - 1 - dst;
    place(t, key, o, b4, tperm, tword, sp4, s4);
    if (tied) {
        const unsigned k = atomicAdd(&flags[kTiedCount], 1u);
        if (k < slots) {
            slot[t] = k;
            extension_words(widen(b4[o]), root, ext + static_cast<size_t>(k) * kExtWords);
        } else {
            atomicOr(&flags[FLAG_LONG_RUN], ORDER_SLOTS);
        }
    }
}

// Small systems (up to kSmallSort): two launches order them. Each workgroup
// computes the keys of a tile of kSortTile1 particles and sorts them by (key,
// index) with a bitonic network, strides below a wave through lane exchanges;
// then every element's position is its rank in its own tile plus, by binary
// search, its rank in every other one. (The radix passes are twelve launches:
// 56 us at 10,000 particles.)
constexpr int kSortTile1 = 1024;
constexpr int kSmallSort = 1 << 15;

// Lane exchange by DPP and row swaps (no LDS), M a power of two below 64.
template <int M>
__device__ inline unsigned lane_xor(unsigned v, int lane) {
    const int i = static_cast<int>(v);
    if constexpr (M == 1) {
        return __builtin_amdgcn_update_dpp(0, i, 0xB1, 0xf, 0xf, true);    // quad_perm 1,0,3,2
    } else if constexpr (M == 2) {
        return __builtin_amdgcn_update_dpp(0, i, 0x4E, 0xf, 0xf, true);    // quad_perm 2,3,0,1
    } else if constexpr (M == 4) {
        const int h = __builtin_amdgcn_update_dpp(0, i, 0x141, 0xf, 0xf, true);   // xor 7
        return __builtin_amdgcn_update_dpp(0, h, 0x1B, 0xf, 0xf, true);           // xor 3
    } else if constexpr (M == 8) {
        return __builtin_amdgcn_update_dpp(0, i, 0x128, 0xf, 0xf, true);   // row_ror:8
    } else if constexpr (M == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
        return (lane & 16) != 0 ? r[0] : r[1];
    } else {
        const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
        return (lane & 32) != 0 ? r[0] : r[1];
    }
}

constexpr int kSortItems = kSortTile1 / kThreads;   // consecutive elements of a thread

struct SortItem {
    uint64_t key;
    uint32_t val;
};

// Keeps the smaller (take_low) or larger of the two in `a`.
__device__ inline void keep(SortItem& a, const SortItem& b, bool take_low) {
    const bool less = b.key < a.key || (b.key == a.key && b.val < a.val);
    if (less == take_low) {
        a = b;
    }
}

// One bitonic step of `size` at `stride` over the tile's elements 4 tid + r.
template <int SIZE, int STRIDE>
__device__ inline void bitonic_step(SortItem (&e)[kSortItems], int tid, uint64_t* skey,
                                    uint32_t* sval) {
    if constexpr (STRIDE < kSortItems) {
#pragma unroll
        for (int r = 0; r < kSortItems; ++r) {
            if ((r & STRIDE) == 0) {
                const bool up = ((tid * kSortItems + r) & SIZE) == 0;
                const SortItem lo = e[r], hi = e[r | STRIDE];
                keep(e[r], hi, up);
                keep(e[r | STRIDE], lo, !up);
            }
        }
    } else {
        constexpr int M = STRIDE / kSortItems;   // thread distance
        const bool low = (tid & M) == 0;
        const bool up = ((tid * kSortItems) & SIZE) == 0;
        SortItem o[kSortItems];
        if constexpr (M < kWave) {
#pragma unroll
            for (int r = 0; r < kSortItems; ++r) {
                const unsigned kl = lane_xor<M>(static_cast<unsigned>(e[r].key), tid);
                const unsigned kh = lane_xor<M>(static_cast<unsigned>(e[r].key >> 32), tid);
                o[r].key = static_cast<uint64_t>(kh) << 32 | kl;
                o[r].val = lane_xor<M>(e[r].val, tid);
            }
        } else {
#pragma unroll
            for (int r = 0; r < kSortItems; ++r) {
                skey[r * kThreads + tid] = e[r].key;
                sval[r * kThreads + tid] = e[r].val;
            }
            __syncthreads();
#pragma unroll
            for (int r = 0; r < kSortItems; ++r) {
                o[r].key = skey[r * kThreads + (tid ^ M)];
                o[r].val = sval[r * kThreads + (tid ^ M)];
            }
            __syncthreads();
        }
#pragma unroll
        for (int r = 0; r < kSortItems; ++r) {
            keep(e[r], o[r], low == up);
        }
    }
}

template <int SIZE, int STRIDE>
__device__ inline void bitonic_merge(SortItem (&e)[kSortItems], int tid, uint64_t* skey,
                                     uint32_t* sval) {
    bitonic_step<SIZE, STRIDE>(e, tid, skey, sval);
    if constexpr (STRIDE > 1) {
        bitonic_merge<SIZE, STRIDE / 2>(e, tid, skey, sval);
    }
}

template <int SIZE>
__device__ inline void bitonic_sort(SortItem (&e)[kSortItems], int tid, uint64_t* skey,
                                    uint32_t* sval) {
    if constexpr (SIZE > 2) {
        bitonic_sort<SIZE / 2>(e, tid, skey, sval);
    }
    bitonic_merge<SIZE, SIZE / 2>(e, tid, skey, sval);
}

template <typename In>
__global__ __launch_bounds__(kThreads) void tile_sort_kernel(
    const In* __restrict__ b4, int n, const double* __restrict__ partial, int bb_blocks,
    double* __restrict__ root, uint64_t* __restrict__ kout, uint32_t* __restrict__ vout,
    unsigned long long* __restrict__ counters) {
    phase_begins(counters, PHASE_SORT);
    __shared__ double s[6][kThreads];
    __shared__ double cube[4];
    __shared__ uint64_t skey[kSortTile1];
    __shared__ uint32_t sval[kSortTile1];
    const int tid = threadIdx.x;
    const int base = blockIdx.x * kSortTile1 + tid * kSortItems;
    double4 p[kSortItems];
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) {
        p[r] = widen(b4[base + r < n ? base + r : n - 1]);
    }
    block_root<kThreads>(partial, bb_blocks, s, cube);
    if (blockIdx.x == 0 && tid < 4) {
        root[tid] = cube[tid];
    }
    SortItem e[kSortItems];
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) {
        double cx = cube[0], cy = cube[1], cz = cube[2], h = cube[3];
        const uint64_t key = path_word(p[r].x, p[r].y, p[r].z, cx, cy, cz, h);
        // past the end: after every key (63 bits)
        e[r].key = base + r < n ? key : ~0ull;
        e[r].val = base + r < n ? static_cast<uint32_t>(base + r) : 0xFFFFFFFFu;
    }
    bitonic_sort<kSortTile1>(e, tid, skey, sval);
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) {
        if (base + r < n) {   // the padding sorted behind every element of the last tile
            kout[base + r] = e[r].key;
            vout[base + r] = e[r].val;
        }
    }
}

// kMergeLanes lanes per element, each searching every kMergeLanes-th tile.
constexpr int kMergeLanes = 4;
template <typename In>
__global__ __launch_bounds__(kThreads) void merge_order_kernel(
    const uint64_t* __restrict__ kin, const uint32_t* __restrict__ vin, int n,
    const In* __restrict__ b4, uint32_t* __restrict__ tperm, uint64_t* __restrict__ tword,
    double4* __restrict__ sp4, float4* __restrict__ s4) {
    const int slot = blockIdx.x * kThreads + threadIdx.x;
    const int q = slot % kMergeLanes;
    const int p = slot / kMergeLanes < n ? slot / kMergeLanes : n - 1;
    const int own = p / kSortTile1;
    const int tiles = (n + kSortTile1 - 1) / kSortTile1;
    const uint64_t key = kin[p];
    const uint32_t o = vin[p];
    int rank = q == 0 ? p - own * kSortTile1 : 0;
    // Elements of an earlier tile with an equal key come first (their indices
    // are smaller): count keys below key + 1 there, below key in later tiles.
    constexpr int kAtOnce = 4;   // independent searches in flight
    for (int t0 = q; t0 < tiles; t0 += kAtOnce * kMergeLanes) {
        int lo[kAtOnce], len[kAtOnce], first[kAtOnce];
        uint64_t lim[kAtOnce];
#pragma unroll
        for (int u = 0; u < kAtOnce; ++u) {
            const int t = t0 + u * kMergeLanes;
            lo[u] = t * kSortTile1;
            lim[u] = key + (t < own ? 1u : 0u);
            len[u] = t < tiles && t != own ? min(kSortTile1, n - lo[u]) : 0;
            first[u] = 0;
        }
#pragma unroll 1
        for (int step = kSortTile1; step > 0; step >>= 1) {
            uint64_t v[kAtOnce];
#pragma unroll
            for (int u = 0; u < kAtOnce; ++u) {
                v[u] = kin[first[u] + step <= len[u] ? lo[u] + first[u] + step - 1 : p];
            }
#pragma unroll
            for (int u = 0; u < kAtOnce; ++u) {
                first[u] += first[u] + step <= len[u] && v[u] < lim[u] ? step : 0;
            }
        }
#pragma unroll
        for (int u = 0; u < kAtOnce; ++u) {
            rank += first[u];
        }
    }
#pragma unroll
    for (int off = 1; off < kMergeLanes; off <<= 1) {
        rank += __shfl_xor(rank, off);
    }
    if (q == 0 && slot / kMergeLanes < n) {
        place(n - 1 - rank, key, o, b4, tperm, tword, sp4, s4);
    }
}

// ---- ordering on the extension words too (FLAG_LONG_RUN after a sort on all the
// key bits, or FLAG_TIE of a small system)
template <typename In>
__global__ void ext_words_kernel(const In* __restrict__ b4, int n,
                                 const double* __restrict__ root, uint64_t* __restrict__ ext) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        extension_words(widen(b4[i]), root, ext + static_cast<size_t>(i) * kExtWords);
    }
}

__global__ void gather_u64_kernel(const uint64_t* __restrict__ src, const uint32_t* __restrict__ idx,
                                  uint64_t* __restrict__ dst, int n, int stride, int offset) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < n) {
        dst[p] = src[static_cast<size_t>(idx[p]) * stride + offset];
    }
}

__global__ void iota_kernel(uint32_t* __restrict__ out, int n) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < n) {
        out[p] = static_cast<uint32_t>(p);
    }
}

// Tree positions from an ascending order of the original indices.
template <typename In>
__global__ void place_kernel(const uint32_t* __restrict__ order, const uint64_t* __restrict__ key,
                             const uint64_t* __restrict__ ext, int n, const In* __restrict__ b4,
                             uint32_t* __restrict__ tperm, uint64_t* __restrict__ tword,
                             uint64_t* __restrict__ ext_tree, double4* __restrict__ sp4,
                             float4* __restrict__ s4) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) {
        return;
    }
    const uint32_t o = order[n - 1 - t];
    place(t, key[o], o, b4, tperm, tword, sp4, s4);
    for (int w = 0; w < kExtWords; ++w) {
        ext_tree[static_cast<size_t>(t) * kExtWords + w] =
            ext[static_cast<size_t>(o) * kExtWords + w];
    }
}

// ---------------------------------------------------------------- topology
// Internal cells are numbered by level index L = doff[d] + k: the k-th cell of
// depth d in tree order (doff = exclusive prefix of the per-depth counts). Tree
// position t starts the cells of depths (delta[t-1], delta[t]] and ends those
// of depths (delta[t], delta[t-1]]; cells of one depth are disjoint, so the
// k-th start of depth d and the k-th end of depth d belong to the same cell.
// The topology kernels give each workgroup one tile of 256 to 1024 consecutive
// positions: per-tile counts of starts and ends per depth, scanned over the
// tiles, plus wave ballots inside a tile, give every start and end its rank
// in position order, with no search and no shared global counters.
//
// A small system is the chain of one tile (its levels, deepest first), so its
// tiles are shorter; a large one has several tiles a CU, and longer ones leave
// fewer cells that span tiles. Measured on MI355X, tree and centre-of-mass
// phases, two-galaxy / uniform cloud, us with tiles of 256, 512 and 1024:
//   8,000    50 / 41, 52 / 43, 58 / 48       24,000   65 / 51, 54 / 45, 65 / 53
//   60,000   69 / 57, 67 / 55, 68 / 56       200,000  80 / 67, 76 / 68, 82 / 72
//   400,000  101 / 90, 99 / 86, 90 / 79
// (256 up to the 64 tiles that one workgroup's span launch covers.)
template <int POSITIONS, int THREADS>
struct Tile {
    static constexpr int kPositions = POSITIONS;
    static constexpr int kBuildThreads = THREADS;                  // of build_kernel
    static constexpr int kBuildItems = POSITIONS / THREADS;
    static constexpr int kBuildWaves = THREADS / kWave;
    static constexpr int kChunks = POSITIONS / kWave;              // 64-position chunks
    static constexpr int kLocalCells = POSITIONS / 4 * 3;   // cells a tile can hold in LDS
                                                            // (usually about half as many as
                                                            // positions)
    static_assert(POSITIONS % kThreads == 0 && POSITIONS % THREADS == 0, "whole items");
};
using TileSmall = Tile<256, 256>;
using TileMedium = Tile<512, 512>;
using TileLarge = Tile<1024, 512>;
constexpr int kTopoWaves = kThreads / kWave;
constexpr int kSpanTiles = 64;   // tiles of a span_com_kernel workgroup

// Positions of a tile for n particles.
inline int tile_positions(size_t n, int cu_count) {
    return n <= static_cast<size_t>(kSpanTiles) * TileSmall::kPositions ? TileSmall::kPositions
           : n <= static_cast<size_t>(cu_count) * TileLarge::kPositions ? TileMedium::kPositions
                                                                        : TileLarge::kPositions;
}

// f(Tile) for that choice.
template <typename F>
auto with_tile(int positions, F f) {
    return positions == TileSmall::kPositions    ? f(TileSmall{})
           : positions == TileMedium::kPositions ? f(TileMedium{})
                                                 : f(TileLarge{});
}
// Rows of the per-tile counts: cells started and ended per depth, and all the
// cells started.
constexpr int kEndRow = kMaxLevels;
constexpr int kCellRow = 2 * kMaxLevels;
constexpr int kTopoRows = 2 * kMaxLevels + 1;


// Whether an earlier kernel of this build found something the host has to
// handle first (the tree is not valid then): later kernels of the evaluation
// do nothing, and the host, which reads the flags once at the end, repeats
// the part.
__device__ inline bool build_failed(const unsigned* __restrict__ flags) {
    const uint4 f = *reinterpret_cast<const uint4*>(flags);
    return (f.x | f.y | f.z | f.w) != 0;
}

// Internal cells by level index.
struct InternalSoA {
    double4* com;     // FP64 centre of mass (x, y, z) and mass
    int4* rec;        // node index, skip (node index past the subtree), first and last tree position
    int32_t* depth;
};

__device__ inline int wave_min_int(int v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const int o = __shfl_xor(v, off);
        v = o < v ? o : v;
    }
    return v;
}

__device__ inline int wave_max_int(int v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const int o = __shfl_xor(v, off);
        v = o > v ? o : v;
    }
    return v;
}

// delta[t] = common levels of tree positions t and t+1 (-1 for the last);
// tile_hist[row * tiles + b] = tile b's counts.
template <int POSITIONS>
__global__ __launch_bounds__(kThreads) void delta_kernel(const uint64_t* __restrict__ w,
                                                        ExtTable ext, int n,
                                                        int tiles, int32_t* __restrict__ delta,
                                                        unsigned* __restrict__ flags,
                                                        unsigned* __restrict__ tile_hist,
                                                        unsigned long long* __restrict__ counters) {
    __shared__ unsigned hist[kTopoRows];
    __shared__ unsigned tile_flags;
    phase_begins(counters, PHASE_TREE);
    if (build_failed(flags)) {
        return;
    }
    for (int d = threadIdx.x; d < kTopoRows; d += kThreads) {
        hist[d] = 0;
    }
    if (threadIdx.x == 0) {
        tile_flags = 0;
    }
    __syncthreads();
    unsigned mine = 0;
    int cells = 0;
    for (int i = 0; i < POSITIONS / kThreads; ++i) {
        const int t = blockIdx.x * POSITIONS + i * kThreads + threadIdx.x;
        if (t >= n) {
            break;
        }
        const int dprev = t > 0 ? common_levels(w, ext, t - 1, t) : -1;
        const int dcur = t < n - 1 ? common_levels(w, ext, t, t + 1) : -1;
        delta[t] = dcur;
        cells += dcur > dprev ? dcur - dprev : 0;
        const int top = dcur < kMaxLevels ? dcur : kMaxLevels - 1;
        for (int d = dprev + 1; d <= top; ++d) {
            atomicAdd(&hist[d], 1u);
        }
        const int etop = dprev < kMaxLevels ? dprev : kMaxLevels - 1;
        for (int d = dcur + 1; d <= etop; ++d) {
            atomicAdd(&hist[kEndRow + d], 1u);
        }
        if (ext.words == nullptr && dcur >= 21) {
            mine |= 1u;
        }
        if (dcur >= kMaxLevels) {
            mine |= 2u;
        }
    }
    if (cells != 0) {
        atomicAdd(&hist[kCellRow], static_cast<unsigned>(cells));
    }
    if (mine != 0) {
        atomicOr(&tile_flags, mine);
    }
    __syncthreads();
    for (int d = threadIdx.x; d < kTopoRows; d += kThreads) {
        tile_hist[static_cast<size_t>(d) * tiles + blockIdx.x] = hist[d];
    }
    if (threadIdx.x == 0) {
        if (tile_flags & 1u) {
            atomicOr(&flags[FLAG_TIE], 1u);
        }
        if (tile_flags & 2u) {
            atomicOr(&flags[FLAG_OVERFLOW], 1u);
        }
    }
}

// One workgroup per row: tile_base[row * tiles + b] = sum of
// tile_hist[row * tiles + b'] over b' < b; dcount[d] = the depth's cell count,
// dcount[kMaxLevels] = all cells.
__global__ __launch_bounds__(kThreads) void depth_scan_kernel(const unsigned* __restrict__ tile_hist,
                                                             int tiles,
                                                             unsigned* __restrict__ tile_base,
                                                             unsigned* __restrict__ flags) {
    __shared__ unsigned wave_sum[kTopoWaves];
    if (build_failed(flags)) {
        return;
    }
    const int row_id = blockIdx.x;
    const unsigned* row = tile_hist + static_cast<size_t>(row_id) * tiles;
    unsigned* out = tile_base + static_cast<size_t>(row_id) * tiles;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    unsigned running = 0;
    for (int base = 0; base < tiles; base += kThreads) {
        const int i = base + threadIdx.x;
        const unsigned v = i < tiles ? row[i] : 0u;
        unsigned x = v;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const unsigned y = __shfl_up(x, off, 64);
            if (lane >= off) {
                x += y;
            }
        }
        if (lane == 63) {
            wave_sum[wv] = x;
        }
        __syncthreads();
        unsigned before = running, total = 0;
#pragma unroll
        for (int k = 0; k < kTopoWaves; ++k) {
            const unsigned ws = wave_sum[k];
            before += k < wv ? ws : 0u;
            total += ws;
        }
        if (i < tiles) {
            out[i] = before + x - v;
        }
        running += total;
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        if (row_id < kMaxLevels) {
            flags[kDCount + row_id] = running;
        } else if (row_id == kCellRow) {
            flags[kDCount + kMaxLevels] = running;
        }
    }
}

// Exclusive offsets of the per-depth level-index ranges, into LDS, by the
// block's first wave (depth pairs per lane, one wave scan). Callers
// synchronise before reading them.
static_assert(kMaxLevels <= 2 * 64 + 1, "depth offsets: two depths per lane plus one");
__device__ inline void depth_offsets(const unsigned* __restrict__ dcount, unsigned* doff) {
    if (threadIdx.x >= 64) {
        return;
    }
    const int l = threadIdx.x;
    const unsigned v0 = 2 * l < kMaxLevels ? dcount[2 * l] : 0u;
    const unsigned v1 = 2 * l + 1 < kMaxLevels ? dcount[2 * l + 1] : 0u;
    const unsigned pair = v0 + v1;
    unsigned incl = pair;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const unsigned y = __shfl_up(incl, off, 64);
        if (l >= off) {
            incl += y;
        }
    }
    const unsigned excl = incl - pair;
    if (2 * l < kMaxLevels) {
        doff[2 * l] = excl;
    }
    if (2 * l + 1 < kMaxLevels) {
        doff[2 * l + 1] = excl + v0;
    }
    if (l == 63 && 2 * 64 < kMaxLevels) {
        doff[2 * 64] = incl;
    }
}

// The FP32 pre-order record of a leaf (tree position t, node index li) and of
// an internal cell (level index L, its FP64 centre of mass and mass, half
// size h, pre-order skip). Only the per-query walks read these records, so
// node_records_kernel writes them on demand after the build.
__device__ inline NodeF32 leaf_record(const float4& q, int li, int t) {
    NodeF32 b;
    b.cx = q.x;
    b.cy = q.y;
    b.cz = q.z;
    b.m = q.w;
    b.size2 = 0.f;
    b.skip = li + 1;
    b.leaf = t;
    b.inv_size2 = 0.f;
    return b;
}

__device__ inline NodeF32 cell_record(const double4& c, double h, int skip, int L) {
    NodeF32 b;
    b.cx = static_cast<float>(c.x);
    b.cy = static_cast<float>(c.y);
    b.cz = static_cast<float>(c.z);
    b.m = static_cast<float>(c.w);
    b.size2 = static_cast<float>(4.0 * h * h);
    b.skip = skip;
    b.leaf = -(L + 2);   // internal: -(level index + 2)
    b.inv_size2 = 1.f / b.size2;
    return b;
}

// What the centre-of-mass pass reads and writes.
template <typename In>
struct CellData {
    GroupNode* gnode;
    InternalSoA in;
    const In* sp4;          // tree-order particles
    const In* b4;           // original order
    const uint32_t* tperm;
    const double* root;
    NodeF64* n64;           // FP64 records (FP64 builds)
    double* im2;            // second moments and quadrupole records (learned path)
    float4* gquad;

    // (x, y, z, mass) of a child table entry, by two 16-byte loads whatever it
    // is (no branch per child, so a cell's loads do not wait for each other).
    __device__ double4 child(int k) const {
        const char* cell = reinterpret_cast<const char*>(in.com + (k >= 0 ? k : 0));
        const char* leaf = reinterpret_cast<const char*>(sp4 + (k < -1 ? -k - 2 : 0));
        const uint4 lo = *reinterpret_cast<const uint4*>(k < -1 ? leaf : cell);
        const uint4 hi = *reinterpret_cast<const uint4*>((k < -1 ? leaf : cell) +
                                                         (k < -1 ? sizeof(In) - 16 : 16));
        double4 q = make_double4(__hiloint2double(lo.y, lo.x), __hiloint2double(lo.w, lo.z),
                                 __hiloint2double(hi.y, hi.x), __hiloint2double(hi.w, hi.z));
        if constexpr (std::is_same_v<In, float4>) {
            if (k < -1) {
                q = make_double4(__uint_as_float(lo.x), __uint_as_float(lo.y),
                                 __uint_as_float(lo.z), __uint_as_float(lo.w));
            }
        }
        if (k == -1) {
            q = make_double4(0.0, 0.0, 0.0, 0.0);
        }
        return q;
    }
};

// The rest of a cell's centre-of-mass pass (barnes_hut.c:214-253) once its
// eight children's (x, y, z, mass) are known: summed in octant order 0..7 (an
// empty slot is zero mass at the origin, which leaves the sums bit for bit as
// skipping it would); a zero-mass cell keeps the position of the particle that
// created it (lowest Morton rank in the cell; for the root the caller's
// particle 0, barnes_hut.c:504-512). Writes every record of the cell but the
// child table and returns its (x, y, z, mass).
template <bool QUAD, typename In>
__device__ inline double4 finish_cell(int L, int depth, const double4 (&q)[8],
                                      const int (&kid)[8], const CellData<In>& c) {
    double mass = 0.0, x = 0.0, y = 0.0, z = 0.0;
#pragma unroll
    for (int o = 0; o < 8; ++o) {
        mass += q[o].w;
        x += q[o].w * q[o].x;
        y += q[o].w * q[o].y;
        z += q[o].w * q[o].z;
    }
    double ox, oy, oz;
    if (mass != 0.0) {
        ox = x / mass;
        oy = y / mass;
        oz = z / mass;
    } else {
        const int4 r = c.in.rec[L];
        double4 p;
        if (r.x == 0) {
            p = widen(c.b4[0]);
        } else {
            // the cell's particles are tree positions r.z .. r.w; the Morton
            // rank orders by (Morton key, original index)
            int minpos = r.z;
            uint64_t minkey = morton_key(widen(c.sp4[r.z]), c.root);
            for (int t = r.z + 1; t <= r.w; ++t) {
                const uint64_t k = morton_key(widen(c.sp4[t]), c.root);
                if (k < minkey || (k == minkey && c.tperm[t] < c.tperm[minpos])) {
                    minkey = k;
                    minpos = t;
                }
            }
            p = widen(c.sp4[minpos]);
        }
        ox = p.x;
        oy = p.y;
        oz = p.z;
    }
    const double4 com = make_double4(ox, oy, oz, mass);
    c.in.com[L] = com;
    const double h = ldexp(c.root[3], -depth);
    if (c.n64 != nullptr) {
        const int4 r = c.in.rec[L];
        NodeF64 a;
        a.cx = ox;
        a.cy = oy;
        a.cz = oz;
        a.m = mass;
        a.size2 = 4.0 * h * h;
        a.skip = r.y;
        a.leaf = -1;
        c.n64[r.x] = a;
    }
    const NodeF32 b = cell_record(com, h, 0, L);
    if (QUAD) {
        // second moment about the centre of mass from the children's
        // (parallel axes), FP64; the walk's traceless FP32 quadrupole
        double xx = 0.0, yy = 0.0, zz = 0.0, xy = 0.0, xz = 0.0, yz = 0.0;
        if (mass != 0.0) {
#pragma unroll
            for (int o = 0; o < 8; ++o) {
                const double dx = q[o].x - ox, dy = q[o].y - oy, dz = q[o].z - oz;
                xx += q[o].w * dx * dx;
                yy += q[o].w * dy * dy;
                zz += q[o].w * dz * dz;
                xy += q[o].w * dx * dy;
                xz += q[o].w * dx * dz;
                yz += q[o].w * dy * dz;
                if (kid[o] >= 0) {
                    const double* cm = c.im2 + 6 * static_cast<size_t>(kid[o]);
                    xx += cm[0];
                    yy += cm[1];
                    zz += cm[2];
                    xy += cm[3];
                    xz += cm[4];
                    yz += cm[5];
                }
            }
        }
        double* om = c.im2 + 6 * static_cast<size_t>(L);
        om[0] = xx;
        om[1] = yy;
        om[2] = zz;
        om[3] = xy;
        om[4] = xz;
        om[5] = yz;
        const double tr = xx + yy + zz;
        c.gquad[2 * L] = make_float4(static_cast<float>(3.0 * xx - tr),
                                     static_cast<float>(3.0 * yy - tr),
                                     static_cast<float>(3.0 * zz - tr),
                                     static_cast<float>(3.0 * xy));
        c.gquad[2 * L + 1] = make_float4(static_cast<float>(3.0 * xz),
                                         static_cast<float>(3.0 * yz), b.size2, b.inv_size2);
    }
    float4* g = reinterpret_cast<float4*>(c.gnode + L);
    g[0] = make_float4(b.cx, b.cy, b.cz, b.m);
    g[1] = make_float4(b.size2, b.inv_size2, 0.f, 0.f);
    return com;
}

__device__ inline void load_kids(const GroupNode* g, int (&kid)[8]) {
    const int4 k0 = reinterpret_cast<const int4*>(g)[2];
    const int4 k1 = reinterpret_cast<const int4*>(g)[3];
    kid[0] = k0.x;
    kid[1] = k0.y;
    kid[2] = k0.z;
    kid[3] = k0.w;
    kid[4] = k1.x;
    kid[5] = k1.y;
    kid[6] = k1.z;
    kid[7] = k1.w;
}

// A cell whose child table and children's records are in memory.
template <bool QUAD, typename In>
__device__ inline void com_node(int L, int depth, const CellData<In>& c) {
    int kid[8];
    load_kids(c.gnode + L, kid);
    double4 q[8];
#pragma unroll
    for (int o = 0; o < 8; ++o) {
        q[o] = c.child(kid[o]);   // all eight in flight together
    }
    finish_cell<QUAD, In>(L, depth, q, kid, c);
}

// Rank bookkeeping of one tile. wcount[k][chunk][d]: starts (k = 0) and ends
// (k = 1) of depth d in the earlier chunks of the tile; base and next: those
// of the earlier tiles, without and with this one; local: number of the
// tile's first cell of depth d among the cells it starts.
template <typename T>
struct TileRanks {
    unsigned short wcount[2][T::kChunks][kMaxLevels + 1];
    unsigned doff[kMaxLevels];
    unsigned base[2][kMaxLevels];
    unsigned next[2][kMaxLevels];
    unsigned local[kMaxLevels];
    unsigned chunk_cells[T::kChunks];
    int deepest;
    unsigned cells;
};

// The tile's part of the tree in LDS: its particles, and the child tables and
// centres of mass of the cells that start in it. A child is -1 for none, a
// position of the tile, or T::kPositions + the number of one of the tile's cells.
template <typename T>
struct TileCells {
    double4 item[T::kPositions + T::kLocalCells];
    short kids[T::kLocalCells][8];
};

// A workgroup barrier that orders LDS only: global stores stay in flight (a
// full barrier waits for every one of them, each level anew).
__device__ inline void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Slots lo .. hi - 1 of a child table have no child.
__device__ inline void empty_slots(int32_t* kids, int lo, int hi) {
    for (int o = lo; o < hi; ++o) {
        kids[o] = -1;
    }
}

// Every internal cell's record and child table, the FP64 walk records of the
// leaves (FP64 builds), the node numbering, and the centre of mass of the
// cells that lie within the tile (span_com_kernel does the others): one
// workgroup per tile.
//
// A cell's fields come from the position where it starts (node index, first
// position, depth) and the one where it ends (skip, last position). A
// position's cells are visited shallow to deep, so each one's parent is the
// cell visited just before it: the depth-delta[t-1] cell that holds t-1 and t
// (already started) for the shallowest, the previous one otherwise.
//
// A tile starts at most one cell per depth that runs past its end (cells of
// one depth are disjoint), the last it starts of that depth. All the others
// are local: their child tables and centres of mass are put together in LDS,
// deepest first, and written once. The child table gnode[L].kids of a cell
// that spans tiles (octant: an internal child's level index; a leaf child's
// -(tree position + 2); -1 for none) is written slot by slot by several
// workgroups: every child writes its own slot and the empty ones up to the
// child before it (children come in descending octant order), the cell's last
// position those below its last child. A tile with more than T::kLocalCells
// cells treats them all like that and sums the local ones from memory.
//
// Measured on MI355X: separate launches for ends, starts and every depth took
// 18 + 20 + 100 us at 1M, and at 10,000 particles 13 + 35 us.
template <bool QUAD, typename In, typename T>
__global__ __launch_bounds__(T::kBuildThreads, 4) void build_kernel(
    const uint64_t* __restrict__ w, ExtTable ext, const int32_t* __restrict__ delta, int n, int tiles, int cell_capacity,
    unsigned* __restrict__ flags, const unsigned* __restrict__ tile_base,
    uint32_t* __restrict__ scan, CellData<In> c) {
    constexpr int kTopoTile = T::kPositions, kTopoChunks = T::kChunks;
    constexpr int kBuildThreads = T::kBuildThreads, kBuildItems = T::kBuildItems;
    constexpr int kBuildWaves = T::kBuildWaves, kLocalCells = T::kLocalCells;
    __shared__ TileRanks<T> r;
    __shared__ TileCells<T> tc;
    if (build_failed(flags)) {
        return;
    }
    const unsigned* dcount = flags + kDCount;
    if (dcount[kMaxLevels] > static_cast<unsigned>(cell_capacity)) {
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            atomicOr(&flags[FLAG_CELLS], 1u);
        }
        return;   // every workgroup: the records would not fit
    }
    const int b = blockIdx.x;
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    for (int k = threadIdx.x; k < 2 * kTopoChunks * (kMaxLevels + 1); k += kBuildThreads) {
        (&r.wcount[0][0][0])[k] = 0;
    }
    for (int k = threadIdx.x; k < kLocalCells * 4; k += kBuildThreads) {
        reinterpret_cast<int*>(&tc.kids[0][0])[k] = -1;   // two empty slots
    }
    for (int k = threadIdx.x; k < 2 * kMaxLevels; k += kBuildThreads) {
        const int kind = k / kMaxLevels, d = k % kMaxLevels;
        const unsigned* row = tile_base + static_cast<size_t>(kind * kEndRow + d) * tiles;
        r.base[kind][d] = row[b];
        r.next[kind][d] = b + 1 < tiles ? row[b + 1] : dcount[d];
    }
    if (threadIdx.x == 0) {
        r.deepest = -1;
    }
    depth_offsets(dcount, r.doff);
    const unsigned tile_cells = tile_base[static_cast<size_t>(kCellRow) * tiles + b];
    // dp, dc: common levels with the previous and the next position
    int dp[kBuildItems], dc[kBuildItems], below[kBuildItems];
    uint64_t word[kBuildItems], before[kBuildItems];
    int deep = -1;
#pragma unroll
    for (int i = 0; i < kBuildItems; ++i) {
        const int u = i * kBuildThreads + threadIdx.x;
        const int t = b * kTopoTile + u;
        const bool valid = t < n;
        dp[i] = valid && t > 0 ? delta[t - 1] : -1;
        dc[i] = valid ? delta[t] : -1;
        word[i] = valid ? w[t] : 0;
        before[i] = valid && t > 0 ? w[t - 1] : 0;
        if (valid) {
            tc.item[u] = widen(c.sp4[t]);
        }
        deep = dc[i] > deep ? dc[i] : deep;
    }
    lds_barrier();   // counts cleared, base read
    deep = wave_max_int(deep);
    if (lane == 0) {
        atomicMax(&r.deepest, deep);
    }
#pragma unroll
    for (int i = 0; i < kBuildItems; ++i) {
        const int chunk = i * kBuildWaves + wave;
        const int wlo = wave_min_int(dp[i] != dc[i] ? min(dp[i], dc[i]) + 1 : 0x7FFFFFFF);
        const int whi = wave_max_int(dp[i] != dc[i] ? max(dp[i], dc[i]) : -1);
        for (int d = wlo; d <= whi; ++d) {
            const uint64_t ms = __ballot(dp[i] < d && d <= dc[i]);
            const uint64_t me = __ballot(dc[i] < d && d <= dp[i]);
            if (lane == 0) {
                r.wcount[0][chunk][d] = static_cast<unsigned short>(__popcll(ms));
                r.wcount[1][chunk][d] = static_cast<unsigned short>(__popcll(me));
            }
        }
        // cells started before this position in its chunk
        const int cells = dc[i] > dp[i] ? dc[i] - dp[i] : 0;
        int x = cells;
#pragma unroll
        for (int off = 1; off < kWave; off <<= 1) {
            const int y = __shfl_up(x, off);
            if (lane >= off) {
                x += y;
            }
        }
        below[i] = x - cells;
        if (lane == kWave - 1) {
            r.chunk_cells[chunk] = static_cast<unsigned>(x);
        }
    }
    lds_barrier();
    for (int k = threadIdx.x; k < 2 * kMaxLevels; k += kBuildThreads) {
        const int kind = k / kMaxLevels, d = k % kMaxLevels;
        unsigned run = 0;
#pragma unroll
        for (int h = 0; h < kTopoChunks; ++h) {
            const unsigned v = r.wcount[kind][h][d];
            r.wcount[kind][h][d] = static_cast<unsigned short>(run);
            run += v;
        }
    }
    if (threadIdx.x == kBuildThreads - 1) {
        unsigned run = 0;
        for (int h = 0; h < kTopoChunks; ++h) {
            const unsigned v = r.chunk_cells[h];
            r.chunk_cells[h] = run;
            run += v;
        }
    }
    if (threadIdx.x == kBuildThreads - 1 - kWave) {
        unsigned run = 0;
        for (int d = 0; d <= r.deepest; ++d) {
            r.local[d] = run;
            run += r.next[0][d] - r.base[0][d];
        }
        r.cells = run;
    }
    lds_barrier();
    const bool in_lds = r.cells <= static_cast<unsigned>(kLocalCells);
    // Child `ref` (its table entry in memory, its entry in LDS) of the cell of
    // rank `rank` at depth d, in octant o; `upto`: the octant of the child
    // before it, 8 for the first.
    auto put_child = [&](int d, unsigned rank, int o, int upto, int ref, int local_ref) {
        if (in_lds && rank >= r.base[0][d] && rank < r.next[1][d]) {
            tc.kids[r.local[d] + rank - r.base[0][d]][o] = static_cast<short>(local_ref);
        } else {
            int32_t* kids = c.gnode[r.doff[d] + rank].kids;
            kids[o] = ref;
            empty_slots(kids, o + 1, upto);
        }
    };
#pragma unroll
    for (int i = 0; i < kBuildItems; ++i) {
        const int chunk = i * kBuildWaves + wave;
        const int u = i * kBuildThreads + threadIdx.x;
        const int t = b * kTopoTile + u;
        const bool valid = t < n;
        const int lo = dp[i] + 1, hi = dc[i];
        const int cells = hi > dp[i] ? hi - dp[i] : 0;
        const uint32_t sc = tile_cells + r.chunk_cells[chunk] + static_cast<unsigned>(below[i]);
        const int li = static_cast<int>(sc) + cells + t;   // the leaf's node index
        auto digit = [&](uint64_t key, int pos, int level) {
            const uint64_t v = level < 21 ? key : ext.of(pos)[level / 21 - 1];
            return static_cast<int>((v >> (60 - 3 * (level % 21))) & 7u);
        };
        if (valid) {
            scan[t] = sc;
        }
        int parent = -1;   // rank of the parent in its depth
        const int wlo = wave_min_int(valid ? max(min(dp[i], hi + 1), 0) : 0x7FFFFFFF);
        const int whi = wave_max_int(valid ? max(dp[i], hi) : -1);
        for (int d = wlo; d <= whi; ++d) {
            const bool starts = valid && lo <= d && d <= hi;
            const bool ends = valid && hi < d && d <= dp[i];
            const uint64_t ms = __ballot(starts);
            const uint64_t me = __ballot(ends);
            if (starts || (valid && d == dp[i])) {
                // a start of its own, or the latest depth-dp start before t
                const int rank = static_cast<int>(r.base[0][d] + r.wcount[0][chunk][d] +
                                                  lanes_below(ms)) -
                                 (starts ? 0 : 1);
                if (starts) {
                    const int L = static_cast<int>(r.doff[d]) + rank;
                    int* rl = reinterpret_cast<int*>(c.in.rec + L);
                    rl[0] = static_cast<int>(sc) + t + (d - lo);
                    rl[2] = t;
                    c.in.depth[L] = d;
                    if (parent >= 0) {
                        const int number =
                            static_cast<int>(r.local[d] + static_cast<unsigned>(rank) - r.base[0][d]);
                        put_child(d - 1, static_cast<unsigned>(parent), digit(word[i], t, d - 1),
                                  d == lo ? digit(before[i], t - 1, d - 1) : 8, L,
                                  kTopoTile + number);
                    }
                }
                parent = rank;
            }
            if (ends) {
                const unsigned rank = r.base[1][d] + r.wcount[1][chunk][d] + lanes_below(me);
                const unsigned L = r.doff[d] + rank;
                int* rl = reinterpret_cast<int*>(c.in.rec + L);
                rl[1] = li + 1;
                rl[3] = t;
                if (!in_lds || rank < r.base[0][d]) {
                    empty_slots(c.gnode[L].kids, 0, digit(word[i], t, d));
                }
            }
        }
        if (valid) {
            const int level = dp[i] > hi ? dp[i] : hi;   // the parent's depth
            if (level >= 0 && parent >= 0) {
                put_child(level, static_cast<unsigned>(parent), digit(word[i], t, level),
                          hi > dp[i] ? 8 : digit(before[i], t - 1, level), -(t + 2), u);
            }
            if constexpr (std::is_same_v<In, double4>) {
                if (c.n64 != nullptr) {   // FP64 records only for the exact FP64 walk
                    const double4 q = tc.item[u];
                    NodeF64 a;
                    a.cx = q.x;
                    a.cy = q.y;
                    a.cz = q.z;
                    a.m = q.w;
                    a.size2 = 0.0;
                    a.skip = li + 1;
                    a.leaf = t;
                    c.n64[li] = a;
                }
            }
        }
    }
    bool synced = false;
    for (int d = r.deepest; d >= 0; --d) {
        // the cells of depth d that start and end in this tile
        const int first = static_cast<int>(r.base[0][d]);
        const int end = static_cast<int>(min(r.next[0][d], r.next[1][d]));
        if (first >= end) {
            continue;   // the same for the whole workgroup
        }
        // this tile's child tables, or the deeper cells, written; in memory
        // those of a tile too full for LDS, the ranges and skips before the
        // first level and the second moments
        if (QUAD || !in_lds || !synced) {
            __syncthreads();
            synced = true;
        } else {
            lds_barrier();
        }
        for (int k = first + threadIdx.x; k < end; k += kBuildThreads) {
            const int L = static_cast<int>(r.doff[d]) + k;
            if (!in_lds) {
                com_node<QUAD, In>(L, d, c);
                continue;
            }
            const int number = static_cast<int>(r.local[d]) + k - first;
            // level index minus number of the tile's depth d + 1 cells
            const int to_level = d + 1 <= r.deepest
                                     ? static_cast<int>(r.doff[d + 1] + r.base[0][d + 1]) -
                                           static_cast<int>(r.local[d + 1])
                                     : 0;
            int kid[8];
            double4 q[8];
#pragma unroll
            for (int o = 0; o < 8; ++o) {
                const int v = tc.kids[number][o];
                const double4 item = tc.item[v >= 0 ? v : 0];
                q[o].x = v < 0 ? 0.0 : item.x;
                q[o].y = v < 0 ? 0.0 : item.y;
                q[o].z = v < 0 ? 0.0 : item.z;
                q[o].w = v < 0 ? 0.0 : item.w;
                kid[o] = v < 0 ? -1
                               : (v >= kTopoTile ? to_level + v - kTopoTile
                                                 : -(b * kTopoTile + v + 2));
            }
            tc.item[kTopoTile + number] = finish_cell<QUAD, In>(L, d, q, kid, c);
            int4* g = reinterpret_cast<int4*>(c.gnode + L);
            g[2] = make_int4(kid[0], kid[1], kid[2], kid[3]);
            g[3] = make_int4(kid[4], kid[5], kid[6], kid[7]);
        }
    }
}

// Centre of mass of the cells that span tiles. A unit is unit_tiles tiles; a
// workgroup takes group_units units and the cells that run past the end of
// the unit they start in (at most one per unit and depth) and end within the
// workgroup's positions, deepest first. Two launches cover all: tiles in
// groups of kSpanTiles, then units of kSpanTiles tiles in one workgroup.
//
// One cell per thread: its children are read up front, all at once, but for
// those among the workgroup's own cells, whose centre of mass the thread
// takes from LDS when its depth's turn comes. (Finding and summing each
// depth's cells from memory: 46 and 33 us for the two launches at 1M.) More
// cells, units or depths than the tables hold are summed that way.
constexpr int kSpanLevels = 40;
template <int T>
struct SpanTable {
    int2 cell[T];                            // level index, depth
    double4 com[T];
    short at[kSpanLevels][T / 4];            // entry of depth d and unit u, or -1
    unsigned count;
    int deepest;
    unsigned doff[kMaxLevels];
    unsigned present[kMaxLevels];
};

template <bool QUAD, typename In, int T, int POSITIONS>
__global__ __launch_bounds__(T) void span_com_kernel(int unit_tiles, int group_units, int tiles,
                                                     const unsigned* __restrict__ flags,
                                                     const unsigned* __restrict__ tile_base,
                                                     CellData<In> c,
                                                     unsigned long long* __restrict__ counters) {
    __shared__ SpanTable<T> s;
    if (unit_tiles == 1) {
        phase_begins(counters, PHASE_COM);
    }
    if (build_failed(flags)) {
        return;
    }
    const unsigned* dcount = flags + kDCount;
    for (int d = threadIdx.x; d < kMaxLevels; d += T) {
        s.present[d] = 0;
    }
    for (int k = threadIdx.x; k < kSpanLevels * (T / 4); k += T) {
        (&s.at[0][0])[k] = -1;
    }
    if (threadIdx.x == 0) {
        s.deepest = -1;
        s.count = 0;
    }
    depth_offsets(dcount, s.doff);
    __syncthreads();
    for (int d = threadIdx.x; d < kMaxLevels; d += T) {
        if (dcount[d] != 0) {
            atomicMax(&s.deepest, d);
        }
    }
    __syncthreads();
    const int unit0 = blockIdx.x * group_units;
    const int units = min(group_units, (tiles + unit_tiles - 1) / unit_tiles - unit0);
    const int limit = min((unit0 + group_units) * unit_tiles, tiles) * POSITIONS;
    const int levels = s.deepest + 1;
    // level index of the cell of depth d that starts in unit u and ends past
    // it, or -1
    auto spanning = [&](int d, int u) {
        const int next = (unit0 + u + 1) * unit_tiles;
        if (next >= tiles) {
            return -1;   // every cell ends within the last unit
        }
        const unsigned* starts = tile_base + static_cast<size_t>(d) * tiles;
        const unsigned past = starts[next];
        const unsigned from = starts[(unit0 + u) * unit_tiles];
        const unsigned ended = tile_base[static_cast<size_t>(kEndRow + d) * tiles + next];
        if (past == from || past <= ended) {
            return -1;
        }
        const int L = static_cast<int>(s.doff[d] + past) - 1;
        return c.in.rec[L].w < limit ? L : -1;
    };
    const bool tabled = levels <= kSpanLevels && units <= T / 4;
    for (int k = threadIdx.x; k < levels * units; k += T) {
        const int d = k / units, u = k - d * units;
        const int L = spanning(d, u);
        if (L >= 0) {
            s.present[d] = 1;
            const unsigned e = atomicAdd(&s.count, 1u);
            if (tabled && e < T) {
                s.cell[e] = make_int2(L, d);
                s.at[d][u] = static_cast<short>(e);
            }
        }
    }
    __syncthreads();
    if (!tabled || s.count > T) {
        for (int d = levels - 1; d >= 0; --d) {
            if (s.present[d] == 0) {
                continue;   // the same for the whole workgroup
            }
            for (int u = threadIdx.x; u < units; u += T) {
                const int L = spanning(d, u);
                if (L >= 0) {
                    com_node<QUAD, In>(L, d, c);
                }
            }
            __syncthreads();
        }
        return;
    }
    int L = -1, depth = -1;
    int kid[8], own[8];
    double4 q[8];
    if (threadIdx.x < s.count) {
        L = s.cell[threadIdx.x].x;
        depth = s.cell[threadIdx.x].y;
        load_kids(c.gnode + L, kid);
        int first[8];
#pragma unroll
        for (int o = 0; o < 8; ++o) {
            q[o] = c.child(kid[o]);
            first[o] = c.in.rec[kid[o] >= 0 ? kid[o] : 0].z;
        }
#pragma unroll
        for (int o = 0; o < 8; ++o) {
            own[o] = -1;
            const int u = first[o] / (unit_tiles * POSITIONS) - unit0;
            if (kid[o] >= 0 && depth + 1 < levels && u >= 0 && u < units) {
                const int e = s.at[depth + 1][u];
                own[o] = e >= 0 && s.cell[e].x == kid[o] ? e : -1;
            }
        }
    }
    for (int d = levels - 1; d >= 0; --d) {
        if (s.present[d] == 0) {
            continue;   // the same for the whole workgroup
        }
        if (depth == d) {
#pragma unroll
            for (int o = 0; o < 8; ++o) {
                if (own[o] >= 0) {
                    q[o] = s.com[own[o]];
                }
            }
            s.com[threadIdx.x] = finish_cell<QUAD, In>(L, d, q, kid, c);
        }
        if (QUAD) {
            __syncthreads();   // second moments go through memory
        } else {
            lds_barrier();
        }
    }
}

// The FP32 pre-order records of every node, for the per-query walks, from a
// finished build: thread k < n writes the leaf at tree position k (its node
// index follows the cells started up to k), thread n + L the internal cell of
// level index L (node index rec[L].x). The values are the build's own FP64
// values rounded to FP32 (the leaves' are the tree-order s4).
__global__ __launch_bounds__(kThreads) void node_records_kernel(
    int n, int internal, const uint32_t* __restrict__ scan, const int32_t* __restrict__ delta,
    const float4* __restrict__ s4, InternalSoA in, const double* __restrict__ root,
    NodeF32* __restrict__ n32) {
    const int k = blockIdx.x * kThreads + threadIdx.x;
    if (k < n) {
        const int dp = k > 0 ? delta[k - 1] : -1;
        const int cells = delta[k] > dp ? delta[k] - dp : 0;
        const int li = static_cast<int>(scan[k]) + cells + k;
        n32[li] = leaf_record(s4[k], li, k);
    } else if (k - n < internal) {
        const int L = k - n;
        const int4 r = in.rec[L];
        n32[r.x] = cell_record(in.com[L], ldexp(root[3], -in.depth[L]), r.y, L);
    }
}

// What the host reads of an evaluation, into its pinned memory: flag words
// and depth counts, the root cube, the walk's counters.
struct BuildReport {
    unsigned flags[kFlagWords];
    double root[4];
    unsigned long long counters[kCounters + kPhases];
    unsigned number;   // of the evaluation, written last: the host waits for it
};
static_assert(2 * sizeof(BuildReport) <= kClocksAt, "the engine's pinned block holds a report");

__global__ __launch_bounds__(kThreads) void report_kernel(const unsigned* __restrict__ flags,
                                                          const double* __restrict__ root,
                                                          const unsigned long long* __restrict__ counters,
                                                          BuildReport* __restrict__ out,
                                                          unsigned number) {
    const int k = threadIdx.x;
    if (k < kFlagWords) {
        out->flags[k] = flags[k];
    }
    if (k < 4) {
        out->root[k] = root[k];
    }
    if (k < kCounters + kPhases - 1) {
        out->counters[k] = counters[k];
    } else if (k == kCounters + PHASE_END) {
        out->counters[k] = static_cast<unsigned long long>(wall_clock64());
    }
    __threadfence_system();
    __syncthreads();
    if (k == 0) {
        __hip_atomic_store(&out->number, number, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}


// ---------------------------------------------------------------- walk
// FP64 variant: the reference arithmetic (barnes_hut.c:574-613), bit-identical.
// One wave per Q consecutive tree positions, one query per lane; it walks the
// union of their lists in pre-order, so nodes come through scalar loads, and
// both nodes that can follow are loaded while a node is tested. The size test
// alone is the reference's (barnes_hut.c:588 also asks for a distance above
// zero: no size is below theta^2 times zero, and the one of a NaN neither).
//
// The bound is the wave's own chain: some 100 instructions a node, one after
// the other, over a union of two to four times one query's list. While there
// are waves to spare it pays to give each fewer queries, whose union is
// shorter: 8 and 16 while that keeps the waves below two per SIMD, 32 up to 2.6
// of them. Measured on MI355X, theta 0.7, us with 64 / 32 / 16 / 8 queries a
// wave, two-galaxy model, in brackets before (64 queries, IEEE square root
// and divide, no loads ahead):
//   3,000    201 / 166 / 148 / 127    (241)    10,000   296 / 252 / 216 / 199  (393)
//   30,000   387 / 326 / 326 / 332    (496)    100,000  556 / 537 / 681 / 1008 (643)
//   300,000  984 / 1222 / 1793 / 2961 (1190)
// Around the line, with 64 / 32, two galaxies of two seeds, Plummer, cloud:
//   70,000   729 / 495, 536 / 466, 690 / 678, 483 / 466
//   82,000   807 / 536, 565 / 525, 720 / 761, 509 / 456
//   88,000   544 / 544, 571 / 556, 716 / 765, 498 / 499
//   97,000   548 / 556, 611 / 556, 733 / 795, 502 / 502
//   115,000  594 / 632, -, 784 / 922, 553 / 581
// (64 a wave are little more than one wave a SIMD there: those SIMDs that get
// two long ones set the time.)
// (Terms noted in lists of 64 and formed four at a time, or held back to form
// two or four at once, were slower: the instructions that hold them cost more
// than the overlap gives.)
template <int Q>
__global__ __launch_bounds__(kWave) void walk_f64_kernel(
    const unsigned* __restrict__ flags, const NodeF64* __restrict__ n64,
    const double4* __restrict__ sp4,
    const uint32_t* __restrict__ tperm, int n, double G, double eps2, double theta2,
    double* __restrict__ ax, double* __restrict__ ay, double* __restrict__ az,
    unsigned long long* __restrict__ counters) {
    phase_begins(counters, PHASE_WALK);
    if (build_failed(flags)) {
        return;
    }
    const int nodes = n + static_cast<int>(flags[kDCount + kMaxLevels]);
    const int lane = threadIdx.x;
    const int t = blockIdx.x * Q + lane;
    const bool valid = lane < Q && t < n;
    int skip_until = valid ? 0 : 0x7FFFFFFF;
    unsigned approx = 0, exact = 0;
    const double4 qp = sp4[valid ? t : n - 1];
    const double qx = qp.x, qy = qp.y, qz = qp.z;
    double acx = 0.0, acy = 0.0, acz = 0.0;
    // (barnes_hut.c:593-603)
    auto add = [&](double dx, double dy, double dz, double d2, double m) {
        const double r2 = d2 + eps2;
        double y;
        const double p = r2 * exact_sqrt(r2, y);
        double inv3 = exact_recip(p, y * y * y);
        if (__builtin_amdgcn_ballot_w64(exact_odd(r2, p)) != 0) {
            asm volatile("");   // a branch, not a select
            inv3 = 1.0 / (r2 * sqrt(r2));
        }
        const double s = G * m * inv3;
        acx += s * dx;
        acy += s * dy;
        acz += s * dz;
    };
    int i = 0;
    NodeF64 nd = n64[0];
    while (i < nodes) {
        const double dx = nd.cx - qx;
        const double dy = nd.cy - qy;
        const double dz = nd.cz - qz;
        const double d2 = dx * dx + dy * dy + dz * dz;
        const bool active = i >= skip_until;
        if (nd.leaf >= 0) {
            const NodeF64 next = n64[i + 1];
            __builtin_amdgcn_sched_barrier(0);
            if (active && nd.leaf != t) {
                ++exact;
                add(dx, dy, dz, d2, nd.m);
            }
            ++i;
            nd = next;
        } else {
            const int skip = nd.skip;
            const NodeF64 first = n64[i + 1];
            const NodeF64 after = n64[skip];
            __builtin_amdgcn_sched_barrier(0);
            const bool accept = nd.size2 < theta2 * d2;
            if (active && accept) {
                ++approx;
                skip_until = skip;
                add(dx, dy, dz, d2, nd.m);
            }
            const bool open = __builtin_amdgcn_ballot_w64(active && !accept) != 0;
            i = open ? i + 1 : skip;
            nd = open ? first : after;
        }
    }
    if (valid) {
        const uint32_t o = tperm[t];
        ax[o] = acx;
        ay[o] = acy;
        az[o] = acz;
    }
    for (int off = 32; off > 0; off >>= 1) {
        approx += __shfl_xor(approx, off);
        exact += __shfl_xor(exact, off);
    }
    if (lane == 0) {
        atomicAdd(&counters[0], static_cast<unsigned long long>(approx));
        atomicAdd(&counters[1], static_cast<unsigned long long>(exact));
    }
}

// MI355X dispatches workgroup b to XCD (b mod 8), and each XCD has its own L2.
// Remap so that XCD x walks one contiguous eighth of the queries (Morton
// order): its L2 then holds that eighth's part of the tree. `grid` is a
// multiple of kXcds; surplus blocks get indices >= n and only walk the root.
constexpr int kXcds = 8;
#ifndef NBX_WALK_QUERIES
#define NBX_WALK_QUERIES 2
#endif
// Queries per lane of the FP32 walk.
constexpr int kWalkQueries = NBX_WALK_QUERIES;
__device__ inline int xcd_block(int b, int grid) {
    return (b % kXcds) * (grid / kXcds) + b / kXcds;
}

// Per-query accumulation of the FP32 walks: the softened interaction terms
// and, with FEATURES, the walk statistics of the learned correction
// (quadrupole force of the accepted cells, sum and minimum of (distance /
// cell edge)^2). G is applied once, when the result is stored.
template <bool FEATURES>
struct WalkAcc {
    float ax = 0.f, ay = 0.f, az = 0.f;
    unsigned approx = 0, exact = 0;
    float qax = 0.f, qay = 0.f, qaz = 0.f;
    float q2_sum = 0.f, q2_min = 3.0e38f;

    __device__ void leaf(float dx, float dy, float dz, float m, float eps2) {
        const float r2 = fmaf(dx, dx, fmaf(dy, dy, fmaf(dz, dz, eps2)));
        const float inv = __builtin_amdgcn_rsqf(r2);
        const float s = (m * inv) * (inv * inv);
        ax = fmaf(s, dx, ax);
        ay = fmaf(s, dy, ay);
        az = fmaf(s, dz, az);
        ++exact;
    }

    // Group-walk terms: the same arithmetic as leaf(), counted per flush by
    // the caller. A staged leaf can be the query itself (dx = dy = dz = 0
    // exactly, both positions being the same float4): with eps2 > 0 its term
    // is s * 0 = +0 and needs no test; with eps2 = 0 leaf_or_self_term gives
    // it no contribution (and no division by a zero distance), branch-free.
    __device__ void leaf_term(float dx, float dy, float dz, float m, float eps2) {
        const float r2 = fmaf(dx, dx, fmaf(dy, dy, fmaf(dz, dz, eps2)));
        const float inv = __builtin_amdgcn_rsqf(r2);
        const float s = (m * inv) * (inv * inv);
        ax = fmaf(s, dx, ax);
        ay = fmaf(s, dy, ay);
        az = fmaf(s, dz, az);
    }

    __device__ void leaf_or_self_term(float dx, float dy, float dz, float m, bool self,
                                      float eps2) {
        const float r2 = self ? 1.f : fmaf(dx, dx, fmaf(dy, dy, fmaf(dz, dz, eps2)));
        const float inv = __builtin_amdgcn_rsqf(r2);
        const float s = ((self ? 0.f : m) * inv) * (inv * inv);
        ax = fmaf(s, dx, ax);
        ay = fmaf(s, dy, ay);
        az = fmaf(s, dz, az);
    }

    // accepted cell, monopole term only
    __device__ void cell_softened(float dx, float dy, float dz, float m, float eps2) {
        const float r2 = fmaf(dx, dx, fmaf(dy, dy, fmaf(dz, dz, eps2)));
        const float inv = __builtin_amdgcn_rsqf(r2);
        const float s = (m * inv) * (inv * inv);
        ax = fmaf(s, dx, ax);
        ay = fmaf(s, dy, ay);
        az = fmaf(s, dz, az);
        ++approx;
    }

    // accepted cell at softened squared distance r2 (the force) and
    // unsoftened d2 (the features); with FEATURES its quadrupole record
    // q0 = (Qxx, Qyy, Qzz, Qxy), q1 = (Qxz, Qyz, size^2, 1 / size^2),
    // Q = sum m (3 x x^T - |x|^2 I) about the centre of mass
    __device__ void cell(float dx, float dy, float dz, float r2, float d2, float m, float4 q0,
                         float4 q1) {
        const float inv = __builtin_amdgcn_rsqf(r2);
        const float inv2 = inv * inv;
        const float s = (m * inv) * inv2;
        ax = fmaf(s, dx, ax);
        ay = fmaf(s, dy, ay);
        az = fmaf(s, dz, az);
        ++approx;
        if (FEATURES) {
            // quadrupole term with d = (cell - query):
            // G (5/2 (d.Q.d) d / r^7 - Q.d / r^5), softened r
            const float qdx = fmaf(q0.x, dx, fmaf(q0.w, dy, q1.x * dz));
            const float qdy = fmaf(q0.w, dx, fmaf(q0.y, dy, q1.y * dz));
            const float qdz = fmaf(q1.x, dx, fmaf(q1.y, dy, q0.z * dz));
            const float dqd = fmaf(dx, qdx, fmaf(dy, qdy, dz * qdz));
            const float inv5 = (inv2 * inv2) * inv;
            const float c = (2.5f * dqd) * inv2;
            qax = fmaf(fmaf(c, dx, -qdx), inv5, qax);
            qay = fmaf(fmaf(c, dy, -qdy), inv5, qay);
            qaz = fmaf(fmaf(c, dz, -qdz), inv5, qaz);
            const float q2 = d2 * q1.w;   // (distance / cell edge)^2
            q2_sum += q2;
            // (d / edge)^2 >= 0, where unsigned order is float order: one
            // v_min_u32 and no NaN canonicalisation
            q2_min = __uint_as_float(min(__float_as_uint(q2_min), __float_as_uint(q2)));
        }
    }

    // FEATURES: the kWalkRecord-float record of tree position t (G not
    // applied; its consumer scatters G * sum). Otherwise the accelerations of
    // particle tperm[t], in original order.
    __device__ void store(int t, const uint32_t* __restrict__ tperm, float G,
                          double* __restrict__ oax, double* __restrict__ oay,
                          double* __restrict__ oaz, float* __restrict__ features) const {
        if (!FEATURES) {
            const uint32_t o = tperm[t];
            oax[o] = static_cast<double>(G * ax);
            oay[o] = static_cast<double>(G * ay);
            oaz[o] = static_cast<double>(G * az);
        } else {
            // total sum xyz, accepted cells; quadrupole sum xyz, exact leaf
            // terms; sum and minimum of (d / edge)^2; zeros
            float4* f = reinterpret_cast<float4*>(features + static_cast<size_t>(t) * kWalkRecord);
            f[0] = make_float4(ax, ay, az, static_cast<float>(approx));
            f[1] = make_float4(qax, qay, qaz, static_cast<float>(exact));
            f[2] = make_float4(q2_sum, approx > 0 ? q2_min : 0.f, 0.f, 0.f);
            f[3] = make_float4(0.f, 0.f, 0.f, 0.f);
        }
    }
};

// One wave-step of the per-query walk at node `cur` (index i) for the query
// at tree position t, position (qx, qy, qz): returns true when this query
// descends into the node.
template <bool FEATURES>
__device__ inline bool walk_visit(const NodeF32& cur, int i, int t, float qx, float qy, float qz,
                                  float eps2, float theta2, int& skip_until,
                                  WalkAcc<FEATURES>& acc, float4 q0, float4 q1) {
    if (i < skip_until) {
        return false;
    }
    const float dx = cur.cx - qx;
    const float dy = cur.cy - qy;
    const float dz = cur.cz - qz;
    if (cur.leaf >= 0) {
        if (cur.leaf != t) {
            acc.leaf(dx, dy, dz, cur.m, eps2);
        }
        return false;
    }
    const float d2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
    if (d2 > 0.f && cur.size2 < theta2 * d2) {
        acc.cell(dx, dy, dz, d2 + eps2, d2, cur.m, q0, q1);
        skip_until = cur.skip;
        return false;
    }
    return true;
}

// FP32 walk with per-query reference interaction lists: one node per wave
// step, node fields in SGPRs (scalar loads of a wave-uniform index); lanes with
// nothing to do at a node are masked off. Each lane owns Q queries (tree
// positions base + 64k + lane, k < Q), so a wave walks the union of 64 Q
// consecutive queries' lists and every node record fetched (the walk's
// latency chain) feeds Q times the arithmetic; each query keeps its own
// skip_until and its reference visit order. (Measured alternatives, slower on
// MI355X: branch-free steps, vector-loaded nodes, prefetching both
// successors, four queries per lane.)
// The quadrupole record of pre-order node `cur` for the per-query walks: an
// internal node carries its level index as leaf = -(L + 2); a leaf has none.
__device__ inline void node_quad(const NodeF32& cur, const float4* __restrict__ gquad,
                                 float4& q0, float4& q1) {
    const int L = -cur.leaf - 2;
    if (L >= 0) {
        q0 = gquad[2 * L];
        q1 = gquad[2 * L + 1];
    } else {
        q0 = make_float4(0.f, 0.f, 0.f, 0.f);
        q1 = q0;
    }
}

// Queries: tree positions 0 .. nq - 1, or with `list` the tree positions
// list[0 .. nq - 1] (the queries a group walk deferred).
template <bool FEATURES, int Q>
__global__ __launch_bounds__(kThreads) void walk_f32_kernel(
    const NodeF32* __restrict__ n32, int nodes, const float4* __restrict__ s4,
    const uint32_t* __restrict__ tperm, const int* __restrict__ list, int nq, float G,
    float eps2, float theta2, double* __restrict__ ax, double* __restrict__ ay,
    double* __restrict__ az, unsigned long long* __restrict__ counters,
    float* __restrict__ features, const float4* __restrict__ gquad) {
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = xcd_block(blockIdx.x, gridDim.x) * (kThreads / kWave) + threadIdx.x / kWave;
    const int base = wave * (kWave * Q);
    int t[Q], skip_until[Q];
    bool valid[Q];
    float qx[Q], qy[Q], qz[Q];
    WalkAcc<FEATURES> acc[Q];
#pragma unroll
    for (int k = 0; k < Q; ++k) {
        const int qi = base + k * kWave + lane;
        valid[k] = qi < nq;
        t[k] = valid[k] ? (list != nullptr ? list[qi] : qi) : -1;
        const float4 q = s4[valid[k] ? t[k] : 0];
        qx[k] = q.x;
        qy[k] = q.y;
        qz[k] = q.z;
        skip_until[k] = valid[k] ? 0 : 0x7FFFFFFF;
    }
    int i = 0;
    while (i < nodes) {
        const int iu = __builtin_amdgcn_readfirstlane(i);
        const NodeF32 cur = n32[iu];
        // with FEATURES the node's quadrupole record
        float4 q0 = make_float4(0.f, 0.f, 0.f, 0.f), q1 = q0;
        if (FEATURES) {
            node_quad(cur, gquad, q0, q1);
        }
        bool descend = false;
#pragma unroll
        for (int k = 0; k < Q; ++k) {
            descend |= walk_visit<FEATURES>(cur, i, t[k], qx[k], qy[k], qz[k], eps2, theta2,
                                            skip_until[k], acc[k], q0, q1);
        }
        i = cur.leaf >= 0 || __builtin_amdgcn_ballot_w64(descend) != 0 ? i + 1 : cur.skip;
    }
    unsigned long long wa = 0, we = 0;
#pragma unroll
    for (int k = 0; k < Q; ++k) {
        if (valid[k]) {
            wa += acc[k].approx;
            we += acc[k].exact;
            acc[k].store(t[k], tperm, G, ax, ay, az, features);
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        wa += __shfl_xor(wa, off);
        we += __shfl_xor(we, off);
    }
    if (lane == 0) {
        atomicAdd(&counters[0], wa);
        atomicAdd(&counters[1], we);
    }
}

// Group walk (FP32). A wave, or in small systems a team of waves, takes 64
// consecutive tree positions as one group and walks the tree once for the group's bounding box: a
// cell is accepted when the reference's test (d^2 > 0 and 4h^2 < theta^2 d^2)
// holds for the box distance d, which implies it holds for every member, so
// each member's interaction set refines its reference set. The walk runs on
// the level-indexed cells: a per-wave stack of cells in LDS is popped up to 64
// at a time (one cell per lane, independent loads), accepted cells are
// staged, and an opened cell pushes its internal children and stages its
// leaf children. The dependent chain is one record load per step, about the
// tree depth in steps, instead of one per node visited in pre-order. Staged
// cells and leaves are evaluated by all 64 lanes without divergence (leaf
// positions are gathered into LDS just before). A group that is not compact
// (64 consecutive positions of the Morton curve can straddle one of its
// jumps) would get a box with most of the tree in its near field: it is split
// into compact parts. The members of a part the split cannot reach within its
// budget, or whose stack would overflow, are deferred to the per-query walk
// with reference lists, which runs after this kernel.
constexpr int kGroupList = 128;      // staged cells per wave
// 96 staged leaves: less LDS per wave, so more waves per CU (measured on
// MI355X against 128: 3% faster walk at 1M particles, 6% at 10M)
constexpr int kGroupLeaves = 96;     // staged leaves per wave
constexpr int kGroupStack = 512;     // pending cells per wave
constexpr int kRangeStack = 32;      // pending sub-ranges per wave
constexpr int kMaxSubWalks = 16;     // shared-list walks per wave
constexpr int kGroupCell = 2048;     // compact: the group's smallest enclosing cell holds <= kGroupCell

// Whether the run of tree positions that share the first c levels with a and
// b (a < b, which share exactly c; tree order is key order, so the run is an
// interval) holds at most kGroupCell positions. Each lane probes one position
// past each end at a stride of kGroupCell / 64 (the in-run probes are a prefix
// of the lanes), then half the lanes probe each end's last stride position by
// position: two rounds of independent loads instead of two galloping binary
// searches of up to ~40 dependent loads.
constexpr int kRunStride = kGroupCell / kWave;
static_assert(kRunStride == kWave / 2, "the fine round probes one stride per half wave");

__device__ inline bool run_compact(const uint64_t* __restrict__ w, const ExtTable& ext, int n,
                                   int a, int b, int c, int lane) {
    const int r = b + kRunStride * (lane + 1);
    const int l = a - kRunStride * (lane + 1);
    const bool in_r = r < n && common_levels(w, ext, b, r) >= c;
    const bool in_l = l >= 0 && common_levels(w, ext, l, a) >= c;
    const int kr = __popcll(__builtin_amdgcn_ballot_w64(in_r));
    const int kl = __popcll(__builtin_amdgcn_ballot_w64(in_l));
    if (kr == kWave || kl == kWave) {
        return false;   // the run reaches kGroupCell positions past one end
    }
    // lanes 0..30 probe the 31 positions after b + stride * kr, lanes 32..62
    // the 31 before a - stride * kl
    const int f = lane & (kRunStride - 1);
    const bool right = lane < kRunStride;
    const int p = right ? b + kRunStride * kr + f + 1 : a - kRunStride * kl - f - 1;
    bool in = false;
    if (f < kRunStride - 1) {
        in = right ? p < n && common_levels(w, ext, b, p) >= c
                   : p >= 0 && common_levels(w, ext, p, a) >= c;
    }
    const uint64_t fine = __builtin_amdgcn_ballot_w64(in);
    const int last = b + kRunStride * kr + __popcll(fine & 0xFFFFFFFFull);
    const int first = a - kRunStride * kl - __popcll(fine >> 32);
    return last - first + 1 <= kGroupCell;
}
// Groups are dealt to the XCDs in chunks of 2^chunk_log consecutive groups
// (chunk c to XCD c mod 8, each XCD's chunks in tree order): every XCD gets a
// share of the dense and the sparse regions, and a chunk's waves still share
// cell records in their XCD's L2. (Measured on MI355X, two-galaxy: with each
// XCD on one contiguous eighth of the groups, the XCDs finished between 630
// and 846 us at 1M and between 12.8 and 16.2 ms at 10M, theta = 0.5; walk
// 0.78 / 16.4 ms. Chunks of 8, 32, 128 groups: 0.80 / 14.4, 0.80 / 14.2,
// 0.78 / 14.2 ms. Teams of four, Plummer, chunks of 32 and 128: 86 and 111 us
// at 10,000, where 128 leave six XCDs without a group, 102 and 135 at 30,000.)
constexpr int kChunkLog = 7;        // a wave a group
constexpr int kTeamChunkLog = 5;    // a team of waves a group

__device__ inline int group_of_block(int b, int chunk_log) {
    const int slot = b / kXcds;   // workgroup b runs on XCD b mod 8
    return (((slot >> chunk_log) * kXcds + b % kXcds) << chunk_log) +
           (slot & ((1 << chunk_log) - 1));
}

// W waves walk one group, a workgroup. One wave, in a large system: its LDS is
// released as soon as it finishes (waves of one region take very different
// times; measured on MI355X, 1M particles: 1.45 ms with one group per
// workgroup, 1.66 ms with four). In a small system the chip is idle and the
// time is that of the longest group, a chain of steps (pop, record load, test,
// push) and of list entries: there two or four waves take one group. They pop
// from one common stack, 64 W cells a step with two barriers, stage and
// evaluate their own cells' lists, and add their sums at the end. A group in
// more than kTeamRanges ranges gives each range to one wave instead. The lists
// are the same for every W; only the order of the FP32 sums differs.
// (Measured on MI355X, walk with its events, theta = 0.7, two-galaxy / Plummer,
// W = 1, 2, 4: 10,000 particles 92, 74, 63 / 153, 110, 87 us; 100,000: 328, 186,
// 144 / 275, 241, 207; 262,144, W = 2, 4: 270, 288 / 321, 352; 500,000, W = 1, 2:
// 450, 435 / 535, 520; 1M: 778, 752 / 862, 916 us. Eight waves: 75 / 82 us at
// 10,000. Ranges up to which the team stays together, 1, 3, 7: 74, 69, 91 us for
// two galaxies of 10,000, 98, 95, 138 for 30,000.)
constexpr int kTeamRanges = 3;

// Waves per group for `groups` groups.
inline int walk_team(size_t groups, int cu_count) {
    const size_t cus = static_cast<size_t>(cu_count);
    return groups <= 8 * cus ? 4 : (groups <= 32 * cus ? 2 : 1);
}

// One query per lane in the group walk (measured on MI355X: two per lane, a
// group of 128, is 7% slower at 10M particles and 16% slower at 1M).

__device__ inline float wave_min(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        v = fminf(v, __shfl_xor(v, off));
    }
    return v;
}

__device__ inline float wave_max(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        v = fmaxf(v, __shfl_xor(v, off));
    }
    return v;
}

// Orders one wave's LDS writes before its later LDS reads.
__device__ inline void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <bool FEATURES, int W>
__global__ __launch_bounds__(W * kWave) void group_walk_kernel(
    const unsigned* __restrict__ flags, int* __restrict__ deferred,
    const GroupNode* __restrict__ gnode, const float4* __restrict__ s4,
    const uint32_t* __restrict__ tperm, const uint64_t* __restrict__ tword,
    ExtTable ext, int n, float G, float eps2, float theta2,
    double* __restrict__ ax, double* __restrict__ ay,
    double* __restrict__ az, unsigned long long* __restrict__ counters,
    float* __restrict__ features, const float4* __restrict__ gquad,
    int max_walks, bool member_test, int chunk_log) {
    phase_begins(counters, PHASE_WALK);
    constexpr int kWaves = W;
    // per wave: pending cells; staged cells (COM, mass; with FEATURES the
    // quadrupole record); staged leaves (tree position, then position and
    // mass); whether each lane's own leaf was staged; pending sub-ranges
    __shared__ int pending_all[kWaves * (kGroupStack + kGroupLeaves + 1)];
    __shared__ int pushed_all[kWaves];
    // FEATURES stages fewer cells per flush: their quadrupole records take LDS.
    // (Measured on MI355X, learned walk at 10M: 96 or 128 staged cells, 8.9 or
    // 10.4 KB of LDS, are 4% and 17% slower; six waves per SIMD through 80
    // VGPRs and 64 staged leaves is 5% slower. A list holds up to one step's
    // accepted cells, one per lane, so it cannot be shorter than a wave.)
    // A staged cell is kCellWords float4 in a row (COM and mass, then with
    // FEATURES the two quadrupole float4), so one LDS pointer walks the list.
    constexpr int kList = FEATURES ? kGroupList / 2 : kGroupList;
    static_assert(kList >= kWave, "a step stages up to one accepted cell per lane");
    constexpr int kTests = 4;   // candidates of the member test side by side
    static_assert(kGroupLeaves >= kWave + kTests, "the member test stages a step's candidates in lleaf");
    // The plain walk evaluates its staged lists four entries per loop trip
    // (LDS loads run ahead, one address update per four; same summation
    // order). Measured on MI355X against one per trip: walk 7% faster at 1M
    // particles and 5% at 10M, at 78 VGPRs; eight per trip takes 98 VGPRs.
    // The feature walk stays at one (two per trip: 99 VGPRs, fewer waves).
    constexpr int kEvalUnroll = FEATURES ? 1 : 4;
    constexpr int kCellWords = FEATURES ? 3 : 1;
    __shared__ float4 lcell_all[kWaves][kList * kCellWords];
    __shared__ float4 lleaf_all[kWaves][kGroupLeaves];
    __shared__ unsigned char selfhit_all[kWaves][kWave];
    __shared__ int2 ranges_all[kWaves][kRangeStack];
    const int lane = threadIdx.x & (kWave - 1);
    const int wid = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
    float4* lcell = lcell_all[wid];
    const int ltag_at = kWaves * kGroupStack + wid * (kGroupLeaves + 1);
    int* ltag = pending_all + ltag_at;
    float4* lleaf = lleaf_all[wid];
    unsigned char* selfhit = selfhit_all[wid];
    int2* ranges = ranges_all[wid];
    const int wave = group_of_block(static_cast<int>(blockIdx.x), chunk_log);
    const int t0 = wave * kWave;
    if (t0 >= n || build_failed(flags)) {
        return;   // whole wave beyond the particles, or no tree to walk
    }
    // the group: tree positions t0 + lane
    const int t = t0 + lane;
    const bool valid = t < n;
    const float4 q = s4[valid ? t : n - 1];
    const float qx = q.x, qy = q.y, qz = q.z;
    WalkAcc<FEATURES> acc;
    bool per_query = false;   // this lane's sub-group could not share a list

    // One shared-list walk for the members [a, b] (tree positions) of the
    // group: box acceptance against the members' bounding box. Returns false,
    // with the members' sums cleared, when the pending cells would overflow
    // the stack.
    auto shared_walk = [&](int a, int b, bool team) -> bool {
        const bool member = valid && t >= a && t <= b;
        const float bx0 = wave_min(member ? qx : 3.0e38f);
        const float by0 = wave_min(member ? qy : 3.0e38f);
        const float bz0 = wave_min(member ? qz : 3.0e38f);
        const float bx1 = wave_max(member ? qx : -3.0e38f);
        const float by1 = wave_max(member ? qy : -3.0e38f);
        const float bz1 = wave_max(member ? qz : -3.0e38f);
        int ccnt = 0, lcnt = 0;            // staged cells, leaves (wave-uniform)
        unsigned ncell = 0, nleaf = 0;     // evaluated per member (wave-uniform)
        // a team's pending cells are its waves' stacks put together
        const int stack_at = team ? 0 : wid * kGroupStack;
        const int room_for = team ? kWaves * kGroupStack : kGroupStack;
        const int lanes = team ? kWaves * kWave : kWave;
        int* stack = pending_all + stack_at;
        selfhit[lane] = 0;
        // evaluate the staged lists for every member
        auto flush = [&]() {
            wave_lds_fence();
            for (int e = lane; e < lcnt; e += kWave) {
                const int tag = ltag[e];
                lleaf[e] = s4[tag];
                const unsigned rel = static_cast<unsigned>(tag - t0);
                if (rel < static_cast<unsigned>(kWave)) {
                    selfhit[rel] = 1;
                }
            }
            wave_lds_fence();
            if (member) {
#pragma unroll kEvalUnroll
                for (int e = 0; e < ccnt; ++e) {
                    const float4 p = lcell[kCellWords * e];
                    const float dx = p.x - qx;
                    const float dy = p.y - qy;
                    const float dz = p.z - qz;
                    if (FEATURES) {
                        const float4 q0 = lcell[kCellWords * e + 1];
                        const float4 q1 = lcell[kCellWords * e + 2];
                        // softened distance from the unsoftened one (within an
                        // ulp of the plain walk's FMA chain)
                        const float d2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
                        acc.cell(dx, dy, dz, d2 + eps2, d2, p.w, q0, q1);
                    } else {
                        // softened distance straight from the FMA chain (the
                        // unsoftened one only feeds the features)
                        acc.cell_softened(dx, dy, dz, p.w, eps2);
                    }
                }
                if (eps2 > 0.f) {
#pragma unroll kEvalUnroll
                    for (int e = 0; e < lcnt; ++e) {
                        const float4 p = lleaf[e];
                        acc.leaf_term(p.x - qx, p.y - qy, p.z - qz, p.w, eps2);
                    }
                } else {
                    for (int e = 0; e < lcnt; ++e) {
                        const float4 p = lleaf[e];
                        acc.leaf_or_self_term(p.x - qx, p.y - qy, p.z - qz, p.w, ltag[e] == t,
                                              eps2);
                    }
                }
            }
            ncell += static_cast<unsigned>(ccnt);
            nleaf += static_cast<unsigned>(lcnt);
            ccnt = 0;
            lcnt = 0;
            wave_lds_fence();
        };
        int sp = 0;   // pending cells (wave-uniform); the root is level index 0
        if (n > 1) {
            if (lane == 0 && (!team || wid == 0)) {
                stack[0] = 0;
            }
            sp = 1;
        }
        bool overflow = false;
        if (team) {
            lds_barrier();
        } else {
            wave_lds_fence();
        }
        while (sp > 0) {
            // (sp goes through readfirstlane so the compiler keeps it, and
            // every test on it, in scalar registers; with the unmasked record
            // loads below, measured on MI355X: walk 0.817 -> 0.794 ms at 1M,
            // 17.07 -> 16.3 ms at 10M and theta = 0.5)
            sp = __builtin_amdgcn_readfirstlane(sp);
            // pop at most 64 cells, and few enough that their children (8
            // each) fit: a wide level then spreads over more steps instead
            // of overflowing
            const int room = (room_for - sp) / 8;
            const int cap = room > 1 ? (room < lanes ? room : lanes) : 1;
            const int take = sp < cap ? sp : cap;
            const int pop = team ? lane * kWaves + wid : lane;
            const bool act = pop < take;
            const int ref = act ? stack[sp - take + pop] : 0;
            sp = __builtin_amdgcn_readfirstlane(sp - take);
            wave_lds_fence();   // pops read before pushes reuse their slots
            // Every lane loads a record (the lanes past `take` the root's) and
            // tests it; `act` masks the outcomes, so idle lanes need no defaults.
            const float4* g = reinterpret_cast<const float4*>(gnode + ref);
            const float4 c0 = g[0];
            const float4 c1 = g[1];
            const int4 k0 = reinterpret_cast<const int4*>(g)[2];
            const int4 k1 = reinterpret_cast<const int4*>(g)[3];
            float4 gq0 = make_float4(0.f, 0.f, 0.f, 0.f), gq1 = gq0;
            if (FEATURES) {
                // the quadrupole record comes with the cell (loads in flight together)
                gq0 = gquad[2 * ref];
                gq1 = gquad[2 * ref + 1];
            }
            const float ddx = fmaxf(0.f, fmaxf(bx0 - c0.x, c0.x - bx1));
            const float ddy = fmaxf(0.f, fmaxf(by0 - c0.y, c0.y - by1));
            const float ddz = fmaxf(0.f, fmaxf(bz0 - c0.z, c0.z - bz1));
            const float d2 = fmaf(ddx, ddx, fmaf(ddy, ddy, ddz * ddz));
            bool accepted = act & (d2 > 0.f) & (c1.x < theta2 * d2);
            if (member_test) {
                // A cell the box test opens is still accepted when every
                // member's own reference test (walk_visit's arithmetic)
                // accepts it: the lists keep refining the members' reference
                // lists. Only cells that pass at the box's far corner from
                // their centre of mass can pass for some member; each such
                // candidate is broadcast and tested by all members at once.
                const float fx = fmaxf(fabsf(c0.x - bx0), fabsf(c0.x - bx1));
                const float fy = fmaxf(fabsf(c0.y - by0), fabsf(c0.y - by1));
                const float fz = fmaxf(fabsf(c0.z - bz0), fabsf(c0.z - bz1));
                const bool cand = act & !accepted &
                                  (c1.x < theta2 * fmaf(fx, fx, fmaf(fy, fy, fz * fz)));
                // The candidates go to LDS in lane order (the staged-leaf
                // buffer: it only holds data inside a flush) and every member
                // reads each one by broadcast; the tests take no branches.
                const uint64_t pending = __builtin_amdgcn_ballot_w64(cand);
                if (pending != 0) {
                    const uint64_t members = __builtin_amdgcn_ballot_w64(member);
                    const int slot = static_cast<int>(lanes_below(pending));
                    if (cand) {
                        lleaf[slot] = make_float4(c0.x, c0.y, c0.z, c1.x);
                    }
                    wave_lds_fence();
                    const int nc = static_cast<int>(__popcll(pending));
                    uint64_t pass = 0;   // bit j: every member accepts candidate j
                    for (int j = 0; j < nc; j += kTests) {
                        float4 cj[kTests];
#pragma unroll
                        for (int u = 0; u < kTests; ++u) {
                            cj[u] = lleaf[j + u];   // (past the last: not looked up)
                        }
                        uint64_t open_for[kTests];
#pragma unroll
                        for (int u = 0; u < kTests; ++u) {
                            const float dx = cj[u].x - qx;
                            const float dy = cj[u].y - qy;
                            const float dz = cj[u].z - qz;
                            const float dj2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
                            // (each comparison balloted on its own: its lane
                            // mask is the ballot, with no VALU round trip)
                            const uint64_t ok = __builtin_amdgcn_ballot_w64(dj2 > 0.f) &
                                                __builtin_amdgcn_ballot_w64(cj[u].w < theta2 * dj2);
                            open_for[u] = members & ~ok;
                        }
#pragma unroll
                        for (int u = 0; u < kTests; ++u) {
                            pass |= open_for[u] == 0 ? 1ull << (j + u) : 0ull;
                        }
                    }
                    wave_lds_fence();   // candidates read before the buffer is reused
                    accepted = accepted | (cand & (((pass >> slot) & 1ull) != 0));
                }
            }
            if (ccnt > kList - kWave) {
                flush();
            }
            const uint64_t cbal = __ballot(accepted);
            if (accepted) {
                const int pos = ccnt + static_cast<int>(lanes_below(cbal));
                lcell[kCellWords * pos] = c0;
                if (FEATURES) {
                    lcell[kCellWords * pos + 1] = gq0;
                    lcell[kCellWords * pos + 2] = gq1;
                }
            }
            ccnt += static_cast<int>(__popcll(cbal));
            // opened cells: children in octant order. The feature walk goes an
            // octant a round (at most 64 new leaves and 64 new cells) and
            // flushes where the leaves of one do not fit, which keeps the order
            // of its sums (a model's features) as it was. The plain walk places
            // all eight octants' children at once, without branches, after one
            // flush where they do not fit; a step with more leaves than the list
            // holds takes the rounds.
            const bool open = act && !accepted;
            const int kid[8] = {k0.x, k0.y, k0.z, k0.w, k1.x, k1.y, k1.z, k1.w};
            if (FEATURES) {
#pragma unroll
                for (int o = 0; o < 8; ++o) {
                    const int ch = open ? kid[o] : -1;
                    const uint64_t lb = __ballot(ch < -1);
                    const uint64_t ib = __ballot(ch >= 0);
                    if (lb != 0) {
                        if (lcnt > kGroupLeaves - kWave) {
                            flush();
                        }
                        if (ch < -1) {
                            ltag[lcnt + static_cast<int>(lanes_below(lb))] = -ch - 2;
                        }
                        lcnt += static_cast<int>(__popcll(lb));
                    }
                    const int np = static_cast<int>(__popcll(ib));
                    if (sp + np > room_for) {
                        overflow = true;
                    } else if (np != 0) {
                        if (ch >= 0) {
                            stack[sp + static_cast<int>(lanes_below(ib))] = ch;
                        }
                        sp = __builtin_amdgcn_readfirstlane(sp + np);
                    }
                }
            } else {
                uint64_t lb[8], ib[8];
                int leaves = 0, cells = 0;
#pragma unroll
                for (int o = 0; o < 8; ++o) {
                    const int ch = open ? kid[o] : -1;
                    lb[o] = __builtin_amdgcn_ballot_w64(ch < -1);
                    ib[o] = __builtin_amdgcn_ballot_w64(ch >= 0);
                    leaves += static_cast<int>(__popcll(lb[o]));
                    cells += static_cast<int>(__popcll(ib[o]));
                }
                int at = sp, all = cells;
                if (team) {
                    // room on the common stack, in the waves' order; no wave
                    // pushes before all have popped
                    if (lane == 0) {
                        pushed_all[wid] = cells;
                    }
                    lds_barrier();
                    all = 0;
#pragma unroll
                    for (int w = 0; w < kWaves; ++w) {
                        const int theirs = __builtin_amdgcn_readfirstlane(pushed_all[w]);
                        at += w < wid ? theirs : 0;
                        all += theirs;
                    }
                }
                overflow = sp + all > room_for;
                if (lcnt + leaves > kGroupLeaves) {
                    flush();
                }
                if (leaves <= kGroupLeaves && !overflow) {
                    sp += all;
                    at += stack_at;
#pragma unroll
                    for (int o = 0; o < 8; ++o) {
                        const int ch = open ? kid[o] : -1;
                        const int cell = at + static_cast<int>(lanes_below(ib[o]));
                        const int leaf = ltag_at + lcnt + static_cast<int>(lanes_below(lb[o]));
                        const int slot = ch >= 0 ? cell : (ch < -1 ? leaf : ltag_at + kGroupLeaves);
                        pending_all[slot] = ch >= 0 ? ch : -ch - 2;
                        at += static_cast<int>(__popcll(ib[o]));
                        lcnt += static_cast<int>(__popcll(lb[o]));
                    }
                } else if (!overflow) {
                    // more leaves than the list holds: an octant at a time
                    sp += all;
                    at += stack_at;
#pragma unroll
                    for (int o = 0; o < 8; ++o) {
                        const int ch = open ? kid[o] : -1;
                        const uint64_t leaf = __builtin_amdgcn_ballot_w64(ch < -1);
                        const uint64_t cell = __builtin_amdgcn_ballot_w64(ch >= 0);
                        if (lcnt > kGroupLeaves - kWave) {
                            flush();
                        }
                        if (ch < -1) {
                            ltag[lcnt + static_cast<int>(lanes_below(leaf))] = -ch - 2;
                        }
                        if (ch >= 0) {
                            pending_all[at + static_cast<int>(lanes_below(cell))] = ch;
                        }
                        at += static_cast<int>(__popcll(cell));
                        lcnt += static_cast<int>(__popcll(leaf));
                    }
                }
            }
            if (overflow) {
                break;
            }
            // pushes visible before the next pops
            if (team) {
                lds_barrier();
            } else {
                wave_lds_fence();
            }
        }
        if (!overflow && ccnt + lcnt > 0) {
            flush();
        }
        wave_lds_fence();
        if (member) {
            if (overflow) {
                acc = WalkAcc<FEATURES>();
            } else {
                // each member evaluated every staged entry but its own leaf
                acc.approx = ncell;
                acc.exact = nleaf - selfhit[lane];
            }
        }
        wave_lds_fence();   // selfhit read before the next walk clears it
        return !overflow;
    };

    // Sub-ranges of the group, split at the Morton curve's jumps until each
    // is compact: its smallest enclosing cell holds <= kGroupCell particles
    // (a range straddling a jump, an outlier, a dense core and its outskirts
    // would otherwise get a box with most of the tree in its near field). A
    // range that is not compact is split at the octant changes of its common
    // cell's children (tree order is key order, so each octant is a run); the
    // members of a range that cannot be split within the budget of
    // `max_walks` shared walks per wave are deferred to the per-query walk.
    const int last = t0 + kWave - 1 < n ? t0 + kWave - 1 : n - 1;
    const int max_level = ext.words != nullptr ? kMaxLevels : 21;
    int rsp = 1, walks = 0;
    if (lane == 0) {
        ranges[0] = make_int2(t0, last);
    }
    wave_lds_fence();
    while (rsp > 0) {
        --rsp;
        const int2 r = ranges[rsp];
        const int a = __builtin_amdgcn_readfirstlane(r.x);
        const int b = __builtin_amdgcn_readfirstlane(r.y);
        wave_lds_fence();   // the pop is read before a push reuses the slot
        const int c =
            __builtin_amdgcn_readfirstlane(a < b ? common_levels(tword, ext, a, b) : max_level);
        const bool shared = c >= max_level || run_compact(tword, ext, n, a, b, c, lane);
        uint64_t cut = 0;
        if (!shared && rsp + 8 <= kRangeStack && walks + rsp + 2 <= max_walks) {
            // octant of each member's depth c + 1 cell; runs of equal octants
            // (a and b differ in that octant, so there are at least two)
            // (lanes outside the range need not have extension words)
            const int dig = digit_at(tword, ext, t >= a && t <= b ? t : a, c);
            const int prev = __shfl_up(dig, 1);
            cut = __ballot(t > a && t <= b && dig != prev);
        }
        if (cut != 0) {
            int s = a;
            while (cut != 0) {
                const int j = __builtin_ctzll(cut);
                cut &= cut - 1;
                if (lane == 0) {
                    ranges[rsp] = make_int2(s, t0 + j - 1);
                }
                ++rsp;
                s = t0 + j;
            }
            if (lane == 0) {
                ranges[rsp] = make_int2(s, b);
            }
            ++rsp;
            wave_lds_fence();
            continue;
        }
        if (shared) {
            if (lane == 0) {
                ranges[kRangeStack - 1 - walks] = make_int2(a, b);
            }
            ++walks;
        } else {
            per_query = per_query || (valid && t >= a && t <= b);
        }
    }
    wave_lds_fence();
    // few ranges: all waves on each in turn; more: a wave a range
    const bool team = W > 1 && walks <= kTeamRanges;
    for (int k = team ? 0 : wid; k < walks; k += team ? 1 : W) {
        const int2 r = ranges[kRangeStack - 1 - k];
        const int a = __builtin_amdgcn_readfirstlane(r.x);
        const int b = __builtin_amdgcn_readfirstlane(r.y);
        if (!shared_walk(a, b, team)) {
            per_query = per_query || (valid && t >= a && t <= b);
        }
    }
    if constexpr (W > 1) {
        // The group's sums: the waves' in their order
        lcell[lane] = make_float4(acc.ax, acc.ay, acc.az, per_query ? 1.f : 0.f);
        lcell[kWave + lane] = make_float4(__uint_as_float(acc.approx), __uint_as_float(acc.exact),
                                          0.f, 0.f);
        __syncthreads();
        if (wid != 0) {
            return;
        }
#pragma unroll
        for (int w = 1; w < W; ++w) {
            const float4 sum = lcell_all[w][lane];
            const float4 count = lcell_all[w][kWave + lane];
            acc.ax += sum.x;
            acc.ay += sum.y;
            acc.az += sum.z;
            per_query = per_query || sum.w != 0.f;
            acc.approx += __float_as_uint(count.x);
            acc.exact += __float_as_uint(count.y);
        }
    }
    // The lanes whose range could not share a list go to the deferred list
    // (counters[2] entries): the per-query reference-list walk takes them after
    // this kernel, and writes their results. Their sums here are empty (never
    // walked, or cleared on overflow).
    const uint64_t deferring = __builtin_amdgcn_ballot_w64(per_query);
    if (deferring != 0) {
        unsigned long long slot = 0;
        if (lane == 0) {
            slot = atomicAdd(&counters[2], static_cast<unsigned long long>(__popcll(deferring)));
        }
        slot = __shfl(slot, 0);
        const unsigned long long k = slot + lanes_below(deferring);
        if (per_query && k < static_cast<unsigned long long>(n)) {
            deferred[k] = t;
        }
    }
    unsigned long long wa = 0, we = 0;
    if (valid && !per_query) {
        wa = acc.approx;
        we = acc.exact;
        acc.store(t, tperm, G, ax, ay, az, features);
    }
    for (int off = 32; off > 0; off >>= 1) {
        wa += __shfl_xor(wa, off);
        we += __shfl_xor(we, off);
    }
    if (lane == 0) {
        atomicAdd(&counters[0], wa);
        atomicAdd(&counters[1], we);
    }
}

template <typename T>
T* B(Buf& b) {
    return b.as<T>();
}

}  // namespace


namespace {

InternalSoA internal_soa(BHState& s) {
    InternalSoA in;
    in.com = B<double4>(s.icom);
    in.rec = B<int4>(s.irec);
    in.depth = B<int32_t>(s.idepth);
    return in;
}

ExtTable ext_table(const BHState& s) {
    return {s.ext_tree, s.ext_slot};
}

double* root_of(BHState& s) {
    return B<double>(s.partial) + 6 * kBBoxBlocks;
}

template <typename In>
const In* tree_inputs(BHState& s) {
    if constexpr (std::is_same_v<In, float4>) {
        return B<float4>(s.s4);
    } else {
        return B<double4>(s.sp4);
    }
}

// Tree positions from the particles in sk0/sv0, sorted by key >> low_bits.
template <typename In>
void enqueue_runs(Engine* e, int low_bits) {
    BHState& s = e->bh;
    order_kernel<In><<<grid_for(s.n, kThreads), kThreads, 0, e->stream>>>(
        B<uint64_t>(s.sk0), B<uint32_t>(s.sv0), static_cast<int>(s.n), B<In>(s.b4), root_of(s),
        B<uint32_t>(s.tperm), B<uint64_t>(s.tword), B<uint64_t>(s.ext), B<uint32_t>(s.tmp32),
        static_cast<unsigned>(s.ext_slots),
        std::is_same_v<In, double4> ? B<double4>(s.sp4) : nullptr, B<float4>(s.s4),
        B<unsigned>(s.flags), low_bits);
    s.sorted_low_bits = low_bits;
    s.ext_tree = B<uint64_t>(s.ext);
    s.ext_slot = B<uint32_t>(s.tmp32);
}

// The bounding cube, the keys and the tree order of e's particles.
template <typename In>
NBodySimProStatus enqueue_order(Engine* e, NBodySimProError* error) {
    BHState& s = e->bh;
    hipStream_t st = e->stream;
    const int ni = static_cast<int>(s.n);
    const unsigned g = grid_for(s.n, kThreads);
    unsigned* flags = B<unsigned>(s.flags);
    In* b4 = B<In>(s.b4);
    double* root = root_of(s);
    unsigned long long* cnts = B<unsigned long long>(s.counters);
    double4* sp4 = std::is_same_v<In, double4> ? B<double4>(s.sp4) : nullptr;
    const unsigned bb_blocks = g < static_cast<unsigned>(kBBoxBlocks) ? g : kBBoxBlocks;
    bbox_partial_kernel<In><<<bb_blocks, kThreads, 0, st>>>(
        e->px, e->py, e->pz, e->m, b4, ni, B<double>(s.partial), flags, kFlagWords,
        cnts);
    if (s.n <= static_cast<size_t>(kSmallSort)) {
        tile_sort_kernel<In><<<grid_for(s.n, kSortTile1), kThreads, 0, st>>>(
            b4, ni, B<double>(s.partial), static_cast<int>(bb_blocks), root, B<uint64_t>(s.sk0),
            B<uint32_t>(s.sv0), cnts);
        merge_order_kernel<In><<<grid_for(s.n * kMergeLanes, kThreads), kThreads, 0, st>>>(
            B<uint64_t>(s.sk0), B<uint32_t>(s.sv0), ni, b4, B<uint32_t>(s.tperm),
            B<uint64_t>(s.tword), sp4, B<float4>(s.s4));
        s.ext_tree = nullptr;   // a shared key raises FLAG_TIE
        s.ext_slot = nullptr;
        s.sorted_low_bits = 0;
    } else {
        keys_kernel<In><<<g < 1024u ? g : 1024u, kThreads, 0, st>>>(
            b4, ni, B<double>(s.partial), static_cast<int>(bb_blocks), root, B<uint64_t>(s.sk0));
        NBX_HIP(error, hipGetLastError());
        NBX_TRY(s.ext.need<uint64_t>(s.ext_slots * kExtWords, error));
        NBX_TRY(s.tmp32.need<uint32_t>(s.n, error));
        // stable on the top key bits (the result stays in sk0/sv0), then the
        // short runs. (Measured on MI355X, two-galaxy, against seven passes
        // on all 63 bits: sort 1M 0.171 -> 0.108 ms, 10M 0.894 -> 0.641 ms.)
        NBX_TRY(radix_sort_pairs(st, B<uint64_t>(s.sk0), B<uint32_t>(s.sv0), B<uint64_t>(s.sk1),
                                 B<uint32_t>(s.sv1), s.n, kSortTopBits, s.hist, error, kSortLowBits,
                                 true, cnts + kCounters + PHASE_SORT));
        enqueue_runs<In>(e, kSortLowBits);
    }
    NBX_HIP(error, hipGetLastError());
    return N_BODY_SIM_PRO_STATUS_OK;
}

// The same order after FLAG_LONG_RUN, from a sort on all the key bits: sk0 and sv0
// still hold the pairs, stably sorted on the top ones from index order.
template <typename In>
NBodySimProStatus enqueue_key_order(Engine* e, NBodySimProError* error) {
    BHState& s = e->bh;
    NBX_TRY(radix_sort_pairs(e->stream, B<uint64_t>(s.sk0), B<uint32_t>(s.sv0),
                             B<uint64_t>(s.sk1), B<uint32_t>(s.sv1), s.n, 63, s.hist, error));
    enqueue_runs<In>(e, 0);
    NBX_HIP(error, hipGetLastError());
    return N_BODY_SIM_PRO_STATUS_OK;
}

// The same order from all the words: (key, ext0, ..., ext5), least significant
// word first, stable from index order.
template <typename In>
NBodySimProStatus enqueue_full_order(Engine* e, NBodySimProError* error) {
    BHState& s = e->bh;
    hipStream_t st = e->stream;
    const size_t n = s.n;
    const int ni = static_cast<int>(n);
    const unsigned g = grid_for(n, kThreads);
    const In* b4 = B<In>(s.b4);
    double* root = root_of(s);
    const unsigned bb_blocks = g < static_cast<unsigned>(kBBoxBlocks) ? g : kBBoxBlocks;
    NBX_TRY(s.mkey.need<uint64_t>(n, error));
    NBX_TRY(s.tmp32.need<uint32_t>(n, error));
    NBX_TRY(s.ext.need<uint64_t>(n * kExtWords, error));
    NBX_TRY(s.ext_orig.need<uint64_t>(n * kExtWords, error));
    uint64_t* key = B<uint64_t>(s.mkey);
    uint64_t* ext = B<uint64_t>(s.ext_orig);
    uint32_t* P = B<uint32_t>(s.tmp32);
    keys_kernel<In><<<g < 1024u ? g : 1024u, kThreads, 0, st>>>(
        b4, ni, B<double>(s.partial), static_cast<int>(bb_blocks), root, key);
    ext_words_kernel<In><<<g, kThreads, 0, st>>>(b4, ni, root, ext);
    iota_kernel<<<g, kThreads, 0, st>>>(P, ni);
    for (int k = kExtWords; k >= 0; --k) {
        if (k > 0) {
            gather_u64_kernel<<<g, kThreads, 0, st>>>(ext, P, B<uint64_t>(s.sk0), ni, kExtWords,
                                                      k - 1);
        } else {
            gather_u64_kernel<<<g, kThreads, 0, st>>>(key, P, B<uint64_t>(s.sk0), ni, 1, 0);
        }
        NBX_HIP(error, hipMemcpyAsync(s.sv0.p, P, n * sizeof(uint32_t), hipMemcpyDeviceToDevice, st));
        NBX_TRY(radix_sort_pairs(st, B<uint64_t>(s.sk0), B<uint32_t>(s.sv0), B<uint64_t>(s.sk1),
                                 B<uint32_t>(s.sv1), n, 63, s.hist, error));
        NBX_HIP(error, hipMemcpyAsync(P, s.sv0.p, n * sizeof(uint32_t), hipMemcpyDeviceToDevice, st));
    }
    place_kernel<In><<<g, kThreads, 0, st>>>(
        P, key, ext, ni, b4, B<uint32_t>(s.tperm), B<uint64_t>(s.tword), B<uint64_t>(s.ext),
        std::is_same_v<In, double4> ? B<double4>(s.sp4) : nullptr, B<float4>(s.s4));
    NBX_HIP(error, hipGetLastError());
    s.ext_tree = B<uint64_t>(s.ext);   // by position
    s.ext_slot = nullptr;
    return N_BODY_SIM_PRO_STATUS_OK;
}

// Neighbour depths, per-depth counts and their scan over the tiles.
NBodySimProStatus enqueue_depths(Engine* e, NBodySimProError* error) {
    BHState& s = e->bh;
    hipStream_t st = e->stream;
    const int ni = static_cast<int>(s.n);
    const int nt = static_cast<int>(grid_for(s.n, s.tile));
    unsigned* flags = B<unsigned>(s.flags);
    with_tile(s.tile, [&](auto tile) {
        delta_kernel<decltype(tile)::kPositions><<<nt, kThreads, 0, st>>>(
            B<uint64_t>(s.tword), ext_table(s), ni, nt, B<int32_t>(s.delta), flags,
            B<unsigned>(s.tile_hist), B<unsigned long long>(s.counters));
    });
    depth_scan_kernel<<<kTopoRows, kThreads, 0, st>>>(B<unsigned>(s.tile_hist), nt,
                                                      B<unsigned>(s.tile_base), flags);
    NBX_HIP(error, hipGetLastError());
    return N_BODY_SIM_PRO_STATUS_OK;
}

// Cell records and centre of mass, in buffers for s.cells cells.
template <bool QUAD, typename In>
NBodySimProStatus enqueue_cells(Engine* e, NBodySimProError* error) {
    BHState& s = e->bh;
    hipStream_t st = e->stream;
    const int ni = static_cast<int>(s.n);
    const int nt = static_cast<int>(grid_for(s.n, s.tile));
    NBX_TRY(s.icom.need<double4>(s.cells, error));
    NBX_TRY(s.irec.need<int4>(s.cells, error));
    NBX_TRY(s.idepth.need<int32_t>(s.cells, error));
    NBX_TRY(s.gnode.need<GroupNode>(s.cells, error));
    if (QUAD) {
        // quadrupole records only for the learned correction's feature walk
        NBX_TRY(s.im2.need<double>(6 * s.cells, error));
        NBX_TRY(s.gquad.need<float4>(2 * s.cells, error));
    }
    constexpr bool fp64 = std::is_same_v<In, double4>;
    if (fp64) {
        // FP64 node records feed only the exact FP64 walk, which loads one ahead
        NBX_TRY(s.n64.need<NodeF64>(s.n + s.cells + 1, error));
    }
    CellData<In> c;
    c.gnode = B<GroupNode>(s.gnode);
    c.in = internal_soa(s);
    c.sp4 = tree_inputs<In>(s);
    c.b4 = B<In>(s.b4);
    c.tperm = B<uint32_t>(s.tperm);
    c.root = root_of(s);
    c.n64 = fp64 ? B<NodeF64>(s.n64) : nullptr;
    c.im2 = QUAD ? B<double>(s.im2) : nullptr;
    c.gquad = QUAD ? B<float4>(s.gquad) : nullptr;
    unsigned* flags = B<unsigned>(s.flags);
    const unsigned* base = B<unsigned>(s.tile_base);
    unsigned long long* cnts = B<unsigned long long>(s.counters);
    with_tile(s.tile, [&](auto tile) {
        using T = decltype(tile);
        constexpr int kPositions = T::kPositions;
        build_kernel<QUAD, In, T><<<nt, T::kBuildThreads, 0, st>>>(
            B<uint64_t>(s.tword), ext_table(s), B<int32_t>(s.delta), ni, nt,
            static_cast<int>(s.cells), flags, base, B<uint32_t>(s.scan), c);
        if (nt > 1) {
            span_com_kernel<QUAD, In, 512, kPositions><<<grid_for(nt, kSpanTiles), 512, 0, st>>>(
                1, kSpanTiles, nt, flags, base, c, cnts);
        }
        if (nt > kSpanTiles) {
            const int units = (nt + kSpanTiles - 1) / kSpanTiles;
            span_com_kernel<QUAD, In, 1024, kPositions><<<1, 1024, 0, st>>>(
                kSpanTiles, units, nt, flags, base, c, cnts);
        }
    });
    NBX_HIP(error, hipGetLastError());
    return N_BODY_SIM_PRO_STATUS_OK;
}

NBodySimProStatus enqueue_cells(Engine* e, NBodySimProError* error) {
    if (e->bh.inputs_fp64) {
        return enqueue_cells<false, double4>(e, error);
    }
    return e->bh.has_quad ? enqueue_cells<true, float4>(e, error)
                          : enqueue_cells<false, float4>(e, error);
}

BuildReport* report_of(BHState& s, int slot) {
    return static_cast<BuildReport*>(s.report) + slot;
}

// Enqueues the report of the evaluation before it in the stream into a slot.
NBodySimProStatus enqueue_report(Engine* e, int slot, NBodySimProError* error) {
    BHState& s = e->bh;
    s.number[slot] = ++s.evaluations;
    report_kernel<<<1, kThreads, 0, e->stream>>>(B<unsigned>(s.flags), root_of(s),
                                                 B<unsigned long long>(s.counters),
                                                 report_of(s, slot), s.number[slot]);
    NBX_HIP(error, hipGetLastError());
    return N_BODY_SIM_PRO_STATUS_OK;
}

// Waits until a slot holds its report. (Polled: the wait then costs no packet
// in the stream, and whatever is enqueued behind the report runs on.)
NBodySimProStatus await_report(Engine* e, int slot, NBodySimProError* error) {
    BHState& s = e->bh;
    const unsigned* number = &report_of(s, slot)->number;
    for (;;) {
        for (int spin = 0; spin < 20000; ++spin) {
            if (__atomic_load_n(number, __ATOMIC_ACQUIRE) == s.number[slot]) {
                return N_BODY_SIM_PRO_STATUS_OK;
            }
            __builtin_ia32_pause();
        }
        // the stream is done or has failed: the report is there, or never will be
        const hipError_t state = hipStreamQuery(e->stream);
        if (state == hipErrorNotReady) {
            (void)hipGetLastError();
            continue;
        }
        NBX_HIP(error, state);
        if (__atomic_load_n(number, __ATOMIC_ACQUIRE) != s.number[slot]) {
            NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_STATE,
                     "a Barnes-Hut evaluation ended without its report");
        }
    }
}

// Whether a report's evaluation needs nothing more from the host.
bool report_clean(const BuildReport* r) {
    return (r->flags[0] | r->flags[1] | r->flags[2] | r->flags[3]) == 0 && r->counters[2] == 0;
}

// Waits for the evaluation in `slot` and reads what its kernels left in the
// flag words. `again` says that the tree was not valid (the walk did nothing)
// and that the part in question has been enqueued anew.
NBodySimProStatus read_build(Engine* e, int slot, bool* again, NBodySimProError* error) {
    BHState& s = e->bh;
    hipStream_t st = e->stream;
    unsigned* flags = B<unsigned>(s.flags);
    NBX_TRY(await_report(e, slot, error));
    const BuildReport* report = report_of(s, slot);
    *again = false;
    if (report->flags[FLAG_LONG_RUN] != 0 || report->flags[FLAG_TIE] != 0) {
        NBX_HIP(error, hipMemsetAsync(flags, 0, kFlagWords * sizeof(unsigned), st));
        if (report->flags[FLAG_LONG_RUN] == ORDER_SLOTS) {
            const size_t tied = report->flags[kTiedCount];
            s.ext_slots = tied + tied / 8;
            NBX_TRY(s.ext.need<uint64_t>(s.ext_slots * kExtWords, error));
            if (s.inputs_fp64) {
                enqueue_runs<double4>(e, s.sorted_low_bits);
            } else {
                enqueue_runs<float4>(e, s.sorted_low_bits);
            }
        } else if (s.sorted_low_bits > 0) {
            NBX_TRY(s.inputs_fp64 ? enqueue_key_order<double4>(e, error)
                                  : enqueue_key_order<float4>(e, error));
        } else {
            NBX_TRY(s.inputs_fp64 ? enqueue_full_order<double4>(e, error)
                                  : enqueue_full_order<float4>(e, error));
        }
        NBX_TRY(enqueue_depths(e, error));
        *again = true;
        return enqueue_cells(e, error);
    }
    if (report->flags[FLAG_OVERFLOW] != 0) {
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_OVERFLOW,
                 "Barnes-Hut tree exceeded maximum depth (duplicate positions?)");
    }
    const unsigned* dcount = report->flags + kDCount;
    if (report->flags[FLAG_CELLS] != 0) {
        s.cells = dcount[kMaxLevels] + static_cast<size_t>(dcount[kMaxLevels]) / 8;
        NBX_HIP(error, hipMemsetAsync(flags, 0, kDCount * sizeof(unsigned), st));
        *again = true;
        return enqueue_cells(e, error);
    }
    std::memcpy(s.root, report->root, sizeof(s.root));
    int deepest = -1;
    for (int d = 0; d < kMaxLevels; ++d) {
        if (dcount[d] != 0) deepest = d;
    }
    s.internal = dcount[kMaxLevels];
    s.nodes = s.n + s.internal;
    // levels of the reference's compute_maximum_depth (barnes_hut.c:269-283):
    // deepest leaf depth + 1, where the deepest leaf sits one below the deepest cell
    s.max_depth = s.n == 1 ? 0 : deepest + 1;
    e->stats.node_count = s.nodes;
    e->stats.leaf_count = s.n;
    e->stats.internal_node_count = s.internal;
    e->stats.maximum_depth = static_cast<size_t>(s.max_depth) + 1;
    e->stats.accepted_approximations = report->counters[0];
    e->stats.exact_interactions = report->counters[1];
    return N_BODY_SIM_PRO_STATUS_OK;
}

}  // namespace

namespace {

// No tree to report on after an evaluation that could not be enqueued or read:
// s.n is the coming tree's already, its node counts still the last one's.
NBodySimProStatus or_no_tree(Engine* e, NBodySimProStatus status) {
    if (status != N_BODY_SIM_PRO_STATUS_OK) {
        e->bh.n = 0;
    }
    return status;
}

NBodySimProStatus enqueue_build(Engine* e, bool fp32_inputs, bool quadrupoles,
                                NBodySimProError* error);

}  // namespace

constexpr size_t kRoomyCells = size_t{1} << 20;   // particles

// Enqueues the whole build. No host read: the kernels of the build and of the
// walk that follows check the flag words, and bh_walk reads them once at its
// end (the read between the per-depth counts and the cell records left the
// GPU idle for about 15 us of every evaluation).
NBodySimProStatus bh_build(Engine* e, bool fp32_inputs, NBodySimProError* error,
                           bool quadrupoles) {
    BHState& s = e->bh;
    const size_t n = e->n;
    // the FP32 pre-order records are written on demand (bh_node_records), the
    // Morton order too (bh_morton_order)
    s.has_n32 = false;
    s.has_morton = false;
    if (n == 0) {
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_ARGUMENT,
                 "cannot build a Barnes-Hut tree for an empty system");
    }
    if (n > 0x3FFFFFFFull) {
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_ARGUMENT, "particle count exceeds 2^30");
    }
    return or_no_tree(e, enqueue_build(e, fp32_inputs, quadrupoles, error));
}

namespace {

NBodySimProStatus enqueue_build(Engine* e, bool fp32_inputs, bool quadrupoles,
                                NBodySimProError* error) {
    BHState& s = e->bh;
    const size_t n = e->n;
    // build inputs: float4 for FP32-rounded inputs, double4 for FP64 ones
    NBX_TRY(s.b4.need<char>(n * (fp32_inputs ? sizeof(float4) : sizeof(double4)), error));
    NBX_TRY(s.partial.need<double>(6 * kBBoxBlocks + 8, error));
    NBX_TRY(s.flags.need<unsigned>(kFlagWords, error));
    NBX_TRY(s.sk0.need<uint64_t>(n, error));
    NBX_TRY(s.sv0.need<uint32_t>(n, error));
    NBX_TRY(s.sk1.need<uint64_t>(n, error));
    NBX_TRY(s.sv1.need<uint32_t>(n, error));
    NBX_TRY(s.tperm.need<uint32_t>(n, error));
    NBX_TRY(s.tword.need<uint64_t>(n, error));
    NBX_TRY(s.delta.need<int32_t>(n, error));
    NBX_TRY(s.scan.need<uint32_t>(n, error));
    if (!fp32_inputs) {
        NBX_TRY(s.sp4.need<double4>(n, error));
    }
    NBX_TRY(s.s4.need<float4>(n, error));
    NBX_TRY(s.counters.need<unsigned long long>(kCounters + kPhases, error));
    NBX_TRY(s.deferred.need<int32_t>(n, error));
    s.tile = tile_positions(n, e->cu_count);
    const size_t tiles = grid_for(n, s.tile);
    NBX_TRY(s.tile_hist.need<unsigned>(kTopoRows * tiles, error));
    NBX_TRY(s.tile_base.need<unsigned>(kTopoRows * tiles, error));
    // Room for the cells of usual inputs and for a few tied positions; a tree
    // with more raises FLAG_CELLS or FLAG_LONG_RUN, and that part is repeated
    // with room for its count. Points of any smooth density make 0.469 n to
    // 0.492 n cells (the sum over levels of 8^d (1 - exp(-u) (1 + u)), u =
    // n / 8^d), two galaxies of 100,000 to 10M 0.503 n to 0.483 n, and points of
    // a plane about n / ln 4 = 0.72 n: there is room for those while it costs
    // little memory, and beyond for a quarter more than the smooth ones.
    if (s.cells_n != n) {
        s.cells = (n <= kRoomyCells ? n / 4 * 3 : n / 8 * 5) + 1024;
        s.ext_slots = n / 64 + 1024;
        s.cells_n = n;
    }
    s.n = n;
    s.inputs_fp64 = !fp32_inputs;
    s.has_n64 = !fp32_inputs;
    s.has_quad = quadrupoles;
    NBX_TRY(fp32_inputs ? enqueue_order<float4>(e, error) : enqueue_order<double4>(e, error));
    NBX_TRY(enqueue_depths(e, error));
    return enqueue_cells(e, error);
}

}  // namespace

NBodySimProStatus bh_node_records(Engine* e, NBodySimProError* error) {
    BHState& s = e->bh;
    if (s.n == 0) {
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_STATE, "no Barnes-Hut build");
    }
    if (s.has_n32) {
        return N_BODY_SIM_PRO_STATUS_OK;
    }
    NBX_TRY(s.n32.need<NodeF32>(s.nodes, error));
    const int ni = static_cast<int>(s.n);
    const int ic = static_cast<int>(s.internal);
    node_records_kernel<<<grid_for(s.nodes, kThreads), kThreads, 0, e->stream>>>(
        ni, ic, B<uint32_t>(s.scan), B<int32_t>(s.delta), B<float4>(s.s4), internal_soa(s),
        root_of(s), B<NodeF32>(s.n32));
    NBX_HIP(error, hipGetLastError());
    s.has_n32 = true;
    return N_BODY_SIM_PRO_STATUS_OK;
}

NBodySimProStatus bh_morton_order(Engine* e, NBodySimProError* error) {
    BHState& s = e->bh;
    if (s.n == 0) {
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_STATE, "no Barnes-Hut build");
    }
    if (s.has_morton) {
        return N_BODY_SIM_PRO_STATUS_OK;
    }
    hipStream_t st = e->stream;
    const unsigned g = grid_for(s.n, kThreads);
    const int ni = static_cast<int>(s.n);
    NBX_TRY(s.mkey.need<uint64_t>(s.n, error));
    NBX_TRY(s.mperm.need<uint32_t>(s.n, error));
    if (s.inputs_fp64) {
        morton_keys_kernel<double4><<<g, kThreads, 0, st>>>(
            B<double4>(s.b4), ni, root_of(s), B<uint64_t>(s.mkey), B<uint64_t>(s.sk0),
            B<uint32_t>(s.sv0));
    } else {
        morton_keys_kernel<float4><<<g, kThreads, 0, st>>>(
            B<float4>(s.b4), ni, root_of(s), B<uint64_t>(s.mkey), B<uint64_t>(s.sk0),
            B<uint32_t>(s.sv0));
    }
    NBX_HIP(error, hipGetLastError());
    NBX_TRY(radix_sort_pairs(st, B<uint64_t>(s.sk0), B<uint32_t>(s.sv0), B<uint64_t>(s.sk1),
                             B<uint32_t>(s.sv1), s.n, 63, s.hist, error));
    NBX_HIP(error, hipMemcpyAsync(s.mperm.p, s.sv0.p, s.n * sizeof(uint32_t),
                                  hipMemcpyDeviceToDevice, st));
    NBX_HIP(error, hipStreamSynchronize(st));
    s.has_morton = true;
    return N_BODY_SIM_PRO_STATUS_OK;
}

namespace {

bool walks_lists(const Engine* e, bool fp64_exact) {
    return !fp64_exact && (e->flags & NBX_FLAG_BH_REFERENCE_LISTS) != 0;
}

// The walk of the build before it in the stream (nothing where the reference
// lists are asked for: those wait for the node records).
NBodySimProStatus enqueue_walk(Engine* e, const NBodySimProGravity* g, bool fp64_exact,
                               float* features, NBodySimProError* error) {
    BHState& s = e->bh;
    hipStream_t st = e->stream;
    const int ni = static_cast<int>(s.n);
    // the counters were cleared by this build's bbox_partial_kernel
    const double theta2 = e->theta * e->theta;
    const unsigned blocks = grid_for(s.n, kThreads);
    if (fp64_exact && !s.has_n64) {
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_STATE,
                 "the exact walk needs a build on FP64 inputs");
    }
    if (features != nullptr && !s.has_quad) {
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_STATE,
                 "the feature walk needs a build with quadrupole records");
    }
    const float4* gq = features != nullptr ? B<float4>(s.gquad) : nullptr;
    const float Gf = static_cast<float>(g->gravitational_constant);
    const float e2 = static_cast<float>(g->softening_squared);
    const float th2 = static_cast<float>(theta2);
    const unsigned* flags = B<unsigned>(s.flags);
    unsigned long long* cnts = B<unsigned long long>(s.counters);
    auto group_walk = [&]() {
        const GroupNode* gn = B<GroupNode>(s.gnode);
        int* deferred = B<int32_t>(s.deferred);
        // one shared walk per group (no split) or the split's budget
        const int max_walks = (e->flags & NBX_FLAG_BH_NO_SPLIT) ? 1 : kMaxSubWalks;
        // The member test is on unless the box test alone is asked for; the
        // feature walk of the learned path always takes it. (Measured on
        // MI355X, two-galaxy, box test alone -> with the member test: plain
        // walk at theta = 0.7, 1M: 0.844 -> 0.819 ms, 1.53G -> 1.18G
        // interactions; theta = 0.5, 10M: 18.3 -> 17.2 ms; feature walk at
        // theta = 1.0, 10M: 9.61 -> 7.96 ms.)
        const bool member_test =
            features != nullptr || (e->flags & NBX_FLAG_BH_BOX_TEST) == 0;
        // (the feature walk's sums keep their order: one wave a group)
        const size_t groups = (s.n + kWave - 1) / kWave;
        const int team = features != nullptr ? 1 : walk_team(groups, e->cu_count);
        const int chunk_log = team > 1 ? kTeamChunkLog : kChunkLog;
        // whole rounds of one chunk per XCD (blocks past the last group exit)
        const size_t round = static_cast<size_t>(kXcds) << chunk_log;
        const unsigned grid_g = static_cast<unsigned>((groups + round - 1) / round * round);
        if (features != nullptr) {
            group_walk_kernel<true, 1><<<grid_g, kWave, 0, st>>>(
                flags, deferred, gn, B<float4>(s.s4), B<uint32_t>(s.tperm),
                B<uint64_t>(s.tword), ext_table(s), ni, Gf, e2, th2, e->ax, e->ay, e->az, cnts,
                features, gq, max_walks, member_test, chunk_log);
        } else {
            auto go = [&](auto kernel) {
                kernel<<<grid_g, team * kWave, 0, st>>>(
                    flags, deferred, gn, B<float4>(s.s4), B<uint32_t>(s.tperm),
                    B<uint64_t>(s.tword), ext_table(s), ni, Gf, e2, th2, e->ax, e->ay, e->az, cnts,
                    nullptr, nullptr, max_walks, member_test, chunk_log);
            };
            if (team == 4) {
                go(group_walk_kernel<false, 4>);
            } else if (team == 2) {
                go(group_walk_kernel<false, 2>);
            } else {
                go(group_walk_kernel<false, 1>);
            }
        }
    };
    if (fp64_exact) {
        auto go = [&](auto kernel, int queries) {
            kernel<<<grid_for(s.n, queries), kWave, 0, st>>>(
                flags, B<NodeF64>(s.n64), B<double4>(s.sp4), B<uint32_t>(s.tperm), ni,
                g->gravitational_constant, g->softening_squared, theta2, e->ax, e->ay, e->az,
                cnts);
        };
        const size_t waves = static_cast<size_t>(e->cu_count) * 8;   // two per SIMD
        if (s.n <= 8 * waves) {
            go(walk_f64_kernel<8>, 8);
        } else if (s.n <= 16 * waves) {
            go(walk_f64_kernel<16>, 16);
        } else if (s.n <= 42 * waves) {
            go(walk_f64_kernel<32>, 32);
        } else {
            go(walk_f64_kernel<64>, 64);
        }
    } else if (!walks_lists(e, fp64_exact)) {
        group_walk();
    }
    NBX_HIP(error, hipGetLastError());
    return N_BODY_SIM_PRO_STATUS_OK;
}

}  // namespace

NBodySimProStatus bh_enqueue(Engine* e, const NBodySimProGravity* g, bool fp64_exact, int slot,
                             NBodySimProError* error) {
    NBX_TRY(bh_build(e, !fp64_exact, error));
    NBX_TRY(or_no_tree(e, enqueue_walk(e, g, fp64_exact, nullptr, error)));
    return or_no_tree(e, enqueue_report(e, slot, error));
}

NBodySimProStatus bh_peek(Engine* e, int slot, bool* clean, NBodySimProError* error) {
    NBX_TRY(or_no_tree(e, await_report(e, slot, error)));
    *clean = report_clean(report_of(e->bh, slot));
    return N_BODY_SIM_PRO_STATUS_OK;
}

bool bh_runs_ahead(const Engine* e, NBXAlgorithm algorithm) {
    return (algorithm == NBX_ALGORITHM_BARNES_HUT &&
            (e->flags & NBX_FLAG_BH_REFERENCE_LISTS) == 0) ||
           algorithm == NBX_ALGORITHM_BARNES_HUT_FP64;
}

EvaluationGate bh_gate(Engine* e) {
    return {B<uint4>(e->bh.flags), B<unsigned long long>(e->bh.counters) + 2};
}

NBodySimProStatus bh_finish(Engine* e, const NBodySimProGravity* g, bool fp64_exact,
                            float* features, int slot, NBodySimProError* error) {
    BHState& s = e->bh;
    hipStream_t st = e->stream;
    const int ni = static_cast<int>(s.n);
    const float Gf = static_cast<float>(g->gravitational_constant);
    const float e2 = static_cast<float>(g->softening_squared);
    const float th2 = static_cast<float>(e->theta * e->theta);
    unsigned long long* cnts = B<unsigned long long>(s.counters);
    // per-query reference-list walk of nq queries (all tree positions, or the
    // listed ones) on the FP32 pre-order records (a repair moves the cells'
    // arrays, so their addresses are taken here)
    auto per_query_walk = [&](const int* list, int nq) -> NBodySimProStatus {
        NBX_TRY(bh_node_records(e, error));
        const unsigned wblocks = grid_for(static_cast<size_t>(nq), kThreads * kWalkQueries);
        const unsigned wgrid = (wblocks + kXcds - 1) / kXcds * kXcds;
        const NodeF32* n32 = B<NodeF32>(s.n32);
        const int nn = static_cast<int>(s.nodes);
        if (features != nullptr) {
            walk_f32_kernel<true, kWalkQueries><<<wgrid, kThreads, 0, st>>>(
                n32, nn, B<float4>(s.s4), B<uint32_t>(s.tperm), list, nq, Gf, e2, th2, e->ax,
                e->ay, e->az, cnts, features, B<float4>(s.gquad));
        } else {
            walk_f32_kernel<false, kWalkQueries><<<wgrid, kThreads, 0, st>>>(
                n32, nn, B<float4>(s.s4), B<uint32_t>(s.tperm), list, nq, Gf, e2, th2, e->ax,
                e->ay, e->az, cnts, nullptr, nullptr);
        }
        NBX_HIP(error, hipGetLastError());
        return N_BODY_SIM_PRO_STATUS_OK;
    };
    const bool lists = walks_lists(e, fp64_exact);
    const bool group = !fp64_exact && !lists;
    float per_query_ms = 0.f;
    s.slot = slot;
    // Each repetition follows a repaired build: an order on all the key bits,
    // then room for the extension words or an order on all of those, then room
    // for its cells, at most.
    bool again = true;
    for (int attempt = 0; again && attempt < 4; ++attempt) {
        if (attempt > 0) {
            NBX_TRY(or_no_tree(e, enqueue_walk(e, g, fp64_exact, features, error)));
            NBX_TRY(or_no_tree(e, enqueue_report(e, slot, error)));
        }
        NBX_TRY(or_no_tree(e, read_build(e, slot, &again, error)));
        s.clean = attempt == 0 && !again && report_of(s, slot)->counters[2] == 0;
    }
    if (again) {
        s.n = 0;
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_STATE, "the tree build did not settle");
    }
    const unsigned long long deferred = report_of(s, slot)->counters[2];
    if (lists || (group && deferred > 0)) {
        // Reference lists for all queries, or for those the group walk could
        // not give a shared list (a range the split could not make compact
        // within its budget, or a stack overflow; none in most evaluations),
        // after the FP32 pre-order records are written.
        if (deferred > s.n) {
            NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_STATE,
                     "deferred query count out of range");
        }
        NBX_HIP(error, hipEventRecord(e->ev[0], st));
        NBX_TRY(lists ? per_query_walk(nullptr, ni)
                      : per_query_walk(B<int32_t>(s.deferred), static_cast<int>(deferred)));
        NBX_HIP(error, hipEventRecord(e->ev[1], st));
        unsigned long long counts[2] = {0, 0};
        NBX_HIP(error, hipMemcpyAsync(counts, s.counters.p, sizeof(counts),
                                      hipMemcpyDeviceToHost, st));
        NBX_HIP(error, hipStreamSynchronize(st));
        e->stats.accepted_approximations = counts[0];
        e->stats.exact_interactions = counts[1];
        NBX_HIP(error, hipEventElapsedTime(&per_query_ms, e->ev[0], e->ev[1]));
    }
    s.per_query_ms = per_query_ms;
    s.walked_lists = lists;
    return N_BODY_SIM_PRO_STATUS_OK;
}

NBodySimProStatus bh_walk(Engine* e, const NBodySimProGravity* g, bool fp64_exact, float* features,
                          NBodySimProError* error) {
    NBX_TRY(or_no_tree(e, enqueue_walk(e, g, fp64_exact, features, error)));
    NBX_TRY(or_no_tree(e, enqueue_report(e, 0, error)));
    return bh_finish(e, g, fp64_exact, features, 0, error);
}

void bh_timings(Engine* e) {
    BHState& s = e->bh;
    // the phases' starts on the device clock, a phase that had no kernel at
    // the next one's
    unsigned long long* at = report_of(s, s.slot)->counters + kCounters;
    if (s.walked_lists) {
        at[PHASE_WALK] = at[PHASE_END];
    }
    if (s.n <= static_cast<size_t>(s.tile)) {
        at[PHASE_COM] = at[PHASE_WALK];
    }
    auto ms = [&](int from, int to) {
        return at[to] > at[from] ? static_cast<double>(at[to] - at[from]) / e->clock_khz : 0.0;
    };
    NBXTimings tm{};
    tm.bbox_keys_ms = ms(PHASE_KEYS, PHASE_SORT);
    tm.sort_ms = ms(PHASE_SORT, PHASE_TREE);
    tm.tree_ms = ms(PHASE_TREE, PHASE_COM);
    tm.com_ms = ms(PHASE_COM, PHASE_WALK);
    tm.walk_ms = ms(PHASE_WALK, PHASE_END) + s.per_query_ms;
    tm.force_ms = ms(PHASE_KEYS, PHASE_END) + s.per_query_ms;
    tm.kernel_ms = tm.walk_ms;
    tm.kernel_flops = 20.0 * static_cast<double>(e->stats.accepted_approximations +
                                                 e->stats.exact_interactions);
    e->timings = tm;
    e->stats.build_time_seconds = ms(PHASE_KEYS, PHASE_WALK) * 1e-3;
    e->stats.evaluation_time_seconds = tm.walk_ms * 1e-3;
}

NBodySimProStatus barnes_hut(Engine* e, const NBodySimProGravity* g, bool fp64_exact,
                             NBodySimProError* error) {
    NBX_TRY(bh_enqueue(e, g, fp64_exact, 0, error));
    return bh_end(e, g, fp64_exact, 0, error);
}

NBodySimProStatus bh_end(Engine* e, const NBodySimProGravity* g, bool fp64_exact, int slot,
                         NBodySimProError* error) {
    NBX_TRY(bh_finish(e, g, fp64_exact, nullptr, slot, error));
    bh_timings(e);
    // walk bytes: every query reads its position (and permutation entry) and
    // writes 3 doubles; the cell records the walk reads are counted once per
    // launch (they stay in L2 across waves): GroupNode records for the group
    // walk, pre-order node records for the per-query walks.
    const bool group = !fp64_exact && !walks_lists(e, fp64_exact);
    const double node_bytes =
        fp64_exact ? static_cast<double>(e->bh.nodes) * sizeof(NodeF64)
        : group    ? static_cast<double>(e->bh.internal) * sizeof(GroupNode)
                   : static_cast<double>(e->bh.nodes) * sizeof(NodeF32);
    e->timings.kernel_bytes = static_cast<double>(e->bh.n) * ((fp64_exact ? 24.0 : 16.0) + 24.0 + 4.0) +
                      node_bytes;
    return N_BODY_SIM_PRO_STATUS_OK;
}

}  // namespace nbx
