// nbx_engine.hip - engine lifecycle, host<->device transfer, force dispatch,
// FP64 integrator and diagnostics, parity probes and the drop-in force
// functions of the C ABI (include/nbx_engine.h).
#include "nbx_exact.h"
#include "nbx_internal.h"

#include <algorithm>
#include <array>
#include <cmath>
#include <cstdio>
#include <mutex>
#include <new>
#include <vector>

namespace nbx {

void set_error(NBodySimProError* error, NBodySimProStatus status, const char* file, int line,
               const char* message) {
    if (error == nullptr) {
        return;
    }
    error->status = status;
    error->source_file = file;
    error->source_line = line;
    if (message == nullptr) {
        error->message[0] = '\0';
        return;
    }
    const size_t len = std::strlen(message);
    const size_t copy = len < sizeof(error->message) ? len : sizeof(error->message) - 1;
    std::memcpy(error->message, message, copy);
    error->message[copy] = '\0';
}

NBodySimProStatus map_hip_error(hipError_t e) {
    switch (e) {
        case hipSuccess:
            return N_BODY_SIM_PRO_STATUS_OK;
        case hipErrorOutOfMemory:
            return N_BODY_SIM_PRO_STATUS_OUT_OF_MEMORY;
        case hipErrorNoDevice:
        case hipErrorInvalidDevice:
        case hipErrorInsufficientDriver:
            return N_BODY_SIM_PRO_STATUS_UNSUPPORTED_PLATFORM;
        default:
            return N_BODY_SIM_PRO_STATUS_INVALID_STATE;
    }
}

NBodySimProStatus ensure(void** ptr, size_t* cap, size_t bytes, NBodySimProError* error) {
    if (bytes <= *cap && *ptr != nullptr) {
        return N_BODY_SIM_PRO_STATUS_OK;
    }
    if (*ptr != nullptr) {
        NBX_HIP(error, hipFree(*ptr));
        *ptr = nullptr;
        *cap = 0;
    }
    // One eighth of headroom: sizes that follow the tree (cells, nodes) move
    // by a fraction of a percent from step to step, and every new maximum
    // would otherwise cost a hipFree (which waits for the device) and a
    // hipMalloc inside the evaluation. (Measured on MI355X, 1M two-galaxy
    // leapfrog: one build in eight paid about 0.2 ms for it.)
    size_t want = bytes + bytes / 8;
    want = want < 256 ? 256 : want;
    NBX_HIP(error, hipMalloc(ptr, want));
    *cap = want;
    return N_BODY_SIM_PRO_STATUS_OK;
}

namespace {

constexpr int kThreads = 256;

// Every grow-on-demand device buffer of an engine (Barnes-Hut build and walk
// arrays, diagnostics scratch); the array's size follows the list.
auto work_buffers(Engine* e) {
    BHState& s = e->bh;
    return std::array{&s.b4, &s.partial, &s.flags, &s.sk0, &s.sk1, &s.sv0, &s.sv1, &s.hist,
            &s.mkey, &s.mperm, &s.tperm, &s.tword, &s.ext, &s.ext_orig, &s.delta, &s.scan,
            &s.sp4, &s.s4, &s.tile_hist, &s.tile_base, &s.n64,
            &s.n32, &s.icom, &s.irec, &s.idepth, &s.gnode, &s.im2, &s.gquad,
            &s.tmp32, &s.counters, &s.deferred, &e->scratch, &e->scratch2};
}

void free_buf(Buf& b) {
    if (b.p != nullptr) {
        (void)hipFree(b.p);
    }
    b.p = nullptr;
    b.cap = 0;
}

// Transfers of pageable memory of up to this many bytes go through the engine's
// pinned block: one copy by the host and one kernel for all arrays, where a
// copy command an array costs 6 to 15 us each; beyond, the host's copy (27
// GB/s) costs as much. Pinned memory needs no block, the kernel reaches it
// itself. (Ten arrays, up / down, us. Copy commands from pageable, from pinned
// memory -> staged, kernel alone: 1,000 particles 92 / 169, 58 / 59 -> 16 / 16,
// 15 / 14; 10,000: 114 / 152, 114 / 114 -> 38 / 46, 28 / 27; 30,000: 143 / 215,
// 141 / 140 -> 90 / 113, 57 / 56; 200,000: 519 / 944, 378 / 380 -> -, 313 /
// 312, which is the link's rate.)
constexpr size_t kStageBytes = size_t{5} << 19;

// ---------------------------------------------------------------- integrator
// src/c/physics/integrator.c:64-83 (compiled with contraction off).
__global__ void kick_drift_kernel(double* __restrict__ px, double* __restrict__ py,
                                  double* __restrict__ pz, double* __restrict__ vx,
                                  double* __restrict__ vy, double* __restrict__ vz,
                                  const double* __restrict__ ax, const double* __restrict__ ay,
                                  const double* __restrict__ az, int n, double half, double dt) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        const double nvx = vx[i] + ax[i] * half;
        const double nvy = vy[i] + ay[i] * half;
        const double nvz = vz[i] + az[i] * half;
        vx[i] = nvx;
        vy[i] = nvy;
        vz[i] = nvz;
        px[i] = px[i] + nvx * dt;
        py[i] = py[i] + nvy * dt;
        pz[i] = pz[i] + nvz * dt;
    }
}

// The kick that ends a step and the kick and drift that begin the next
// (integrator.c:77-83 and :64-75), with the same two roundings of the
// velocity: 72 bytes a particle less than the two kernels (1M particles: 14 +
// 20 us, now 20). Nothing moves unless the gate is open: the evaluation before
// may have been left unfinished, which the host learns later.
__global__ void kick_kick_drift_kernel(double* __restrict__ px, double* __restrict__ py,
                                       double* __restrict__ pz, double* __restrict__ vx,
                                       double* __restrict__ vy, double* __restrict__ vz,
                                       const double* __restrict__ ax,
                                       const double* __restrict__ ay,
                                       const double* __restrict__ az, int n, double half,
                                       double dt, EvaluationGate gate) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && gate.open()) {
        const double hx = ax[i] * half, hy = ay[i] * half, hz = az[i] * half;
        const double nvx = (vx[i] + hx) + hx;
        const double nvy = (vy[i] + hy) + hy;
        const double nvz = (vz[i] + hz) + hz;
        vx[i] = nvx;
        vy[i] = nvy;
        vz[i] = nvz;
        px[i] = px[i] + nvx * dt;
        py[i] = py[i] + nvy * dt;
        pz[i] = pz[i] + nvz * dt;
    }
}

__global__ void kick_kernel(double* __restrict__ vx, double* __restrict__ vy,
                            double* __restrict__ vz, const double* __restrict__ ax,
                            const double* __restrict__ ay, const double* __restrict__ az, int n,
                            double half,
                            unsigned long long* __restrict__ clock) {
    clock_in(clock);
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        vx[i] = vx[i] + ax[i] * half;
        vy[i] = vy[i] + ay[i] * half;
        vz[i] = vz[i] + az[i] * half;
    }
}

// integrator.c:35-43
__global__ void euler_kernel(double* __restrict__ px, double* __restrict__ py,
                             double* __restrict__ pz, double* __restrict__ vx,
                             double* __restrict__ vy, double* __restrict__ vz,
                             const double* __restrict__ ax, const double* __restrict__ ay,
                             const double* __restrict__ az, int n, double dt,
                             unsigned long long* __restrict__ clock) {
    clock_in(clock);
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        px[i] = px[i] + vx[i] * dt;
        py[i] = py[i] + vy[i] * dt;
        pz[i] = pz[i] + vz[i] * dt;
        vx[i] = vx[i] + ax[i] * dt;
        vy[i] = vy[i] + ay[i] * dt;
        vz[i] = vz[i] + az[i] * dt;
    }
}

// ---------------------------------------------------------------- diagnostics
constexpr int kDiag = 11;

// Per-block FP64 partial sums of the numerics.c:5-81 terms (fixed order).
__global__ __launch_bounds__(kThreads) void diag_partial_kernel(
    const double* __restrict__ px, const double* __restrict__ py, const double* __restrict__ pz,
    const double* __restrict__ vx, const double* __restrict__ vy, const double* __restrict__ vz,
    const double* __restrict__ m, int n, double* __restrict__ partial) {
    __shared__ double s[kDiag][kThreads];
    double acc[kDiag];
#pragma unroll
    for (int k = 0; k < kDiag; ++k) {
        acc[k] = 0.0;
    }
    for (int i = blockIdx.x * kThreads + threadIdx.x; i < n; i += gridDim.x * kThreads) {
        const double mass = m[i];
        const double x = px[i], y = py[i], z = pz[i];
        const double u = vx[i], v = vy[i], w = vz[i];
        acc[0] += 0.5 * mass * (u * u + v * v + w * w);
        acc[1] += mass;
        acc[2] += mass * u;
        acc[3] += mass * v;
        acc[4] += mass * w;
        acc[5] += mass * (y * w - z * v);
        acc[6] += mass * (z * u - x * w);
        acc[7] += mass * (x * v - y * u);
        acc[8] += mass * x;
        acc[9] += mass * y;
        acc[10] += mass * z;
    }
#pragma unroll
    for (int k = 0; k < kDiag; ++k) {
        s[k][threadIdx.x] = acc[k];
    }
    __syncthreads();
    for (int off = kThreads / 2; off > 0; off >>= 1) {
        if (threadIdx.x < static_cast<unsigned>(off)) {
#pragma unroll
            for (int k = 0; k < kDiag; ++k) {
                s[k][threadIdx.x] += s[k][threadIdx.x + off];
            }
        }
        __syncthreads();
    }
    if (threadIdx.x < kDiag) {
        partial[blockIdx.x * kDiag + threadIdx.x] = s[threadIdx.x][0];
    }
}

// Softened potential, pairs j > i (numerics.c:83-116). The triangle is cut into
// units of 64 targets (one per lane) by 16 sources (scalar loads), dealt out
// in equal runs to at most 8,192 waves, so that the last rows of targets, which
// have few sources left, cost no more than the first; each wave keeps its
// row's targets from unit to unit. The bound is FP64 issue. (20,000 particles:
// 131 us, 1.5 T pairs/s; 3.0 ms with a thread per target and the IEEE
// operations, the first targets' waves running longest.)
constexpr int kPotWaves = kThreads / kWave;
constexpr int64_t kPotMaxWaves = 8192;

// Units before row r of 64 targets, of `chunks` source chunks.
__host__ __device__ inline int64_t pot_units_before(int64_t r, int64_t chunks) {
    return r * chunks - (kWave / kPotSources) * (r * (r - 1) / 2);
}

__global__ __launch_bounds__(kThreads) void potential_partial_kernel(
    const double* __restrict__ px, const double* __restrict__ py, const double* __restrict__ pz,
    const double* __restrict__ m, int n, double eps2, int64_t units, double* __restrict__ partial) {
    __shared__ double s[kPotWaves];
    const int lane = threadIdx.x & (kWave - 1);
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int64_t wave = static_cast<int64_t>(blockIdx.x) * kPotWaves + wid;
    const int64_t waves = static_cast<int64_t>(gridDim.x) * kPotWaves;
    const int64_t each = units / waves, more = units % waves;
    int64_t left = each + (wave < more ? 1 : 0);
    double sum = 0.0;
    if (left > 0) {
        const int64_t u = wave * each + (wave < more ? wave : more);
        const int64_t chunks = (n + kPotSources - 1) / kPotSources;
        const double b = static_cast<double>(chunks) + 2.0;
        int64_t row = static_cast<int64_t>((b - sqrt(fmax(b * b - 8.0 * u, 0.0))) * 0.25);
        while (row > 0 && pot_units_before(row, chunks) > u) {
            --row;
        }
        while (pot_units_before(row + 1, chunks) <= u) {
            ++row;
        }
        const int last = static_cast<int>(chunks);
        int r = __builtin_amdgcn_readfirstlane(static_cast<int>(row));
        int c = __builtin_amdgcn_readfirstlane(
            static_cast<int>(u - pot_units_before(row, chunks)) + r * (kWave / kPotSources));
        while (left > 0) {
            const int i = r * kWave + lane;
            const int ic = min(i, n - 1);
            const double x = px[ic], y = py[ic], z = pz[ic], mi = m[ic];
            const int end = left < last - c ? c + static_cast<int>(left) : last;
            left -= end - c;
            // the row's first chunks hold its own targets, the last may be cut
            for (; c < end; ++c) {
                const int j0 = c * kPotSources;
                if (j0 < (r + 1) * kWave || j0 + kPotSources > n) {
                    sum += pot_unit<true>(px, py, pz, m, n, j0, i, x, y, z, mi, eps2);
                } else {
                    sum += pot_unit<false>(px, py, pz, m, n, j0, i, x, y, z, mi, eps2);
                }
            }
            ++r;
            c = r * (kWave / kPotSources);
        }
    }
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) {
        sum += __shfl_xor(sum, off);
    }
    if (lane == 0) {
        s[wid] = sum;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = s[0];
        for (int k = 1; k < kPotWaves; ++k) {
            t += s[k];
        }
        partial[blockIdx.x] = t;
    }
}

// Fixed-order reduction of `count` rows of kDiag partials, one workgroup a
// column, and of the potential's `pot_count` partials by one more.
__global__ __launch_bounds__(kThreads) void reduce_rows_kernel(const double* __restrict__ partial,
                                                              int count,
                                                              const double* __restrict__ pot,
                                                              int pot_count,
                                                              double* __restrict__ out) {
    __shared__ double s[kThreads];
    const int k = blockIdx.x;
    const bool column = k < kDiag;
    const double* p = column ? partial + k : pot;
    const int rows = column ? count : pot_count;
    const int stride = column ? kDiag : 1;
    double acc = 0.0;
    for (int r = threadIdx.x; r < rows; r += kThreads) {
        acc += p[r * stride];
    }
    s[threadIdx.x] = acc;
    __syncthreads();
    for (int off = kThreads / 2; off > 0; off >>= 1) {
        if (threadIdx.x < static_cast<unsigned>(off)) {
            s[threadIdx.x] += s[threadIdx.x + off];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[k] = s[0];
    }
}

NBodySimProStatus check_engine(NBXEngine* engine, NBodySimProError* error) {
    if (engine == nullptr) {
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_ARGUMENT, "engine must not be null");
    }
    NBX_HIP(error, hipSetDevice(engine->e.device));
    return N_BODY_SIM_PRO_STATUS_OK;
}

// The non-null arrays of a transfer: host and device side, n doubles each.
struct ArrayList {
    double* host[10];
    double* dev[10];
    int count = 0;

    void add(double* h, double* d) {
        if (h != nullptr && d != nullptr) {
            host[count] = h;
            dev[count++] = d;
        }
    }
};

// One array a grid row, between the device arrays and pinned host memory.
template <bool TO_HOST>
__global__ __launch_bounds__(kThreads) void stage_kernel(ArrayList list, int n,
                                                         unsigned long long* __restrict__ clock) {
    if (blockIdx.y == 0) {
        clock_in(clock);
    }
    const int i = blockIdx.x * kThreads + threadIdx.x;
    if (i < n) {
        double* d = list.dev[blockIdx.y] + i;
        double* h = list.host[blockIdx.y] + i;
        if (TO_HOST) {
            *h = *d;
        } else {
            *d = *h;
        }
    }
}

template <bool TO_HOST>
NBodySimProStatus enqueue_stage(Engine* e, const ArrayList& list, size_t n,
                                NBodySimProError* error) {
    stage_kernel<TO_HOST><<<dim3(grid_for(n, kThreads), list.count), kThreads, 0, e->stream>>>(
        list, static_cast<int>(n), TO_HOST ? direct_end(e) : nullptr);
    NBX_HIP(error, hipGetLastError());
    return N_BODY_SIM_PRO_STATUS_OK;
}

// Pinned memory. An engine that can stage all it holds gets one block for the
// reports and the stage when it is created (an allocation takes 260 us and
// more); a larger one gets its stage with its first small transfer.
bool pinned(void** p, size_t bytes) {
    if (*p == nullptr && hipHostMalloc(p, bytes, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        *p = nullptr;
    }
    return *p != nullptr;
}

bool pinned_report(Engine* e) {
    const size_t bytes = e->capacity * 10 * sizeof(double);
    const bool both = e->capacity <= kStageBytes / (10 * sizeof(double));
    if (!pinned(&e->bh.report, kReportBytes + (both ? bytes : 0))) {
        return false;
    }
    std::memset(e->bh.report, 0, kReportBytes);   // no evaluation's number
    if (both) {
        e->stage = static_cast<char*>(e->bh.report) + kReportBytes;
        e->stage_bytes = bytes;
        e->stage_in_report = true;
    }
    return true;
}

// Whether two host arrays of a transfer share memory.
bool host_arrays_overlap(const ArrayList& list, size_t bytes) {
    for (int k = 1; k < list.count; ++k) {
        for (int j = 0; j < k; ++j) {
            const uintptr_t a = reinterpret_cast<uintptr_t>(list.host[k]);
            const uintptr_t b = reinterpret_cast<uintptr_t>(list.host[j]);
            if (a < b + bytes && b < a + bytes) {
                return true;
            }
        }
    }
    return false;
}

// How a transfer goes: KERNEL where every host array is pinned memory that
// the device addresses as the host does (one kernel in place of a copy command
// an array), STAGED through the engine's pinned block where the host's
// processor can copy the arrays there, COPIES otherwise. The kernel stores the
// arrays in any order: to host arrays that share memory it does not go, so the
// later array of the view stays where they do.
enum class Route { KERNEL, STAGED, COPIES };

Route route_of(Engine* e, const ArrayList& list, size_t n, bool to_host) {
    const size_t bytes = n * sizeof(double);
    if (list.count == 0 || n == 0 || n > 0x7FFFFF00u) {
        return Route::COPIES;   // (the kernel's positions are ints)
    }
    int direct = 0;
    for (int k = 0; k < list.count; ++k) {
        hipPointerAttribute_t at{};
        if (hipPointerGetAttributes(&at, list.host[k]) != hipSuccess) {
            (void)hipGetLastError();   // memory HIP does not know: the host's
            continue;
        }
        if (at.type == hipMemoryTypeDevice) {
            return Route::COPIES;
        }
        if (at.type == hipMemoryTypeHost && at.device == e->device &&
            at.devicePointer == list.host[k]) {
            hipDeviceptr_t base = nullptr;
            size_t size = 0;
            if (hipMemGetAddressRange(&base, &size, list.host[k]) != hipSuccess) {
                (void)hipGetLastError();
                continue;
            }
            const char* first = reinterpret_cast<const char*>(list.host[k]);
            const char* start = static_cast<const char*>(base);
            direct += first >= start && first + bytes <= start + size;   // the whole array
        }
    }
    if (direct == list.count && !(to_host && host_arrays_overlap(list, bytes))) {
        return Route::KERNEL;
    }
    if (list.count * bytes > kStageBytes) {
        return Route::COPIES;
    }
    if (e->stage == nullptr && pinned(&e->stage, kStageBytes)) {
        e->stage_bytes = kStageBytes;
    }
    return list.count * bytes <= e->stage_bytes ? Route::STAGED : Route::COPIES;
}

ArrayList stage_places(Engine* e, const ArrayList& list, size_t n) {
    ArrayList places = list;
    for (int k = 0; k < list.count; ++k) {
        places.host[k] = static_cast<double*>(e->stage) + k * n;
    }
    return places;
}

// Host -> device. *enqueued: the staged values are on their way, and the
// pinned block must not be written again before the stream has passed them.
// Else complete.
NBodySimProStatus copy_in(Engine* e, const ArrayList& list, size_t n, bool* enqueued,
                          NBodySimProError* error) {
    const Route route = route_of(e, list, n, false);
    *enqueued = route == Route::STAGED;
    if (route == Route::STAGED) {
        const ArrayList places = stage_places(e, list, n);
        for (int k = 0; k < list.count; ++k) {
            std::memcpy(places.host[k], list.host[k], n * sizeof(double));
        }
        return enqueue_stage<false>(e, places, n, error);
    }
    if (route == Route::KERNEL) {
        NBX_TRY(enqueue_stage<false>(e, list, n, error));
    } else {
        for (int k = 0; k < list.count && n > 0; ++k) {
            NBX_HIP(error, hipMemcpyAsync(list.dev[k], list.host[k], n * sizeof(double),
                                          hipMemcpyHostToDevice, e->stream));
        }
    }
    NBX_HIP(error, hipStreamSynchronize(e->stream));
    return N_BODY_SIM_PRO_STATUS_OK;
}

// Device -> host, complete on return.
NBodySimProStatus copy_out(Engine* e, const ArrayList& list, size_t n, NBodySimProError* error) {
    const Route route = route_of(e, list, n, true);
    if (route == Route::STAGED) {
        const ArrayList places = stage_places(e, list, n);
        NBX_TRY(enqueue_stage<true>(e, places, n, error));
        NBX_HIP(error, hipStreamSynchronize(e->stream));
        for (int k = 0; k < list.count; ++k) {
            std::memcpy(list.host[k], places.host[k], n * sizeof(double));
        }
        return N_BODY_SIM_PRO_STATUS_OK;
    }
    if (route == Route::KERNEL) {
        NBX_TRY(enqueue_stage<true>(e, list, n, error));
    } else {
        NBX_TRY(direct_timings(e, error));   // (the copies are no part of the evaluation)
        for (int k = 0; k < list.count && n > 0; ++k) {
            NBX_HIP(error, hipMemcpyAsync(list.host[k], list.dev[k], n * sizeof(double),
                                          hipMemcpyDeviceToHost, e->stream));
        }
    }
    NBX_HIP(error, hipStreamSynchronize(e->stream));
    return N_BODY_SIM_PRO_STATUS_OK;
}

std::mutex g_default_mutex;
NBXEngine* g_default = nullptr;

}  // namespace

NBodySimProStatus compute_force(Engine* e, NBXAlgorithm algorithm, const NBodySimProGravity* g,
                                NBodySimProError* error) {
    e->pending = 0;
    e->ended = false;
    switch (algorithm) {
        case NBX_ALGORITHM_DIRECT_FP64:
            return direct_fp64(e, g, error);
        case NBX_ALGORITHM_DIRECT_FP32:
            return direct_fp32(e, g, error);
        case NBX_ALGORITHM_BARNES_HUT:
            return barnes_hut(e, g, false, error);
        case NBX_ALGORITHM_BARNES_HUT_FP64:
            return barnes_hut(e, g, true, error);
        case NBX_ALGORITHM_BH_LEARNED:
            return bh_learned(e, g, error);
    }
    NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_ARGUMENT, "unknown force algorithm");
}

}  // namespace nbx

using nbx::Engine;

extern "C" {

int nbx_device_count(void) {
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess) {
        return 0;
    }
    return count;
}

int nbx_device_info(int device, char* name, size_t len, int* compute_units) {
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || device < 0 || device >= count) {
        return -1;
    }
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) != hipSuccess) {
        return -1;
    }
    if (name != nullptr && len > 0) {
        std::snprintf(name, len, "%s (%s)", prop.name, prop.gcnArchName);
    }
    if (compute_units != nullptr) {
        *compute_units = prop.multiProcessorCount;
    }
    return 0;
}

int nbx_algorithm_from_name(const char* name) {
    if (name == nullptr) {
        return -1;
    }
    static const char* names[] = {"hip_direct_fp64", "hip_direct_fp32", "hip_barnes_hut",
                                  "hip_barnes_hut_fp64", "hip_bh_learned"};
    for (int k = 0; k < 5; ++k) {
        if (std::strcmp(name, names[k]) == 0) {
            return k;
        }
    }
    return -1;
}

const char* nbx_algorithm_name(int algorithm) {
    static const char* names[] = {"hip_direct_fp64", "hip_direct_fp32", "hip_barnes_hut",
                                  "hip_barnes_hut_fp64", "hip_bh_learned"};
    return (algorithm >= 0 && algorithm < 5) ? names[algorithm] : nullptr;
}

NBXEngine* nbx_engine_create(const NBXConfig* config, NBodySimProError* error) {
    if (config == nullptr || config->capacity == 0) {
        nbx::set_error(error, N_BODY_SIM_PRO_STATUS_INVALID_ARGUMENT, __FILE__, __LINE__,
                       "config must be non-null with capacity > 0");
        return nullptr;
    }
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count == 0) {
        nbx::set_error(error, N_BODY_SIM_PRO_STATUS_UNSUPPORTED_PLATFORM, __FILE__, __LINE__,
                       "no HIP device is visible");
        return nullptr;
    }
    if (config->device < 0 || config->device >= count) {
        nbx::set_error(error, N_BODY_SIM_PRO_STATUS_INVALID_ARGUMENT, __FILE__, __LINE__,
                       "device ordinal out of range");
        return nullptr;
    }
    NBXEngine* engine = new (std::nothrow) NBXEngine();
    if (engine == nullptr) {
        nbx::set_error(error, N_BODY_SIM_PRO_STATUS_OUT_OF_MEMORY, __FILE__, __LINE__,
                       "engine allocation failed");
        return nullptr;
    }
    Engine* e = &engine->e;
    e->device = config->device;
    e->capacity = config->capacity;
    e->theta = config->theta > 0.0 ? config->theta : 0.7;
    e->flags = config->flags;
    bool ok = hipSetDevice(e->device) == hipSuccess &&
              hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking) == hipSuccess;
    int cus = 0;
    if (ok && hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, e->device) ==
                  hipSuccess &&
        cus > 0) {
        e->cu_count = cus;
    }
    int khz = 0;
    if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, e->device) == hipSuccess &&
        khz > 0) {
        e->clock_khz = khz;
    }
    double** arrays[] = {&e->px, &e->py, &e->pz, &e->vx, &e->vy, &e->vz,
                         &e->ax, &e->ay, &e->az, &e->m};
    for (double** a : arrays) {
        ok = ok && hipMalloc(reinterpret_cast<void**>(a), e->capacity * sizeof(double)) == hipSuccess;
    }
    ok = ok && hipMalloc(reinterpret_cast<void**>(&e->pos4), e->capacity * sizeof(float4)) == hipSuccess;
    for (auto& ev : e->ev) {
        ok = ok && hipEventCreate(&ev) == hipSuccess;
    }
    ok = ok && nbx::pinned_report(e);
    if (!ok) {
        nbx::set_error(error, N_BODY_SIM_PRO_STATUS_OUT_OF_MEMORY, __FILE__, __LINE__,
                       "device allocation failed while creating the engine");
        nbx_engine_destroy(engine);
        return nullptr;
    }
    return engine;
}

void nbx_mlp_release(void* mlp);

void nbx_engine_destroy(NBXEngine* engine) {
    if (engine == nullptr) {
        return;
    }
    Engine* e = &engine->e;
    (void)hipSetDevice(e->device);
    if (e->stream != nullptr) {
        (void)hipStreamSynchronize(e->stream);
    }
    double* arrays[] = {e->px, e->py, e->pz, e->vx, e->vy, e->vz, e->ax, e->ay, e->az, e->m};
    for (double* a : arrays) {
        if (a != nullptr) (void)hipFree(a);
    }
    if (e->pos4 != nullptr) (void)hipFree(e->pos4);
    for (nbx::Buf* b : nbx::work_buffers(e)) {
        nbx::free_buf(*b);
    }
    if (e->stage != nullptr && !e->stage_in_report) (void)hipHostFree(e->stage);
    if (e->bh.report != nullptr) (void)hipHostFree(e->bh.report);
    if (e->mlp != nullptr) {
        nbx_mlp_release(e->mlp);
    }
    for (auto& ev : e->ev) {
        if (ev != nullptr) (void)hipEventDestroy(ev);
    }
    if (e->stream != nullptr) (void)hipStreamDestroy(e->stream);
    delete engine;
}

size_t nbx_engine_device_bytes(const NBXEngine* engine) {
    if (engine == nullptr) {
        return 0;
    }
    Engine* e = const_cast<Engine*>(&engine->e);
    size_t bytes = e->capacity * (10 * sizeof(double) + sizeof(float4));
    for (const nbx::Buf* b : nbx::work_buffers(e)) {
        bytes += b->cap;
    }
    return bytes;
}

void nbx_engine_set_theta(NBXEngine* engine, double theta) {
    if (engine != nullptr) {
        engine->e.theta = theta;
    }
}

double nbx_engine_theta(const NBXEngine* engine) {
    return engine == nullptr ? 0.0 : engine->e.theta;
}

// wait: the view's values have reached the device on return; else the
// caller waits for the stream before the next transfer.
static NBodySimProStatus upload(NBXEngine* engine, const NBodySimProParticleSystemView* view,
                                bool wait, NBodySimProError* error) {
    NBX_TRY(nbx::check_engine(engine, error));
    if (view == nullptr) {
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_ARGUMENT, "view must not be null");
    }
    Engine* e = &engine->e;
    const size_t n = view->particle_count;
    if (n > e->capacity) {
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INSUFFICIENT_MEMORY,
                 "particle count exceeds the engine capacity");
    }
    if (n > 0 && (view->positions_x == nullptr || view->positions_y == nullptr ||
                  view->positions_z == nullptr || view->masses == nullptr)) {
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_ARGUMENT, "view positions/masses are null");
    }
    nbx::ArrayList list;
    list.add(view->positions_x, e->px);
    list.add(view->positions_y, e->py);
    list.add(view->positions_z, e->pz);
    list.add(view->masses, e->m);
    list.add(view->velocities_x, e->vx);
    list.add(view->velocities_y, e->vy);
    list.add(view->velocities_z, e->vz);
    list.add(view->accelerations_x, e->ax);
    list.add(view->accelerations_y, e->ay);
    list.add(view->accelerations_z, e->az);
    bool enqueued = false;
    NBX_TRY(nbx::copy_in(e, list, n, &enqueued, error));
    if (enqueued && wait) {
        NBX_HIP(error, hipStreamSynchronize(e->stream));
    }
    e->n = n;
    e->pos4_valid = false;
    return N_BODY_SIM_PRO_STATUS_OK;
}

NBodySimProStatus nbx_engine_upload(NBXEngine* engine, const NBodySimProParticleSystemView* view,
                                    NBodySimProError* error) {
    return upload(engine, view, true, error);
}

size_t nbx_engine_particle_count(const NBXEngine* engine) {
    return engine != nullptr ? engine->e.n : 0;
}

size_t nbx_engine_capacity(const NBXEngine* engine) {
    return engine != nullptr ? engine->e.capacity : 0;
}

NBodySimProStatus nbx_engine_download(NBXEngine* engine, const NBodySimProParticleSystemView* view,
                                      NBodySimProError* error) {
    NBX_TRY(nbx::check_engine(engine, error));
    if (view == nullptr) {
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_ARGUMENT, "view must not be null");
    }
    Engine* e = &engine->e;
    if (view->particle_count != e->n) {
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_ARGUMENT,
                 "view particle count differs from the uploaded count");
    }
    nbx::ArrayList list;
    list.add(view->positions_x, e->px);
    list.add(view->positions_y, e->py);
    list.add(view->positions_z, e->pz);
    list.add(view->masses, e->m);
    list.add(view->velocities_x, e->vx);
    list.add(view->velocities_y, e->vy);
    list.add(view->velocities_z, e->vz);
    list.add(view->accelerations_x, e->ax);
    list.add(view->accelerations_y, e->ay);
    list.add(view->accelerations_z, e->az);
    return nbx::copy_out(e, list, e->n, error);
}

NBodySimProStatus nbx_engine_compute_force(NBXEngine* engine, NBXAlgorithm algorithm,
                                           const NBodySimProGravity* gravity,
                                           NBodySimProError* error) {
    NBX_TRY(nbx::check_engine(engine, error));
    if (gravity == nullptr) {
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_ARGUMENT, "gravity must not be null");
    }
    NBX_TRY(nbx::compute_force(&engine->e, algorithm, gravity, error));
    return nbx::direct_timings(&engine->e, error);
}

NBodySimProStatus nbx_engine_advance(NBXEngine* engine, NBXAlgorithm algorithm,
                                     const NBodySimProGravity* gravity,
                                     NBodySimProIntegratorType integrator, double timestep,
                                     int steps, NBodySimProError* error) {
    NBX_TRY(nbx::check_engine(engine, error));
    if (gravity == nullptr) {
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_ARGUMENT, "gravity must not be null");
    }
    if (!(timestep > 0.0)) {
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_ARGUMENT, "timestep must be positive");
    }
    if (steps < 0) {
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_ARGUMENT, "steps must be non-negative");
    }
    if (integrator != N_BODY_SIM_PRO_INTEGRATOR_EULER &&
        integrator != N_BODY_SIM_PRO_INTEGRATOR_LEAPFROG &&
        integrator != N_BODY_SIM_PRO_INTEGRATOR_VELOCITY_VERLET) {
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_ARGUMENT, "unknown integrator type");
    }
    Engine* e = &engine->e;
    const int n = static_cast<int>(e->n);
    if (n == 0) {
        return N_BODY_SIM_PRO_STATUS_OK;
    }
    hipEvent_t t0, t1;
    NBX_HIP(error, hipEventCreate(&t0));
    NBX_HIP(error, hipEventCreate(&t1));
    NBX_HIP(error, hipEventRecord(t0, e->stream));
    const unsigned g = nbx::grid_for(e->n, nbx::kThreads);
    const double half = 0.5 * timestep;
    NBodySimProStatus st = N_BODY_SIM_PRO_STATUS_OK;
    auto launched = [&]() {
        if (hipGetLastError() != hipSuccess) {
            nbx::set_error(error, N_BODY_SIM_PRO_STATUS_INVALID_STATE, __FILE__, __LINE__,
                           "integrator kernel launch failed");
            st = N_BODY_SIM_PRO_STATUS_INVALID_STATE;
        }
        return st == N_BODY_SIM_PRO_STATUS_OK;
    };
    auto kick_drift = [&](int k, nbx::EvaluationGate gate) {
        if (k == 0) {
            nbx::kick_drift_kernel<<<g, nbx::kThreads, 0, e->stream>>>(
                e->px, e->py, e->pz, e->vx, e->vy, e->vz, e->ax, e->ay, e->az, n, half, timestep);
        } else {   // the previous step's closing kick rides along
            nbx::kick_kick_drift_kernel<<<g, nbx::kThreads, 0, e->stream>>>(
                e->px, e->py, e->pz, e->vx, e->vy, e->vz, e->ax, e->ay, e->az, n, half, timestep,
                gate);
        }
        e->pos4_valid = false;
        return launched();
    };
    auto euler = [&]() {
        for (int k = 0; k < steps; ++k) {
            e->timed = k + 1 == steps;   // the timings tell of the last evaluation
            st = nbx::compute_force(e, algorithm, gravity, error);
            if (st != N_BODY_SIM_PRO_STATUS_OK) return;
            nbx::euler_kernel<<<g, nbx::kThreads, 0, e->stream>>>(e->px, e->py, e->pz, e->vx, e->vy,
                                                                  e->vz, e->ax, e->ay, e->az, n,
                                                                  timestep, nbx::direct_end(e));
            e->pos4_valid = false;
            if (!launched()) return;
        }
    };
    auto leapfrog = [&]() {
        for (int k = 0; k < steps; ++k) {
            if (!kick_drift(k, {nullptr, nullptr})) return;
            e->timed = k + 1 == steps;
            st = nbx::compute_force(e, algorithm, gravity, error);
            if (st != N_BODY_SIM_PRO_STATUS_OK) return;
        }
    };
    // Barnes-Hut: a step is enqueued while the one before it runs, so that the
    // stream does not stand still while the host reads its report. Where that
    // evaluation turns out to need the host (a repair of the tree, a
    // per-query walk), the kick behind it has not moved anything, the
    // evaluation behind that is the same one again, and the host completes
    // it; until one goes without the host again, none is run ahead of.
    // (20 steps with a snapshot, each evaluation read before the next was
    // enqueued / run ahead: 10,000 particles 3.46 / 3.20 ms, 1M 23.9 / 23.8.)
    auto leapfrog_ahead = [&]() {
        const bool fp64 = algorithm == NBX_ALGORITHM_BARNES_HUT_FP64;
        bool ahead = false;   // the last evaluation enqueued has not been read
        int slot = 0;
        int k = 0;
        while (k < steps) {
            if (!kick_drift(k, ahead ? nbx::bh_gate(e) : nbx::EvaluationGate{nullptr, nullptr})) {
                return;
            }
            slot ^= 1;
            st = nbx::bh_enqueue(e, gravity, fp64, slot, error);
            if (st != N_BODY_SIM_PRO_STATUS_OK) return;
            bool repeated = false;
            if (ahead) {
                bool clean = false;
                st = nbx::bh_peek(e, slot ^ 1, &clean, error);
                if (st != N_BODY_SIM_PRO_STATUS_OK) return;
                repeated = !clean;
            }
            if (!repeated) {
                ++k;
            }
            ahead = !repeated && k < steps && e->bh.clean;
            if (!ahead) {
                st = nbx::bh_end(e, gravity, fp64, slot, error);
                if (st != N_BODY_SIM_PRO_STATUS_OK) return;
            }
        }
    };
    if (integrator == N_BODY_SIM_PRO_INTEGRATOR_EULER) {
        euler();
    } else {
        if (nbx::bh_runs_ahead(e, algorithm)) {
            leapfrog_ahead();
        } else {
            leapfrog();
        }
        if (st == N_BODY_SIM_PRO_STATUS_OK && steps > 0) {
            nbx::kick_kernel<<<g, nbx::kThreads, 0, e->stream>>>(e->vx, e->vy, e->vz, e->ax, e->ay,
                                                                 e->az, n, half, nbx::direct_end(e));
            (void)launched();
        }
    }
    e->timed = true;
    hipError_t done = hipEventRecord(t1, e->stream);
    const hipError_t waited = hipEventSynchronize(t1);
    done = done != hipSuccess ? done : waited;
    float ms = 0.f;
    (void)hipEventElapsedTime(&ms, t0, t1);
    (void)hipEventDestroy(t0);
    (void)hipEventDestroy(t1);
    if (st == N_BODY_SIM_PRO_STATUS_OK) {
        NBX_HIP(error, done);   // all-pairs steps were not waited for before
        st = nbx::direct_timings(e, error);
    }
    e->timings.integrate_ms = ms;
    return st;
}

NBodySimProStatus nbx_engine_diagnostics(NBXEngine* engine, const NBodySimProGravity* gravity,
                                         NBodySimProDiagnosticsQuantities* q, double* potential,
                                         NBodySimProError* error) {
    NBX_TRY(nbx::check_engine(engine, error));
    if (q == nullptr || (potential != nullptr && gravity == nullptr)) {
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_ARGUMENT,
                 "quantities (and gravity when a potential is requested) must not be null");
    }
    Engine* e = &engine->e;
    const int n = static_cast<int>(e->n);
    const unsigned blocks = n == 0 ? 1u : (nbx::grid_for(e->n, nbx::kThreads) < 512u
                                               ? nbx::grid_for(e->n, nbx::kThreads) : 512u);
    const int64_t units = nbx::pot_units_before((n + nbx::kWave - 1) / nbx::kWave,
                                                (n + nbx::kPotSources - 1) / nbx::kPotSources);
    const unsigned pblocks = nbx::grid_for(
        static_cast<size_t>(std::max<int64_t>(1, std::min(units, nbx::kPotMaxWaves))),
        nbx::kPotWaves);
    NBX_TRY(e->scratch.need<double>(blocks * nbx::kDiag + pblocks + 16, error));
    double* part = e->scratch.as<double>();
    double* pot = part + blocks * nbx::kDiag;
    double* out = pot + pblocks;
    double sums[nbx::kDiag + 1];
    nbx::diag_partial_kernel<<<blocks, nbx::kThreads, 0, e->stream>>>(
        e->px, e->py, e->pz, e->vx, e->vy, e->vz, e->m, n, part);
    if (potential != nullptr) {
        nbx::potential_partial_kernel<<<pblocks, nbx::kThreads, 0, e->stream>>>(
            e->px, e->py, e->pz, e->m, n, gravity->softening_squared, units, pot);
    }
    const unsigned columns = nbx::kDiag + (potential != nullptr ? 1u : 0u);
    nbx::reduce_rows_kernel<<<columns, nbx::kThreads, 0, e->stream>>>(
        part, static_cast<int>(blocks), pot, static_cast<int>(pblocks), out);
    NBX_HIP(error, hipGetLastError());
    NBX_HIP(error, hipMemcpyAsync(sums, out, columns * sizeof(double), hipMemcpyDeviceToHost,
                                  e->stream));
    NBX_HIP(error, hipStreamSynchronize(e->stream));
    q->kinetic_energy = sums[0];
    q->total_mass = sums[1];
    q->total_momentum_x = sums[2];
    q->total_momentum_y = sums[3];
    q->total_momentum_z = sums[4];
    q->total_angular_momentum_x = sums[5];
    q->total_angular_momentum_y = sums[6];
    q->total_angular_momentum_z = sums[7];
    if (sums[1] != 0.0) {
        q->center_of_mass_x = sums[8] / sums[1];
        q->center_of_mass_y = sums[9] / sums[1];
        q->center_of_mass_z = sums[10] / sums[1];
    } else {
        q->center_of_mass_x = q->center_of_mass_y = q->center_of_mass_z = 0.0;
    }
    if (potential != nullptr) {
        *potential = -gravity->gravitational_constant * sums[nbx::kDiag];
    }
    return N_BODY_SIM_PRO_STATUS_OK;
}

int nbx_engine_stats(const NBXEngine* engine, NBodySimProBarnesHutStats* stats) {
    if (engine == nullptr || stats == nullptr) {
        return 1;
    }
    *stats = engine->e.stats;
    return 0;
}

int nbx_engine_timings(const NBXEngine* engine, NBXTimings* timings) {
    if (engine == nullptr || timings == nullptr) {
        return 1;
    }
    *timings = engine->e.timings;
    return 0;
}

NBodySimProStatus nbx_engine_bh_morton(NBXEngine* engine, double* root, uint64_t* keys,
                                       int64_t* permutation, NBodySimProError* error) {
    NBX_TRY(nbx::check_engine(engine, error));
    Engine* e = &engine->e;
    const size_t n = e->bh.n;
    if (n == 0) {
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_STATE, "no Barnes-Hut build to report");
    }
    if (root != nullptr) {
        for (int k = 0; k < 4; ++k) root[k] = e->bh.root[k];
    }
    if (keys != nullptr || permutation != nullptr) {
        NBX_TRY(nbx::bh_morton_order(e, error));
    }
    if (keys != nullptr) {
        NBX_HIP(error, hipMemcpy(keys, e->bh.mkey.p, n * sizeof(uint64_t), hipMemcpyDeviceToHost));
    }
    if (permutation != nullptr) {
        std::vector<uint32_t> p(n);
        NBX_HIP(error, hipMemcpy(p.data(), e->bh.mperm.p, n * sizeof(uint32_t), hipMemcpyDeviceToHost));
        for (size_t i = 0; i < n; ++i) permutation[i] = static_cast<int64_t>(p[i]);
    }
    return N_BODY_SIM_PRO_STATUS_OK;
}

NBodySimProStatus nbx_engine_bh_export_nodes(NBXEngine* engine, double* rows,
                                             NBodySimProError* error) {
    NBX_TRY(nbx::check_engine(engine, error));
    Engine* e = &engine->e;
    nbx::BHState& s = e->bh;
    if (s.n == 0 || rows == nullptr) {
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_STATE, "no Barnes-Hut build to export");
    }
    const size_t n = s.n, nodes = s.nodes, internal = s.internal;
    std::vector<double> cx(nodes), cy(nodes), cz(nodes), m(nodes);
    std::vector<int32_t> depth(nodes), start(nodes), count(nodes), leaf(nodes);
    std::vector<uint64_t> word(n), ext;
    std::vector<uint32_t> trank(n);
    {
        // internal nodes: records by internal id, placed at their node index
        std::vector<double> com(4 * internal);
        std::vector<int32_t> rec(4 * internal), idepth(internal);
        NBX_HIP(error, hipMemcpy(com.data(), s.icom.p, internal * 32, hipMemcpyDeviceToHost));
        NBX_HIP(error, hipMemcpy(rec.data(), s.irec.p, internal * 16, hipMemcpyDeviceToHost));
        NBX_HIP(error, hipMemcpy(idepth.data(), s.idepth.p, internal * 4, hipMemcpyDeviceToHost));
        for (size_t i = 0; i < internal; ++i) {
            const size_t k = static_cast<size_t>(rec[4 * i]);
            cx[k] = com[4 * i];
            cy[k] = com[4 * i + 1];
            cz[k] = com[4 * i + 2];
            m[k] = com[4 * i + 3];
            depth[k] = idepth[i];
            start[k] = rec[4 * i + 2];
            count[k] = rec[4 * i + 3] - rec[4 * i + 2] + 1;   // last - first + 1
        }
    }
    {
        NBX_TRY(nbx::bh_node_records(e, error));
        NBX_HIP(error, hipStreamSynchronize(e->stream));
        std::vector<nbx::NodeF32> recs(nodes);
        NBX_HIP(error, hipMemcpy(recs.data(), s.n32.p, nodes * sizeof(nbx::NodeF32),
                                 hipMemcpyDeviceToHost));
        for (size_t k = 0; k < nodes; ++k) leaf[k] = recs[k].leaf;
    }
    NBX_HIP(error, hipMemcpy(word.data(), s.tword.p, n * 8, hipMemcpyDeviceToHost));
    {
        // Morton rank of each tree position's particle
        NBX_TRY(nbx::bh_morton_order(e, error));
        std::vector<uint32_t> mperm(n), tperm(n), rank(n);
        NBX_HIP(error, hipMemcpy(mperm.data(), s.mperm.p, n * 4, hipMemcpyDeviceToHost));
        NBX_HIP(error, hipMemcpy(tperm.data(), s.tperm.p, n * 4, hipMemcpyDeviceToHost));
        for (size_t k = 0; k < n; ++k) rank[mperm[k]] = static_cast<uint32_t>(k);
        for (size_t k = 0; k < n; ++k) trank[k] = rank[tperm[k]];
    }
    // A leaf's row comes from its tree position t: depth one below the deeper
    // neighbour cell, the particle itself as mass and centre of mass.
    std::vector<int32_t> delta(n);
    std::vector<double> sp(4 * n);
    NBX_HIP(error, hipMemcpy(delta.data(), s.delta.p, n * 4, hipMemcpyDeviceToHost));
    if (s.inputs_fp64) {
        NBX_HIP(error, hipMemcpy(sp.data(), s.sp4.p, n * 32, hipMemcpyDeviceToHost));
    } else {
        // FP32 inputs: the tree-order float4 values, widened exactly
        std::vector<float> sf(4 * n);
        NBX_HIP(error, hipMemcpy(sf.data(), s.s4.p, n * 16, hipMemcpyDeviceToHost));
        for (size_t k = 0; k < 4 * n; ++k) sp[k] = static_cast<double>(sf[k]);
    }
    for (size_t k = 0; k < nodes; ++k) {
        const int t = leaf[k];
        if (t < 0) {
            continue;
        }
        const int a = t > 0 ? delta[t - 1] : -1;
        depth[k] = 1 + (a > delta[t] ? a : delta[t]);
        start[k] = t;
        count[k] = 1;
        cx[k] = sp[4 * t];
        cy[k] = sp[4 * t + 1];
        cz[k] = sp[4 * t + 2];
        m[k] = sp[4 * t + 3];
    }
    std::vector<uint32_t> slot;
    if (s.ext_tree != nullptr) {
        ext.resize((s.ext_slot != nullptr ? s.ext_slots : n) * 6);
        NBX_HIP(error, hipMemcpy(ext.data(), s.ext_tree, ext.size() * 8, hipMemcpyDeviceToHost));
    }
    if (s.ext_slot != nullptr) {
        slot.resize(n);
        NBX_HIP(error, hipMemcpy(slot.data(), s.ext_slot, n * 4, hipMemcpyDeviceToHost));
    }
    for (size_t k = 0; k < nodes; ++k) {
        // Replay the cell centre from the root along the node's octant path
        // with the reference's FP64 operations (barnes_hut.c:202-211).
        double c[3] = {s.root[0], s.root[1], s.root[2]};
        double h = s.root[3];
        const int t = start[k];
        for (int d = 0; d < depth[k]; ++d) {
            const size_t at = d < 21 || slot.empty() ? static_cast<size_t>(t) : slot[t];
            uint64_t w = d < 21 ? word[t] : ext[at * 6 + (d / 21 - 1)];
            const int o = static_cast<int>((w >> (60 - 3 * (d % 21))) & 7u);
            const double off = h * 0.5;
            c[0] = c[0] + ((o & 1) ? off : -off);
            c[1] = c[1] + ((o & 2) ? off : -off);
            c[2] = c[2] + ((o & 4) ? off : -off);
            h = 0.5 * h;
        }
        double* r = rows + 11 * k;
        r[0] = depth[k];
        r[1] = c[0];
        r[2] = c[1];
        r[3] = c[2];
        r[4] = h;
        r[5] = count[k];
        r[6] = m[k];
        r[7] = cx[k];
        r[8] = cy[k];
        r[9] = cz[k];
        r[10] = leaf[k] >= 0 ? static_cast<double>(trank[leaf[k]]) : -1.0;
    }
    return N_BODY_SIM_PRO_STATUS_OK;
}

static NBodySimProStatus dropin(const NBodySimProParticleSystemView* view,
                                const NBodySimProGravity* gravity, void* context,
                                NBodySimProError* error, NBXAlgorithm algorithm) {
    if (view == nullptr || gravity == nullptr) {
        NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_ARGUMENT,
                 "view and gravity parameters must not be null");
    }
    const size_t n = view->particle_count;
    if (n == 0) {
        if (algorithm == NBX_ALGORITHM_BARNES_HUT || algorithm == NBX_ALGORITHM_BARNES_HUT_FP64 ||
            algorithm == NBX_ALGORITHM_BH_LEARNED) {
            NBX_FAIL(error, N_BODY_SIM_PRO_STATUS_INVALID_ARGUMENT,
                     "cannot build a Barnes-Hut tree for an empty system");
        }
        return N_BODY_SIM_PRO_STATUS_OK;
    }
    std::unique_lock<std::mutex> lock(nbx::g_default_mutex, std::defer_lock);
    NBXEngine* engine = static_cast<NBXEngine*>(context);
    if (engine == nullptr) {
        lock.lock();
        if (nbx::g_default != nullptr && nbx::g_default->e.capacity < n) {
            nbx_engine_destroy(nbx::g_default);
            nbx::g_default = nullptr;
        }
        if (nbx::g_default == nullptr) {
            NBXConfig cfg{n, 0, 0.7, 0u};
            nbx::g_default = nbx_engine_create(&cfg, error);
            if (nbx::g_default == nullptr) {
                return error != nullptr ? error->status : N_BODY_SIM_PRO_STATUS_INVALID_STATE;
            }
        }
        engine = nbx::g_default;
    }
    NBodySimProParticleSystemView in{};
    in.particle_count = n;
    in.positions_x = view->positions_x;
    in.positions_y = view->positions_y;
    in.positions_z = view->positions_z;
    in.masses = view->masses;
    NBX_TRY(upload(engine, &in, false, error));
    const NBodySimProStatus st = nbx::compute_force(&engine->e, algorithm, gravity, error);
    if (st != N_BODY_SIM_PRO_STATUS_OK) {
        (void)hipStreamSynchronize(engine->e.stream);   // the pinned block is free again
        return st;
    }
    NBodySimProParticleSystemView out{};
    out.particle_count = n;
    out.accelerations_x = view->accelerations_x;
    out.accelerations_y = view->accelerations_y;
    out.accelerations_z = view->accelerations_z;
    NBX_TRY(nbx_engine_download(engine, &out, error));
    return nbx::direct_timings(&engine->e, error);
}

NBodySimProStatus nbx_hip_direct_fp64(const NBodySimProParticleSystemView* view,
                                      const NBodySimProGravity* gravity, void* context,
                                      NBodySimProError* error) {
    return dropin(view, gravity, context, error, NBX_ALGORITHM_DIRECT_FP64);
}

NBodySimProStatus nbx_hip_direct_fp32(const NBodySimProParticleSystemView* view,
                                      const NBodySimProGravity* gravity, void* context,
                                      NBodySimProError* error) {
    return dropin(view, gravity, context, error, NBX_ALGORITHM_DIRECT_FP32);
}

NBodySimProStatus nbx_hip_barnes_hut(const NBodySimProParticleSystemView* view,
                                     const NBodySimProGravity* gravity, void* context,
                                     NBodySimProError* error) {
    return dropin(view, gravity, context, error, NBX_ALGORITHM_BARNES_HUT);
}

NBodySimProStatus nbx_hip_barnes_hut_fp64(const NBodySimProParticleSystemView* view,
                                          const NBodySimProGravity* gravity, void* context,
                                          NBodySimProError* error) {
    return dropin(view, gravity, context, error, NBX_ALGORITHM_BARNES_HUT_FP64);
}

NBodySimProStatus nbx_hip_bh_learned(const NBodySimProParticleSystemView* view,
                                     const NBodySimProGravity* gravity, void* context,
                                     NBodySimProError* error) {
    return dropin(view, gravity, context, error, NBX_ALGORITHM_BH_LEARNED);
}

}  // extern "C"
