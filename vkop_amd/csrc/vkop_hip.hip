// C ABI of the softmax / top-k library (declared in include/vkop_hip.h):
// argument checking, kernel selection and launches (the only kernel here clears a workspace).
#include "../../include/vkop_hip.h"
#include "vkop_hip_internal.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "kernels_general.hpp"
#include "kernels_rows.hpp"
#include "rows_launch.hpp"
#include "kernels_joined.hpp"
#include "kernels_softmax.hpp"
#include "kernels_bigk.hpp"
#include "kernels_nms.hpp"

namespace vkop {

// workspace clear (a kernel, not a memset: safe inside a captured graph)
__global__ void fill_zero_kernel(uint32_t *p, size_t words) {
    const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < words) p[i] = 0u;
}

}  // namespace vkop

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof g_err, fmt, ap);
    va_end(ap);
    return code;
}

#define VKOP_HIP_TRY(expr)                                                                        \
    do {                                                                                          \
        hipError_t e_ = (expr);                                                                   \
        if (e_ != hipSuccess) return fail(VKOP_HIP_ERR_DEVICE, "%s: %s", #expr, hipGetErrorString(e_)); \
    } while (0)

inline hipStream_t as_stream(void *s) { return static_cast<hipStream_t>(s); }

// (outer, n, inner) view of a dense tensor around `axis`.
struct View {
    vkop::LineGeom g;
    uint64_t elems;
};

int make_view(const int *shape, int ndim, int axis, View *v) {
    if (shape == nullptr) return fail(VKOP_HIP_ERR_INVALID, "shape is null");
    if (ndim < 1 || ndim > 4) return fail(VKOP_HIP_ERR_INVALID, "rank %d outside 1..4", ndim);
    if (axis < 0) axis += ndim;
    if (axis < 0 || axis >= ndim) return fail(VKOP_HIP_ERR_INVALID, "axis outside the tensor's rank %d", ndim);
    uint64_t outer = 1, inner = 1;
    for (int d = 0; d < ndim; d++) {
        if (shape[d] < 0) return fail(VKOP_HIP_ERR_INVALID, "negative extent %d at dim %d", shape[d], d);
        if (d < axis) outer *= static_cast<uint64_t>(shape[d]);
        if (d > axis) inner *= static_cast<uint64_t>(shape[d]);
    }
    const uint64_t n = static_cast<uint64_t>(shape[axis]);
    const uint64_t elems = outer * n * inner;
    if (outer * inner >= (1ull << 31) || elems >= (1ull << 40))
        return fail(VKOP_HIP_ERR_UNSUPPORTED, "tensor too large (%llu elements)", static_cast<unsigned long long>(elems));
    v->g.outer = static_cast<uint32_t>(outer);
    v->g.n = static_cast<uint32_t>(n);
    v->g.inner = static_cast<uint32_t>(inner);
    v->elems = elems;
    return VKOP_HIP_OK;
}

int check_dtype(int dtype) {
    if (dtype != VKOP_HIP_F32 && dtype != VKOP_HIP_F16) return fail(VKOP_HIP_ERR_INVALID, "unknown dtype %d", dtype);
    return VKOP_HIP_OK;
}

int check_k(const View &v, int k) {
    if (k < 1) return fail(VKOP_HIP_ERR_INVALID, "k = %d must be at least 1", k);
    if (static_cast<uint64_t>(k) > v.g.n)
        return fail(VKOP_HIP_ERR_INVALID, "k = %d exceeds the axis extent %u", k, v.g.n);
    if (k > VKOP_HIP_MAX_K) return fail(VKOP_HIP_ERR_UNSUPPORTED, "k = %d exceeds VKOP_HIP_MAX_K = %d", k, VKOP_HIP_MAX_K);
    return VKOP_HIP_OK;
}

int launched(const char *what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(VKOP_HIP_ERR_DEVICE, "launch of %s failed: %s", what, hipGetErrorString(e));
    return VKOP_HIP_OK;
}

// ---- scratch of the entry point that allocates nothing ------------------------
// One array per GPU, created when the library's code is loaded on that GPU and
// held until the process ends.  In host code the array's name is only a handle:
// its device address is looked up once per device (resolve_static_scratch) and
// that address is what kernels, fills and copies are given.
static __device__ __align__(256) unsigned char scratch[VKOP_HIP_STATIC_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;
std::atomic<void *> g_scratch_ptr[kMaxDevices];
// set when a call on the static scratch may have left a row's arrival counter
// non-zero (a launch failed half way): the next call clears the counters first
std::atomic<int> g_scratch_dirty[kMaxDevices];

// Device address of `scratch` on the current device (looked up on the first call
// per device, with that device current), and the device's ordinal.
int resolve_static_scratch(void **ptr, int *device) {
    int dev = 0;
    VKOP_HIP_TRY(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return fail(VKOP_HIP_ERR_UNSUPPORTED, "device ordinal %d beyond %d", dev, kMaxDevices);
    void *p = g_scratch_ptr[dev].load(std::memory_order_acquire);
    if (p == nullptr) {
        VKOP_HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (p == nullptr) return fail(VKOP_HIP_ERR_DEVICE, "hipGetSymbolAddress gave no address for the static scratch");
        g_scratch_ptr[dev].store(p, std::memory_order_release);
    }
    *ptr = p;
    *device = dev;
    return VKOP_HIP_OK;
}

// vkop_hip_tune state
std::atomic<int> g_rows_threads{0}, g_rows_loads{0}, g_rows_chunks{0}, g_rows_fused{0}, g_rows_path{0},
    g_nms_threads{0};
// Which kernels of a two-kernel streaming call are launched: both, except in the benchmark build of the
// library (-DVKOP_BENCH_HOOKS, libvkop_hip_bench.so), where vkop_hip_measure_stages can leave one out.
#ifdef VKOP_BENCH_HOOKS
std::atomic<int> g_rows_stages{3};
inline int measured_stages() { return g_rows_stages.load(); }
std::atomic<uint32_t> g_joined_polls{100};
inline uint32_t joined_polls() { return g_joined_polls.load(); }
inline uint32_t nms_polls() { return g_joined_polls.load() * 40u; }
#else
inline int measured_stages() { return 3; }
// How often a workgroup of softmax_joined_kernel looks for its row's other chunks before it reads what it misses: a look takes
// about a microsecond, the wait for a row whose workgroups run a few of them.
constexpr uint32_t joined_polls() { return 100; }
// The same of nms_kernel, whose pairs take from 6 to 700 us.
constexpr uint32_t nms_polls() { return 4000; }
#endif
// (what tells the records of a call of softmax_joined_kernel from whatever the workspace held before)
std::atomic<uint32_t> g_joined_calls{0};

// The per-row arrival counters of the one-kernel top-k variant sit at a fixed
// place, the first kTicketRows words of every workspace, whatever the operator
// and tensor: each call leaves them at zero, so a workspace cleared once can
// serve calls of different kinds and shapes in turn.  Nothing else is ever
// stored there.
constexpr size_t kTicketRows = 16384;
constexpr size_t kTicketBytes = kTicketRows * sizeof(uint32_t);  // a multiple of the workspace alignment

constexpr int kLineThreads = 256;
constexpr size_t kAlign = 256;
inline size_t align_up(size_t b) { return (b + kAlign - 1) / kAlign * kAlign; }

// ---------------------------------------------------------------- softmax ----
// Threads per workgroup and 128-bit loads per thread.
struct RowShape {
    int nt, v;
};

// HIP takes no grid of 2^32 threads or more: launch(first, count) for as many of `units` -- rows, or blocks of them -- at a
// time as stay below that, the last workgroup's idle threads among them (all units in every case but tensors of tens of gigabytes).
template <typename F> int in_slices(uint64_t units, uint64_t threads_per_unit, F &&launch) {
    constexpr uint64_t kGridThreads = 0xFFFFFFFFull - 1024;
    const uint64_t most = std::max<uint64_t>(1, kGridThreads / threads_per_unit);
    for (uint64_t first = 0; first < units; first += most)
        if (const int rc = launch(first, static_cast<uint32_t>(std::min(most, units - first)))) return rc;
    return VKOP_HIP_OK;
}

struct SoftmaxPlan {
    enum Kind { kGeneralLines, kGeneralStrided, kThread, kGroup, kRow, kChunked, kLinesRegs, kStridedRegs, kStridedTile } kind = kGeneralLines;
    RowShape shape{0, 0};  // kChunked; kGroup: lanes a row and vectors a lane; kRow: threads and vectors a thread
    uint32_t g = 1, per = 0;
    bool joined = false;  // kChunked: in one launch where the tensors allow it (joined_fits)
    uint32_t lines_k = 0, lines_p = 0, lines_w = 0;  // kLinesRegs: LinesLaunch
    uint32_t ti_shift = 0;  // kStridedTile: log2 of the lines a tile
    size_t workspace = 0;
    size_t pair_workspace = 0;  // kChunked: what the pair of kernels needs, at most `workspace`
};

// Lines of up to kStridedMaxN elements along a non-last axis, held in registers: the
// kernel is compiled for a few bounds of n and the smallest that fits is launched;
// longer lines are shared by two or four lanes.
template <typename T, bool MAX_ONLY>
void launch_strided_reg(const T *in, T *out, const View &v, int nan_where, float nan_value, hipStream_t st) {
    const uint32_t lines = v.g.outer * v.g.inner;
#define VKOP_STRIDED_CASE(NMAX, P)                                                          \
    if (v.g.n <= NMAX) {                                                                    \
        const uint32_t per_block = vkop::kStridedThreads / P;                               \
        vkop::softmax_strided_reg_kernel<T, NMAX, P, MAX_ONLY>                              \
            <<<(lines + per_block - 1) / per_block, vkop::kStridedThreads, 0, st>>>(in, out, v.g, nan_where, nan_value); \
        return;                                                                             \
    }
    VKOP_STRIDED_CASE(16, 1)
    VKOP_STRIDED_CASE(32, 2)
    VKOP_STRIDED_CASE(48, 4)
    VKOP_STRIDED_CASE(64, 4)
    VKOP_STRIDED_CASE(80, 4)
    VKOP_STRIDED_CASE(96, 4)
    VKOP_STRIDED_CASE(128, 4)
#undef VKOP_STRIDED_CASE
}

// Threads that the register kernel for lines takes for one outer index.
uint64_t lines_threads(const View &v, uint32_t vec, uint32_t P, uint32_t W) {
    return static_cast<uint64_t>((v.g.inner + vec - 1) / vec) * P * W;
}

// The register kernel for lines along a non-last axis (kernels_lines.hpp) and its shape: lane groups of a
// wave a line (P), waves a line (W) and elements a lane (K).  False: the kernels of one element a load.
// us a call, those against this one: f32 [8,21,262144] 81.5 -> 66.3, [16,80,8400] max only 19.1 -> 15.1,
// [16,512,784] 28.6 -> 14.3, [8,1000,8000] 192 -> 113, [32,1000,64] 18.4 -> 10.0; f16 [8,21,262144] 49.9 ->
// 38.6, [2,512,3136] 20.9 -> 9.8, [8,200,65536] 179 -> 96.
bool plan_lines(const View &v, uint32_t vec, SoftmaxPlan *p) {
    const uint32_t n = v.g.n;
    if (v.g.inner < vec || n > vkop::kLinesMaxN) return false;
    const bool half = vec == 8;
    const uint64_t vectors = static_cast<uint64_t>(v.g.outer) * ((v.g.inner + vec - 1) / vec);
    // Short lines of few elements in all have too few lanes with 16 bytes each (f32 [1,4,65536] 3.1 against 3.2 us
    // here, [1,80,8400] 5.8 against 4.9).  Halves, twice as many lines a lane: [1,80,8400] 4.2 against 6.1,
    // [4,91,12345] 7.6 against 9.9, but [4,24,65536] 8.6 against 8.1, [8,48,65536] 30.4 against 22.5 and
    // [8,100,65536] 64 against 60; their lines of up to 16 never gain more than they lose ([8,16,262144] 26.9 / 28.3).
    // Halves' rows off 16 bytes, or off the cache lines, ask for more of them: [8,32,81921] 18.1 against 23.0, [8,64,40961]
    // 18.8 / 25.4, [8,48,54612] 18.4 / 22.2, but [8,32,131073] 36.3 / 31.9, [8,64,65537] 46.8 / 35.2.
    // (The largest probability alone takes the same kernel as the tensor, whose maximum it is bit for bit, whichever of the two
    // is the better one for it: [8,128,65536] 42.8 against 39.2, [8,65,129055] 49 / 55.)
    if (n <= 128) {
        if (v.elems < (1u << 19)) return false;
        if (half) {
            const bool off16 = v.g.inner % 8 != 0, off128 = v.g.inner % 64 != 0;
            const uint64_t least = n <= 32 ? (off16 && n > 20 ? 3ull << 23 : 5ull << 20) : n <= 64 ? (off128 ? 3ull << 23 : 1ull << 24) : 1ull << 25;
            if (n <= 16 || v.elems < least) return false;
        }
    } else if (vectors < 32) {  // ([1,1000,64] f16 10.2 against 11.9, f32 max only 8.3 against 9.2)
        return false;
    }
    // As many elements a lane as its registers hold (f32 16, f16 8: their 64 terms either way), and pieces of a row
    // of 128 bytes at least (P = 8) before a line takes several waves: a workgroup of many holds a CU on its
    // barriers ([8,1000,8000] f32 with P = 4 126, 8 113, 16 157 us).  With too few workgroups for the chip, more of
    // them: P = 16, half the lines ([32,1000,64] f32 13.0 -> 10.5, f16 17.5 -> 12.0).
    const uint32_t kmax = half ? 8 : 16, need = (n + kmax - 1) / kmax;
    uint32_t P = 1;
    while (P < 8 && P < need) P *= 2;
    if (half && n > 64 && n <= 128) P = 16;  // ([8,100,65536] max only: 36.1 us, with P = 8 41.8)
    if (n > 128 && vectors / 8 < (half ? 512u : 128u)) P = 16;
    uint32_t W = (need + P - 1) / P, K = (n + P * W - 1) / (P * W);
    // fewer than 512 waves: fewer elements a lane, while that is more than 4 and a line has at most 4 waves
    // ([1,80,8400] f32 6.3 -> 4.9, [1,200,1000] 8.2 -> 5.7; [32,777,65] f16 with 14 waves 14.7, with 7 12.6)
    while (K > 4 && W <= 4 && vectors * P * W < 512ull * vkop::kWave) {
        if (P < 16) P *= 2;
        else W *= 2;
        K = (n + P * W - 1) / (P * W);
    }
    if (lines_threads(v, vec, P, W) > 0xFFFFFFFFull - 1024) return false;  // (an outer index of 2^31 lines)
    p->kind = SoftmaxPlan::kLinesRegs;
    p->lines_k = K, p->lines_p = P, p->lines_w = W;
    return true;
}

// The shape of softmax_joined_kernel for rows of a tensor, false where the pair of kernels is the faster one: below 150 workgroups,
// and with a row in more chunks than 16, 20 of the narrow shape, or 8 of small ones and of fewer than 32 rows of halves -- every
// workgroup of a row reads the records of all, again and again until they are there.  us, the pair / this: f32
// [16,262144] 14.0 / 13.2 with 16 chunks, [16,65536] 7.8 / 8.0 with 8 in 128 workgroups, 9.1 with 16; [8,262144] 9.6 / 10.2 with
// 16, 10.7 with 32; [32,33001] 8.7 / 8.0; f16 [32,200000] 14.5 / 13.1, [32,65536] 8.4 / 7.8, [64,262144] 23.7 / 20.9,
// [16,262144] 10.5 / 11.3.
// Up to two of the widest shape a CU, the one whose workgroups end first (the narrow one where the widest leaves 150 too): so much a
// call and so much for each one that a CU has to run, and every chunk that a workgroup reads a record of (in 0.01 us, fitted to 176 tensors of 64 to 510 rows of 8200 to 33000
// elements in every shape).  With the widest ones that leave 150 workgroups instead, most of a chunk may be empty: f32 [150,12000] 9.9
// / 7.7, [100,20000] 10.2 / 7.9, [300,12000] 13.6 / 10.9, [300,16400] 13.8 either way; f16 [150,20000] 9.6 / 8.6, [300,12000]
// 11.4 / 9.9.
// More: the widest, or the narrow one where it leaves 3 % less empty.  us, 512 threads / 256: f32 [500,50257] 49.5 / 43.7, [64,200000] 28.5 / 24.8; f16
// [500,33001] 30.1 / 24.5, [500,100003] 65.9 / 57.4.
bool plan_joined(const View &v, uint32_t vec, RowShape *shape) {
    struct Candidate {
        RowShape shape;
        uint32_t call, each, most;
    };
    const uint64_t n = v.g.n, rows = v.g.outer;
    const bool many = vec == 4 || rows >= 32;
    const Candidate f32[] = {{{512, 8}, 520, 460, 16}, {{256, 10}, 690, 235, 20}, {{512, 4}, 540, 225, 8}, {{512, 2}, 480, 150, 8}};
    const Candidate f16[] = {{{512, 4}, 490, 330, many ? 16u : 8u}, {{256, 5}, 630, 175, many ? 20u : 8u}, {{512, 2}, 480, 190, 8}, {{512, 1}, 500, 133, 8}};
    const auto &of = vec == 4 ? f32 : f16;
    auto chunks = [&](const Candidate &c) { return (n + c.shape.nt * c.shape.v * vec - 1) / (c.shape.nt * c.shape.v * vec); };
    auto held = [&](const Candidate &c) { return chunks(c) * c.shape.nt * c.shape.v; };
    const Candidate *best = nullptr;
    if (rows * chunks(of[0]) > 512) {
        best = held(of[1]) * 103 < held(of[0]) * 100 ? &of[1] : &of[0];
        if (chunks(*best) > best->most) return false;
    } else {
        uint64_t least = 0;
        for (const Candidate &c : of) {
            const uint64_t groups = rows * chunks(c), cost = c.call + (groups + 255) / 256 * c.each + chunks(c) * 15;
            if (groups < 150 || groups > 1024 || chunks(c) > c.most || (best != nullptr && cost >= least)) continue;
            if (&c == &of[1] && rows * chunks(of[0]) < 150) continue;
            best = &c, least = cost;
        }
        if (best == nullptr) return false;
    }
    *shape = best->shape;
    return true;
}

SoftmaxPlan plan_softmax(const View &v, int dtype) {
    SoftmaxPlan p;
    if (v.elems == 0) return p;  // (nothing to launch; no tiles or rows to divide by)
    const uint32_t vec = dtype == VKOP_HIP_F32 ? 4u : 8u;
    const uint32_t n = v.g.n, rows = v.g.outer;
    if (v.g.inner != 1) {
        if (plan_lines(v, vec, &p)) return p;
        if (n <= static_cast<uint32_t>(vkop::kStridedMaxN)) p.kind = SoftmaxPlan::kStridedRegs;
        else {
            // a tile of TI lines (the power of two at or above min(inner, 64)) per workgroup; with too
            // few tiles to fill the chip, every tile's rows are split over G workgroups (two launches)
            p.kind = SoftmaxPlan::kStridedTile;
            while (p.ti_shift < 6 && (1u << p.ti_shift) < v.g.inner) p.ti_shift++;
            const uint32_t ti = 1u << p.ti_shift;
            const uint64_t tiles = static_cast<uint64_t>(rows) * ((v.g.inner + ti - 1) >> p.ti_shift);
            const uint32_t turn = (vkop::kStridedTileThreads / vkop::kWave) * (vkop::kWave >> p.ti_shift);  // rows per turn
            p.g = 1;
            p.per = n;
            if (tiles < 256 && n >= 8 * turn) {
                uint32_t want = static_cast<uint32_t>((512 + tiles - 1) / tiles);
                want = std::min(want, static_cast<uint32_t>(vkop::kStridedTileThreads) >> p.ti_shift);
                uint32_t per = (n + want - 1) / want;
                per = std::max((per + turn - 1) / turn * turn, 4 * turn);
                p.g = (n + per - 1) / per;
                p.per = per;
                if (p.g > 1)
                    p.workspace = kTicketBytes + align_up(static_cast<size_t>(tiles) * p.g * ti * sizeof(vkop::ChunkStat));
                else p.per = n;
            }
        }
        return p;
    }
    if (n < vec) {
        p.kind = SoftmaxPlan::kThread;
        return p;
    }
    // Rows that 8 to 64 lanes of a wave hold: the fewest lanes that need at most VT vectors each (16 to
    // 24 elements a lane: the cross-lane steps and the reciprocal are paid once for that many).
    const uint32_t nvec = (n + vec - 1) / vec, vt = dtype == VKOP_HIP_F32 ? 4u : 3u;
    if (nvec <= vt * vkop::kWave && (n <= 512 || rows >= 1024)) {
        uint32_t g = 8;
        while ((nvec + g - 1) / g > vt) g *= 2;
        p.kind = SoftmaxPlan::kGroup;
        p.shape = RowShape{static_cast<int>(g), static_cast<int>((nvec + g - 1) / g)};
        return p;
    }
    // A row per workgroup where that fills the chip or the row is short: with many rows four (f16:
    // two) vectors a thread, else as few as the 1024 threads of a workgroup allow.
    const uint32_t vmax = dtype == VKOP_HIP_F32 ? 8u : 4u;
    if (nvec <= vmax * 1024u && (n <= 8192 || rows >= 512)) {
        uint32_t v = rows >= 1024 ? vmax / 2 : 1u;
        while ((nvec + v - 1) / v > 1024u) v++;
        const uint32_t nt = ((nvec + v - 1) / v + vkop::kWave - 1) / vkop::kWave * vkop::kWave;
        p.kind = SoftmaxPlan::kRow;
        p.shape = RowShape{static_cast<int>(nt), static_cast<int>((nvec + nt - 1) / nt)};
        return p;
    }
    if (n > (1u << 25)) return p;  // (the general kernel)
    p.joined = plan_joined(v, vec, &p.shape);
    uint32_t nt = static_cast<uint32_t>(p.shape.nt), loads = static_cast<uint32_t>(p.shape.v);
    auto chunks = [&] { return (n + nt * loads * vec - 1) / (nt * loads * vec); };
    if (!p.joined) {
        // the largest chunk that still leaves 512 workgroups, else the smallest; beyond
        // 1024 chunks a row, workgroups of 1024 threads ([8,262144] f32 with 512 / 1024: 10.0 / 10.5 us;
        // [4,1048576] 14.4 / 15.4: every workgroup of the scale kernel combines all chunks of its row)
        const uint32_t loads_max = 32u / vec;
        nt = 256, loads = loads_max;
        while (loads > 1 && static_cast<uint64_t>(rows) * chunks() < 512) loads /= 2;
        if (chunks() > 1024) nt = 1024, loads = loads_max;
    }
    p.per = nt * loads * vec;
    p.g = chunks();
    p.kind = SoftmaxPlan::kChunked;
    p.shape = RowShape{static_cast<int>(nt), static_cast<int>(loads)};
    const size_t total = static_cast<size_t>(rows) * p.g;
    constexpr size_t record = vkop::kJoinedWords * sizeof(uint64_t);
    static_assert(record >= sizeof(vkop::ChunkStat), "the larger of the two");
    p.pair_workspace = kTicketBytes + align_up(total * sizeof(vkop::ChunkStat));
    p.workspace = p.joined ? kTicketBytes + align_up(total * record) : p.pair_workspace;
    return p;
}

// Which accesses of the kernels that hold a row (group, row) or a line (lines) in registers are ordinary ones.  Non-temporal ones
// keep a stream out of the caches: the better way for a tensor that those cannot serve.
// * The chip's last cache (256 MB) holds an input of up to 90 MB until it is read again, or since it was written, beside two more
//   like it (ordinary loads); the L2s (32 MB in all) those of up to 10 MB.  Between the two floats' whole lines lose a little by it.
// * Two outputs of up to half of it wait there for their reader instead of for memory (ordinary stores).  Smaller ones have to leave
//   the L2s at the kernel's end all the same, which a stream has done by then.
// * A piece of a row that begins or ends inside a 128-byte line shares that line with another wave's, and past the caches each of the
//   two fetches and stores it by itself: pieces of at most 256 bytes of rows, and lines whose rows lie off the 128 bytes, want both.
// us a call, none / loads / stores / both (three inputs and two outputs in turn):
//   rows of whole lines: f32 n = 256  8 MB 4.6 / 4.0 / 4.6 / 4.6, 16 MB 8.1 / 8.4 / 11.2 / 10.6, 50 MB 17.0 / 15.7 / 17.3 / 15.0,
//   120 MB 39.6 / 41.1 / 38.2 / 43.4, 250 MB 82 / 86 / 87 / 90; f16 n = 8192  50 MB 17.6 / 16.0 / 18.1 / 16.0
//   off the lines: f32 n = 197 (pieces of 256 bytes)  50 MB 22.4 / 19.3 / 20.0 / 17.0, 400 MB 173 / 166 / 150 / 140, f16 n = 197  64 MB
//   26.2 / 22.0 / 24.4 / 21.7, 250 MB 99 / 93 / 98 / 91; of 512 bytes f16 n = 500  180 MB 63 / 62 / 65 / 63; a lane's only
//   vector, where a wave's rows are one piece, f16 n = 50  180 MB 73 / 72 / 75 / 74
//   lines: f32 [8,21,n] of 50 MB 21.5 / 18.0 / 20.8 / 20.4, of 180 MB 68 / 70 / 71 / 75; off the 128 bytes f32 [8,100,n] of 50 MB
//   40 / 36 / 27 / 21, 180 MB 145 / 135 / 97 / 87, f16 [8,80,n] of 120 MB 93 / 82 / 55 / 56, 250 MB 190 / 163 / 131 / 105
// How much of it is the residency of those five buffers, all non-temporal / so: the shared lines' part hardly (f32 [300000,100] 64.6 /
// 46.4, of buffers that each wait for a gigabyte of others 65.5 / 46.5, [482233,197] 166 / 132 and 166 / 132, f16 [8,80,93750] axis 1
// 144 / 68 and 145 / 77, [302592,197] 46.8 / 43.7 and 47.1 / 43.9), the whole lines' all: f32 [60000,256] 25.9 / 19.4, of buffers that come from
// memory 26.1 / 27.9, behind a kernel that writes the input 40.1 / 39.7 with it, between that and one that reads the output, a
// buffer each, 61.4 / 60.2; [2400,8192] 31.8 / 25.3, 32.7 / 33.4, 50.2 / 49.9, 75.6 / 76.3; with stores [120000,256] 44.0 / 39.1, 47.0 / 45.2, 75.2 / 89.2
// (what waits is written back under the next kernel's reads), 122.8 / 118.8; lines [8,21,180224] 50.2 / 42.3, 50.5 / 50.0, 82.9 / 85.4, 123 / 126.
// (The one-launch kernel of long rows, whose tensor is in registers before any of it is written, is as fast or faster without:
// f32 [64,128256] 15.7 / 16.4 / 18.0 / 17.7.)
template <typename T> int softmax_caching(const View &v, const SoftmaxPlan &p, const T *in, const T *out, bool max_only) {
    constexpr size_t kMega = 1000000, kHalfLastCache = size_t{128} << 20;
    const size_t bytes = v.elems * sizeof(T), row_bytes = static_cast<size_t>(v.g.inner == 1 ? v.g.n : v.g.inner) * sizeof(T);
    const uintptr_t places = reinterpret_cast<uintptr_t>(in) | (max_only ? 0u : reinterpret_cast<uintptr_t>(out)) | row_bytes;
    const bool lines = p.kind == SoftmaxPlan::kLinesRegs, group = p.kind == SoftmaxPlan::kGroup, off128 = places % 128 != 0;
    if (!lines && !group && p.kind != SoftmaxPlan::kRow) return vkop::kCacheNone;
    const bool in_last = bytes >= (lines ? 30 : 24) * kMega && bytes <= 90 * kMega;
    if (max_only) return in_last ? vkop::kCacheLoads : vkop::kCacheNone;
    const bool in_l2s = bytes <= 10 * kMega || (bytes < 24 * kMega && !lines && (sizeof(T) == 2 || off128));
    const int loads = in_last || (in_l2s && !(p.kind == SoftmaxPlan::kRow)) ? vkop::kCacheLoads : vkop::kCacheNone;
    if (lines && off128) {
        // (a wave's piece of a row of a kilobyte, or pieces that start on 16 bytes, have fewer lines in part: from 40 MB on, the
        // others from 28.  At 33.5 MB f32, none / stores: [8,80,13107] 24.5 / 18.4, [8,80,13108] 23.1 / 18.6, but [8,200,5240]
        // 16.5 / 18.0 and [8,16,65537] 16.2 / 17.4)
        const bool on16 = places % 16 == 0, late = p.lines_p == 1 || (on16 && !(p.lines_p == 8 && p.lines_w == 1));
        if (bytes < (late ? 40u : 28u) * kMega) return loads;
        if (bytes <= 80 * kMega) return on16 ? vkop::kCacheLoads : vkop::kCacheBoth;
        return bytes > kHalfLastCache ? vkop::kCacheBoth : vkop::kCacheStores;
    }
    if (group && off128 && p.shape.v > 1 && p.shape.nt <= 16 && bytes >= 24 * kMega) return vkop::kCacheBoth;
    if (loads != vkop::kCacheNone) return loads;
    const bool one_piece = group && off128 && p.shape.v == 1;
    return (lines || (group && !one_piece)) && bytes > 90 * kMega && bytes <= kHalfLastCache ? vkop::kCacheStores : vkop::kCacheNone;
}
// f(std::integral_constant<int, CACHE>) for a run-time `caching`
template <typename F> void with_caching(int caching, F &&f) {
    switch (caching) {
    case vkop::kCacheLoads: return f(std::integral_constant<int, vkop::kCacheLoads>{});
    case vkop::kCacheStores: return f(std::integral_constant<int, vkop::kCacheStores>{});
    case vkop::kCacheBoth: return f(std::integral_constant<int, vkop::kCacheBoth>{});
    default: return f(std::integral_constant<int, vkop::kCacheNone>{});
    }
}

template <typename T>
int launch_lines(const T *in, T *out, const View &v, const SoftmaxPlan &p, bool max_only, int nan_where, float nan_value,
                 hipStream_t st) {
    return in_slices(v.g.outer, lines_threads(v, 16 / sizeof(T), p.lines_p, p.lines_w), [&](uint64_t first, uint32_t outer) {
        vkop::LinesLaunch a{in + first * v.g.n * v.g.inner, out + first * (max_only ? 1u : v.g.n) * v.g.inner, v.g, p.lines_k, p.lines_p,
                            p.lines_w, max_only, softmax_caching(v, p, in, out, max_only), nan_where, nan_value, st};
        a.g.outer = outer;
        if (!vkop::launch_softmax_lines<T>(a))
            return fail(VKOP_HIP_ERR_UNSUPPORTED, "no softmax_lines_reg_kernel for %u elements x %u", a.k, a.p);
        return launched("softmax_lines_reg_kernel");
    });
}

// Whether softmax_joined_kernel may run on these tensors: they share no byte, or are the same and no row's last vector reaches
// back into the chunk before its own.
template <typename T> bool joined_fits(const T *in, const T *out, const View &v, const SoftmaxPlan &p) {
    const auto x = reinterpret_cast<uintptr_t>(in), y = reinterpret_cast<uintptr_t>(out);
    const uint32_t last = v.g.n % p.per;
    return x == y ? last == 0 || last >= 16 / sizeof(T) : (x < y ? y - x : x - y) >= v.elems * sizeof(T);
}

template <typename T>
int launch_joined(const T *in, T *out, const View &v, const SoftmaxPlan &p, int nan_where, float nan_value, void *ws, hipStream_t st) {
    auto *done = static_cast<uint32_t *>(ws);
    auto *recs = reinterpret_cast<uint64_t *>(static_cast<unsigned char *>(ws) + kTicketBytes);
    // (a counter a row: as many rows a launch as there are of them)
    for (uint64_t row0 = 0; row0 < v.g.outer; row0 += kTicketRows) {
        const uint32_t rows = static_cast<uint32_t>(std::min<uint64_t>(kTicketRows, v.g.outer - row0));
        const uint32_t tag = vkop::launch_tag(g_joined_calls.fetch_add(1, std::memory_order_relaxed));
        const T *from = in + row0 * v.g.n;
        T *to = out + row0 * v.g.n;
        auto launch = [&](auto kernel) {
            kernel<<<rows * p.g, p.shape.nt, 0, st>>>(from, to, recs + row0 * p.g * vkop::kJoinedWords, done, v.g.n, p.g, tag,
                                                      joined_polls(), nan_where, nan_value);
            return launched("softmax_joined_kernel");
        };
        int rc = -1;
#define VKOP_JOINED(NT, V) \
    if (p.shape.nt == NT && p.shape.v == V) rc = launch(vkop::softmax_joined_kernel<T, NT, V>);
        VKOP_JOINED(512, 2) VKOP_JOINED(512, 4)
        if constexpr (sizeof(T) == 4) { VKOP_JOINED(256, 10) VKOP_JOINED(512, 8) }
        else { VKOP_JOINED(256, 5) VKOP_JOINED(512, 1) }
#undef VKOP_JOINED
        if (rc < 0) return fail(VKOP_HIP_ERR_UNSUPPORTED, "no softmax_joined_kernel for %d x %d", p.shape.nt, p.shape.v);
        if (rc != VKOP_HIP_OK) return rc;
    }
    return VKOP_HIP_OK;
}

// The softmax of last-axis rows, or (MAX_ONLY) each row's largest probability: the kernels of kThread ... kChunked.
template <typename T, bool MAX_ONLY>
int softmax_rows(const T *in, T *out, const View &v, const SoftmaxPlan &p, int nan_where, float nan_value, void *ws,
                 size_t ws_bytes, hipStream_t st) {
    const uint32_t lines = v.g.outer;
    const uint64_t out_row = MAX_ONLY ? 1u : v.g.n;
    const int caching = softmax_caching(v, p, in, out, MAX_ONLY);
    const auto kind = MAX_ONLY && v.g.n <= vkop::kSoftmaxThreadMaxN ? SoftmaxPlan::kThread : p.kind;
    switch (kind) {
    case SoftmaxPlan::kThread: {
        const uint32_t blocks = (lines + vkop::kSoftmaxGroupThreads - 1) / vkop::kSoftmaxGroupThreads;
        vkop::softmax_thread_kernel<T, MAX_ONLY><<<blocks, vkop::kSoftmaxGroupThreads, 0, st>>>(in, out, lines, v.g.n, nan_where, nan_value);
        return launched("softmax_thread_kernel");
    }
    case SoftmaxPlan::kGroup: {
        const uint32_t per_block = static_cast<uint32_t>(vkop::kSoftmaxGroupThreads / p.shape.nt);
        return in_slices((lines + per_block - 1) / per_block, vkop::kSoftmaxGroupThreads, [&](uint64_t first, uint32_t blocks) {
            const uint64_t row0 = first * per_block;
            const T *from = in + row0 * v.g.n;
            T *to = out + row0 * out_row;
            const uint32_t rows = static_cast<uint32_t>(std::min<uint64_t>(lines - row0, static_cast<uint64_t>(blocks) * per_block));
#define VKOP_GROUP(G, V)                                                                                                       \
    if (p.shape.nt == G && p.shape.v == V) {                                                                                   \
        with_caching(caching, [&](auto cache) {                                                                                \
            constexpr int CACHE = MAX_ONLY ? cache & vkop::kCacheLoads : cache;                                                \
            vkop::softmax_group_kernel<T, G, V, MAX_ONLY, CACHE>                                                               \
                <<<blocks, vkop::kSoftmaxGroupThreads, 0, st>>>(from, to, rows, v.g.n, nan_where, nan_value);                  \
        });                                                                                                                    \
        return launched("softmax_group_kernel");                                                                               \
    }
#define VKOP_GROUPS(G) VKOP_GROUP(G, 1) VKOP_GROUP(G, 2) VKOP_GROUP(G, 3) if constexpr (sizeof(T) == 4) { VKOP_GROUP(G, 4) }
            VKOP_GROUPS(8) VKOP_GROUPS(16) VKOP_GROUPS(32) VKOP_GROUPS(64)
#undef VKOP_GROUPS
#undef VKOP_GROUP
            return fail(VKOP_HIP_ERR_UNSUPPORTED, "no softmax_group_kernel for %d lanes x %d", p.shape.nt, p.shape.v);
        });
    }
    case SoftmaxPlan::kRow: {
        return in_slices(lines, p.shape.nt, [&](uint64_t row0, uint32_t rows) {
            const T *from = in + row0 * v.g.n;
            T *to = out + row0 * out_row;
#define VKOP_ROW(V)                                                                                     \
    if (p.shape.v == V) {                                                                               \
        with_caching(caching, [&](auto cache) {                                                         \
            constexpr int CACHE = cache & vkop::kCacheLoads; /* (no more: softmax_caching) */            \
            vkop::softmax_row_kernel<T, V, MAX_ONLY, CACHE><<<rows, p.shape.nt, 0, st>>>(from, to, v.g.n, nan_where, nan_value); \
        });                                                                                             \
        return launched("softmax_row_kernel");                                                          \
    }
            VKOP_ROW(1) VKOP_ROW(2) VKOP_ROW(3) VKOP_ROW(4)
            if constexpr (sizeof(T) == 4) { VKOP_ROW(5) VKOP_ROW(6) VKOP_ROW(7) VKOP_ROW(8) }
#undef VKOP_ROW
            return fail(VKOP_HIP_ERR_UNSUPPORTED, "no softmax_row_kernel for %d x %d", p.shape.nt, p.shape.v);
        });
    }
    case SoftmaxPlan::kChunked: {
        if (ws == nullptr || ws_bytes < p.pair_workspace)
            return fail(VKOP_HIP_ERR_WORKSPACE, "workspace of %zu bytes given, %zu needed", ws_bytes, p.pair_workspace);
        // (a record is larger than a chunk's statistics: in a workspace that holds only those, the pair)
        if (!MAX_ONLY && p.joined && ws_bytes >= p.workspace && joined_fits(in, out, v, p) &&
            reinterpret_cast<uintptr_t>(ws) % sizeof(uint64_t) == 0)
            return launch_joined(in, out, v, p, nan_where, nan_value, ws, st);
        auto *stats = reinterpret_cast<vkop::ChunkStat *>(static_cast<unsigned char *>(ws) + kTicketBytes);
        // the most vectors a thread (four floats', two halves') that leave 2048 workgroups: with fewer in all
        // their stores wait for each other, with smaller ones more of them combine the same chunks
        const uint32_t vec = 16 / sizeof(T);
        auto pieces = [&](uint32_t loads) { return (v.g.n + vkop::kSoftmaxScaleThreads * loads * vec - 1) / (vkop::kSoftmaxScaleThreads * loads * vec); };
        uint32_t loads = 16 / vec;
        while (loads > 1 && static_cast<uint64_t>(v.g.outer) * pieces(loads) < 2048) loads /= 2;
        const uint32_t gs = pieces(loads);
        const uint64_t threads = std::max<uint64_t>(static_cast<uint64_t>(p.g) * p.shape.nt, static_cast<uint64_t>(gs) * vkop::kSoftmaxScaleThreads);
        return in_slices(v.g.outer, threads, [&](uint64_t row0, uint32_t rows) {
            const T *from = in + row0 * v.g.n;
            T *to = out + row0 * out_row;
            auto *row_stats = stats + row0 * p.g;
            bool done = false;
#define VKOP_STATS(NT, V)                                                                                \
    if (!done && p.shape.nt == NT && p.shape.v == V) {                                                   \
        vkop::softmax_stats_kernel<T, NT, V><<<rows * p.g, NT, 0, st>>>(from, row_stats, v.g.n, p.g);    \
        done = true;                                                                                     \
    }
            VKOP_STATS(256, 1) VKOP_STATS(256, 2) VKOP_STATS(256, 4) VKOP_STATS(512, 2) VKOP_STATS(512, 4)
            if constexpr (sizeof(T) == 4) { VKOP_STATS(256, 8) VKOP_STATS(256, 10) VKOP_STATS(512, 8) VKOP_STATS(1024, 8) }
            else { VKOP_STATS(256, 5) VKOP_STATS(512, 1) VKOP_STATS(1024, 4) }
#undef VKOP_STATS
            if (!done) return fail(VKOP_HIP_ERR_UNSUPPORTED, "no softmax_stats_kernel for %d x %d", p.shape.nt, p.shape.v);
            if constexpr (MAX_ONLY) {
                vkop::softmax_fold_max_kernel<T><<<rows, vkop::kSoftmaxScaleThreads, 0, st>>>(to, row_stats, p.g);
                return launched("softmax_stats_kernel / softmax_fold_max_kernel");
            }
#define VKOP_SCALE(V) \
    if (loads == V)   \
        vkop::softmax_scale_kernel<T, V><<<rows * gs, vkop::kSoftmaxScaleThreads, 0, st>>>(from, to, row_stats, v.g.n, p.g, gs, nan_where, nan_value);
            VKOP_SCALE(1) VKOP_SCALE(2)
            if constexpr (sizeof(T) == 4) { VKOP_SCALE(4) }
#undef VKOP_SCALE
            return launched("softmax_stats_kernel / softmax_scale_kernel");
        });
    }
    default:
        return fail(VKOP_HIP_ERR_UNSUPPORTED, "not a plan of last-axis rows");
    }
}

template <typename T>
int softmax_impl(const T *in, T *out, const View &v, int dtype, int nan_where, float nan_value, void *ws,
                 size_t ws_bytes, hipStream_t st) {
    const SoftmaxPlan p = plan_softmax(v, dtype);
    const uint32_t lines = v.g.outer * v.g.inner;
    switch (p.kind) {
    case SoftmaxPlan::kThread:
    case SoftmaxPlan::kGroup:
    case SoftmaxPlan::kRow:
    case SoftmaxPlan::kChunked:
        return softmax_rows<T, false>(in, out, v, p, nan_where, nan_value, ws, ws_bytes, st);
    case SoftmaxPlan::kLinesRegs: {
        return launch_lines(in, out, v, p, false, nan_where, nan_value, st);
    }
    case SoftmaxPlan::kStridedRegs: {
        launch_strided_reg<T, false>(in, out, v, nan_where, nan_value, st);
        return launched("softmax_strided_reg_kernel");
    }
    case SoftmaxPlan::kStridedTile: {
        const uint32_t tiles = v.g.outer * ((v.g.inner + (1u << p.ti_shift) - 1) >> p.ti_shift);
        if (p.g == 1) {
            vkop::softmax_strided_tile_kernel<T, vkop::kTileWhole>
                <<<tiles, vkop::kStridedTileThreads, 0, st>>>(in, out, nullptr, v.g, p.ti_shift, 1, v.g.n, nan_where, nan_value);
            return launched("softmax_strided_tile_kernel");
        }
        if (ws == nullptr || ws_bytes < p.workspace)
            return fail(VKOP_HIP_ERR_WORKSPACE, "workspace of %zu bytes given, %zu needed", ws_bytes, p.workspace);
        auto *stats = reinterpret_cast<vkop::ChunkStat *>(static_cast<unsigned char *>(ws) + kTicketBytes);
        vkop::softmax_strided_tile_kernel<T, vkop::kTileStats>
            <<<tiles * p.g, vkop::kStridedTileThreads, 0, st>>>(in, out, stats, v.g, p.ti_shift, p.g, p.per, nan_where, nan_value);
        vkop::softmax_strided_tile_kernel<T, vkop::kTileScale>
            <<<tiles * p.g, vkop::kStridedTileThreads, 0, st>>>(in, out, stats, v.g, p.ti_shift, p.g, p.per, nan_where, nan_value);
        return launched("softmax_strided_tile_kernel (split)");
    }
    case SoftmaxPlan::kGeneralLines:
        vkop::softmax_lines_kernel<T, kLineThreads>
            <<<lines, kLineThreads, 0, st>>>(in, out, v.g, nan_where, nan_value, nullptr);
        return launched("softmax_lines_kernel");
    case SoftmaxPlan::kGeneralStrided:
    default: {
        const uint32_t blocks = (lines + kLineThreads - 1) / kLineThreads;
        vkop::softmax_strided_kernel<T, kLineThreads><<<blocks, kLineThreads, 0, st>>>(in, out, v.g, nan_where, nan_value);
        return launched("softmax_strided_kernel");
    }
    }
}

// ------------------------------------------------- streaming rows kernel ----
// Launch shape of rows_chunk_kernel: NT threads, V 128-bit loads per thread,
// G chunks per row of `per` elements each, `cap` candidate slots per chunk.
struct RowsCfg {
    bool ok = false;
    int nt = 0, v = 0;
    uint32_t g = 0, per = 0;
    uint32_t cap = 0, cap_shift = 0;
    bool forced = false;  // the shape that rows.threads, rows.loads and rows.chunks ask for
    // a row that one workgroup holds never leaves it: list and records stay in LDS
    bool local() const { return g == 1 && cap <= static_cast<uint32_t>(vkop::kLocalCap); }
};

// Candidate slots per chunk: 2.5 times the k+1 wanted elements (a chunk of
// identically distributed data has about 1.2 times k+1 at or above its
// threshold), at least 64, power of two.
uint32_t rows_cap(int k) {
    const uint32_t want = static_cast<uint32_t>(k) + 1u;
    uint32_t cap = 64;
    while (2u * cap < 5u * want) cap <<= 1;
    return cap;
}

constexpr int kWaveRowMaxK = 32;  // largest k served by the one-wave-per-row launch
constexpr int kTwoAndHalfListsMaxK = 408;  // largest k with rows_cap(k) <= kLocalCap
constexpr int kWideRowMinK = 64;  // above it a row that fits one workgroup is given to one (of enough threads)

enum RowsKind { kPlainRows, kFusedRows, kScaledRows };  // top-k, softmax and top-k, the sampling form of that

// (for_size: what a call could use whatever rows.path says at that time.  kind: which call it is for.
// full_list: also a k whose places the list of a one-workgroup row holds less than 2.5 times, 409 to 511: usual rows list 1.2 to 1.4 times the places, and a second listing at most
// 2 k + 1 elements, 1023 of the list's 1024.)
RowsCfg choose_rows_cfg(const View &v, int k, int dtype, bool for_size = false, bool full_list = false, RowsKind kind = kFusedRows) {
    RowsCfg c;
    if (v.g.inner != 1 || k > vkop::kFastMaxK || v.g.n == 0 || v.g.outer == 0) return c;
    const uint32_t vec = dtype == VKOP_HIP_F32 ? 4u : 8u;
    const uint32_t n = v.g.n, rows = v.g.outer;
    static const int shapes_f32[][2] = {{256, 1}, {256, 2}, {256, 4}, {256, 8}, {512, 8}, {1024, 8}};
    static const int shapes_f16[][2] = {{256, 1}, {256, 2}, {256, 4}, {512, 4}, {1024, 4}, {1024, 4}};
    const auto *shapes = dtype == VKOP_HIP_F32 ? shapes_f32 : shapes_f16;
    int forced_nt = g_rows_threads.load(), forced_v = g_rows_loads.load(), forced_g = g_rows_chunks.load();
    if (forced_nt <= 0 || forced_v <= 0 || forced_g <= 0) forced_nt = 0;
    const uint32_t nvec = (n + vec - 1) / vec;
    const uint32_t cap = full_list ? std::min(rows_cap(k), static_cast<uint32_t>(vkop::kLocalCap)) : rows_cap(k);
    auto fits = [&](int nt, int vv, uint32_t g) {
        const uint32_t nw = static_cast<uint32_t>(nt) / 64u;
        if (g < 1 || g > static_cast<uint32_t>(vkop::kMergeChunksMax)) return false;
        if (static_cast<uint64_t>(g) * nw > static_cast<uint64_t>(vkop::kMergeWavesMax)) return false;
        if (static_cast<uint64_t>(g) * cap > static_cast<uint64_t>(vkop::kMergeRecsMax)) return false;
        const uint64_t span = static_cast<uint64_t>(nt) * vv * vec;
        return span * g >= n && static_cast<uint64_t>(rows) * g < (1ull << 31);
    };
    // short rows and a small k: one wave per row (64 threads, up to 8 loads each)
    const uint32_t wave_loads = (nvec + 63) / 64;
    // A large k on a row that one workgroup can hold: that workgroup takes the whole
    // row, list in LDS, if it has at least 2 (k + 1) threads (its waves share the
    // staging of the candidates, 64 vectors each, and the ranking; several chunks of
    // 256 threads would hand a merge of 256 threads more candidates than it ranks
    // quickly).  Beyond 255 ranks it is the only way: the merge kernel has a thread
    // per rank.
    int wide = -1;
    if (cap <= static_cast<uint32_t>(vkop::kLocalCap)) {
        for (int i = 0; i < 6 && wide < 0; i++) {
            const uint64_t span = static_cast<uint64_t>(shapes[i][0]) * shapes[i][1] * vec;
            if (span >= n && shapes[i][0] >= 2 * (k + 1)) wide = i;
        }
    }
    if (k > vkop::kMergeThreads - 1 && wide < 0) return c;
    if (wide >= 0 && (k > vkop::kMergeThreads - 1 || (k > kWideRowMinK && !forced_nt))) {
        c.nt = shapes[wide][0], c.v = shapes[wide][1], c.g = 1;
    } else if (forced_nt) {
        if (!fits(forced_nt, forced_v, static_cast<uint32_t>(forced_g)) || (n < vec && forced_v > 1)) return c;
        c.nt = forced_nt, c.v = forced_v, c.g = static_cast<uint32_t>(forced_g), c.forced = true;
    } else if (k <= kWaveRowMaxK && wave_loads <= (dtype == VKOP_HIP_F32 ? 8u : 4u)) {
        c.nt = 64, c.g = 1;
        c.v = wave_loads <= 1 ? 1 : wave_loads <= 2 ? 2 : wave_loads <= 4 ? 4 : 8;
    } else {
        // Several chunks a row.  With a k above 64 (only rows the scan kernels do not take
        // get here: half-precision rows of 32K to 64K elements, rows beyond 8192 blocks) the
        // chunks' lists overflow on anything but well-spread data and are made again from an
        // exact select, 70 to 700 us measured; the multi-pass radix select takes 50 us
        // whatever the data.  (rows.path = 1 keeps these kernels on every shape they can do.)
        if (!for_size && k > kWideRowMinK && g_rows_path.load() != 1) return c;
        // a row that one workgroup of 256 threads can hold: the smallest such shape (many short rows
        // would otherwise get the largest workgroup, most of its threads without an element); else the
        // largest per-workgroup chunk that still leaves >= 1024 workgroups; if the
        // tensor is too small for that, the smallest shape that covers a row
        int pick = -1;
        for (int i = 0; i < 4 && pick < 0; i++) {
            const uint64_t span = static_cast<uint64_t>(shapes[i][0]) * shapes[i][1] * vec;
            if (shapes[i][0] == 256 && span >= n && fits(shapes[i][0], shapes[i][1], 1)) pick = i;
        }
        // a row just past those shapes that has too few blocks for the scan kernels (8193 to 8320 elements at
        // k = 64): the wider workgroup that holds it, rather than several chunks and a merge
        const uint32_t blocks = (n + vkop::kBlockLanes * vec - 1) / (vkop::kBlockLanes * vec);
        if (pick < 0 && wide >= 0 && !forced_nt && g_rows_path.load() != 1 &&
            4ull * blocks < (rows <= 16 ? 8ull : 7ull) * (static_cast<uint64_t>(k) + 1u))
            pick = wide;
        // The rows that 512 threads hold (to 16384 elements), and in plain top-k of halves with k > 32 those that 1024
        // hold, on up to a row a CU: one launch that reads a row once and keeps it, for the scan's two.  us a call, scan
        // and pick / one workgroup a row: top-k [64,16384] f16 k = 64 14.6 / 7.6, k = 5 9.0 / 6.5, [256,8400] f32 k = 40
        // 11.2 / 7.4, [64,24000] f16 k = 64 12.0 / 9.1; fused [256,16384] f16 k = 64 20.5 / 13.2, [16,12000] f32 k = 20
        // 10.2 / 9.3.  Beyond 16384 elements the scan stays
        // ahead where it spreads the work over more CUs: fused ([16,28000] f32 k = 20 10.0 / 12.0, all exponentials of a
        // row on one), and in rows of few values ([64,24000] k = 5 f32 10.0 / 13.8, f16 10.6 / 13.1; k = 40 f16 13.7 /
        // 13.1, f32 10.6 / 12.9); and so it does in the scaled form of a few float rows whose length takes them off 16 bytes
        // ([2,12001] k = 20 10.6 / 11.0, [200,12001] 12.8 / 11.7; rows of a whole number of vectors in a tensor that starts off
        // them are as fast either way or faster so, [64,16384] k = 50 12.3 / 10.2).
        // With more rows than CUs the workgroups take turns, and the scan is ahead again: fused f32 k = 5 [256,12000] 12.4 /
        // 10.0, [257,12000] 13.4 / 16.8, k = 20 [768,16384] 20.7 / 30.0, [3000,16384] 68 / 113, f16 k = 5 [3000,12000] 71 / 97;
        // scaled f32 k = 40 of 513 values [300,12000] 16.8 / 28.8; top-k k = 5 f32 [300,12000] 11.6 / 13.6, f16 [1000,10001]
        // 21.3 / 27.0, smallest first f32 k = 20 [1500,10001] 33 / 78.  Not in plain top-k of few blocks a place, which the
        // scan's threshold hardly tells apart: f16 [300,10001] k = 40 17.6 / 13.9, [300,16384] k = 64 17.7 / 13.5, f32
        // [768,8400] k = 64 28.3 / 23.3; at 2.7 a place f16 k = 40 [300,14003] 13.9 / 14.2, of 513 values 19.9 / 16.1, [1000,14003]
        // 25.5 / 28.4.
        if (pick < 0 && wide >= 0 && !forced_nt && !for_size && g_rows_path.load() != 1 && g_rows_fused.load() == 0) {
            const bool narrow = shapes[wide][0] <= 512, half = vec == 8u, plain = kind == kPlainRows;
            const bool few_blocks = plain && 4ull * blocks < (half && rows <= 768 ? 11ull : 9ull) * (static_cast<uint64_t>(k) + 1u);
            const bool one = narrow ? kind != kScaledRows || rows > 64 || half || n % vec == 0u : plain && half && k > kWaveRowMaxK;
            if (one && rows > 256 && !few_blocks) return c;
            if (one) pick = wide;
        }
        const bool one_workgroup = pick >= 0;
        for (int i = 0; i < 6 && !one_workgroup; i++) {
            const uint32_t span = static_cast<uint32_t>(shapes[i][0]) * shapes[i][1] * vec;
            const uint32_t g = (n + span - 1) / span;
            if (!fits(shapes[i][0], shapes[i][1], g)) continue;
            if (pick < 0) pick = i;
            if (static_cast<uint64_t>(rows) * g >= 1024) pick = i;
        }
        if (pick < 0) return c;
        c.nt = shapes[pick][0], c.v = shapes[pick][1];
        const uint32_t span = static_cast<uint32_t>(c.nt) * c.v * vec;
        c.g = (n + span - 1) / span;
    }
    // chunks are whole multiples of the workgroup's capacity wherever the row allows
    // it, so that all but the last chunk of a row run the unmasked code
    c.per = static_cast<uint32_t>(c.nt) * c.v * vec;
    if (static_cast<uint64_t>(c.per) * (c.g - 1) >= n) c.per = (nvec + c.g - 1) / c.g * vec;
    c.cap = cap;
    while ((1u << c.cap_shift) < c.cap) c.cap_shift++;
    c.ok = true;
    return c;
}

// Short last-axis rows, largest first, k up to kTinyMaxK: one wave per row
// (kernels_tiny.hpp); v = 128-bit loads per lane, 0 = not for this tensor.
int choose_tiny_loads(const View &v, int k, int dtype) {
    if (v.g.inner != 1 || k < 1 || k > vkop::kTinyMaxK || v.g.n == 0 || v.g.outer == 0) return 0;
    if (g_rows_path.load() == 1) return 0;
    if (g_rows_threads.load() > 0 && g_rows_loads.load() > 0 && g_rows_chunks.load() > 0) return 0;
    const uint32_t vec = dtype == VKOP_HIP_F32 ? 4u : 8u;
    const int vmax = dtype == VKOP_HIP_F32 ? 8 : 4;
    for (int vv = 1; vv <= vmax; vv *= 2)
        if (static_cast<uint32_t>(vkop::kWave) * vv * vec >= v.g.n) return vv;
    return 0;
}

template <typename T, bool SOFTMAX>
int launch_tiny(const T *in, T *values, int32_t *indices, const View &v, int k, int loads, hipStream_t st,
                bool smallest = false, bool sampling = false, float scale = 1.f, int32_t *counts = nullptr, float top_p = 0.f) {
    vkop::TinyLaunch a;
    a.in = in;
    a.values = values;
    a.indices = indices;
    a.rows = v.g.outer;
    a.n = v.g.n;
    a.k = static_cast<uint32_t>(k);
    a.v = static_cast<uint32_t>(loads);
    a.aligned = (reinterpret_cast<uintptr_t>(in) % 16 == 0) && (v.g.n % (16 / sizeof(T)) == 0);
    a.smallest = smallest;
    a.stream = st;
    a.sampling = sampling;
    a.scale = scale;
    a.counts = counts;
    a.top_p = top_p;
    if (!vkop::launch_rows_tiny<T, SOFTMAX>(a)) return fail(VKOP_HIP_ERR_UNSUPPORTED, "no rows_tiny_kernel for %d loads", loads);
    return launched("rows_tiny_kernel");
}

// Launch shape of the streaming pair rows_scan_kernel + rows_pick_kernel: 256 threads,
// V 128-bit loads per thread, G chunks per row; blocks = 256-byte blocks per row.
struct ScanCfg {
    bool ok = false;
    int v = 0;
    uint32_t g = 0, blocks = 0;
    uint32_t g2 = 0;  // k beyond the pick kernel's list: workgroups a row of the gather kernel (kernels_bigpick.hpp)
};

// Long last-axis rows, largest first: the scan kernel followed by the pick kernel (k up to
// kFastMaxK) or by the large-k pair (g2 != 0: beyond that k, and on up to 16 rows from k = 256,
// or from k = 160 where the pick kernel has too few blocks).  The largest chunk that still
// leaves 512 workgroups (else the smallest); rows too short to be split, or with too few
// blocks per wanted place (below), or with more blocks than the kernel behind the scan takes
// in, are left to the other kernels.
// (for_size: what a call could use whatever the tuning knobs say at that time)
ScanCfg choose_scan_cfg(const View &v, int k, int dtype, bool for_size = false, RowsKind kind = kFusedRows) {
    ScanCfg c;
    if (v.g.inner != 1 || k > vkop::kMaxK || v.g.n == 0 || v.g.outer == 0) return c;
    const uint32_t vec = dtype == VKOP_HIP_F32 ? 4u : 8u;
    const uint32_t n = v.g.n, rows = v.g.outer;
    // The pick kernel ranks a row in one workgroup, the large-k pair spreads it over many: on up to 16
    // rows that pair is the faster one from k = 256 on ([8,262144] k = 256: 17.7 against 23.1 us;
    // [4,100000] k = 500: 15.6 against 44 us), with more rows the pick kernel stays ahead up to its
    // limit ([64,128256] k = 500 fused: 50 against 52 us; [128,65536] k = 256: 24 against 39 us).
    const bool few_rows = rows <= 16;
    bool big = k > vkop::kFastMaxK || (few_rows && k >= 256);
    if (!for_size) {
        if (g_rows_path.load() == 1) return c;
        // a forced shape of the other streaming kernels
        if (g_rows_threads.load() > 0 && g_rows_loads.load() > 0 && g_rows_chunks.load() > 0) return c;
    }
    const uint32_t blocks = (n + vkop::kBlockLanes * vec - 1) / (vkop::kBlockLanes * vec);
    // Blocks per wanted place, in quarters.  The pick kernel's threshold is the (k+1)-th largest of its
    // 512 threads' maxima: at or above their median -- k + 1 <= 256, twice as many blocks -- few blocks
    // and elements reach it; closer to the smallest of them, more blocks have to stand behind every
    // thread -- which costs one workgroup per row less when other rows keep the chip busy: with more
    // than 16 rows, 1.75 blocks a place are enough at every k ([64,128256] f16 k = 300, 3.3 a place:
    // 28.9 us, fused 34.5, against 49 / 132 us of the radix select; [32,50257] f16 k = 200, 1.95 a
    // place: 24.4 against 46.8 us).  The large-k kernels get by with 1.25 a place on a few rows (they
    // read most of the row again then, and still beat the radix select: [8,262144] f16 k = 1024, 2048
    // blocks: 21.7 against 42.8 us; [2,65536] k = 512: 16.0 against 37.8 us); with many rows their
    // ranking is what the time goes into ([64,100000] k = 1240: 125 against 64 us).
    const uint64_t places = static_cast<uint64_t>(k) + 1u;
    uint32_t quarters = big ? (few_rows ? 5u : 8u) : (!few_rows ? 7u : (places <= 256 ? 8u : 16u));
    if (!big && few_rows && k >= 160 && 4ull * blocks < quarters * places) {
        // too few blocks for the pick kernel on a few rows: the large-k pair again, from k = 160 on (below,
        // rows sorted in runs cost it several times the radix select: [16,128256] k = 128: 422 us)
        // ([8,50257] f16 k = 200: 16.8 against 44.5 us of the radix select; [16,100000] f16 k = 400: 21.0 against 38.9)
        big = true;
        quarters = 5u;
    }
    if (4ull * blocks < quarters * places) return c;
    if (k <= vkop::kFastMaxK && !for_size) {
        // a row that ONE workgroup of the chunk kernel holds (up to 16384 elements, for a larger k up to
        // 32768): one launch instead of two, measured 1.1 to 1.9 times faster on spread-out
        // rows ([1024,4096] k = 16: 9.0 against 14.5 us; [64,32768] k = 200: 12.5 against 20.3 us)
        const RowsCfg one = choose_rows_cfg(v, k, dtype, false, false, kind);
        if (one.ok && one.g == 1 && one.nt >= 256) return c;
    }
    if (!big && (blocks + vkop::kPickThreads - 1) / vkop::kPickThreads > 32u) return c;
    if (big && (blocks + vkop::kBigPickThreads - 1) / vkop::kBigPickThreads > 32u) return c;
    if (big && static_cast<uint64_t>(rows) * (vkop::kBigPickCap / vkop::kBigPickMine) >= (1ull << 31)) return c;
    const uint32_t waves_max = big ? static_cast<uint32_t>(vkop::kBigPickRecsMax) : static_cast<uint32_t>(vkop::kMergeWavesMax);
    const int vmax = dtype == VKOP_HIP_F32 ? 16 : 8;
    int pick = 0;
    for (int vv = 2; vv <= vmax; vv *= 2) {
        const uint32_t per = static_cast<uint32_t>(vkop::kScanThreads) * vv * vec;
        const uint32_t g = (n + per - 1) / per;
        if (g < 2 || g * vkop::kScanWaves > waves_max) continue;
        if (static_cast<uint64_t>(rows) * g >= (1ull << 31)) continue;
        if (pick == 0) pick = vv;
        if (static_cast<uint64_t>(rows) * g >= 512) pick = vv;
    }
    if (pick == 0) return c;
    c.v = pick;
    const uint32_t per = static_cast<uint32_t>(vkop::kScanThreads) * pick * vec;
    c.g = (n + per - 1) / per;
    c.blocks = blocks;
    if (big) {
        // a share of at most 256 blocks (a thread each) and, rows permitting, of at least 32;
        // about 512 workgroups in all
        const uint32_t least = (blocks + 255u) / 256u, most = (blocks + 31u) / 32u;
        const uint32_t fill = (512u + rows - 1u) / rows;
        c.g2 = std::max(least, std::min(fill, most));
        if (static_cast<uint64_t>(rows) * c.g2 >= (1ull << 31)) return c;
    }
    c.ok = true;
    return c;
}

struct RowsLayout {
    size_t tickets = 0, sums = 0, cand = 0, stats = 0, total = 0;
    // scan + pick pair (kernels_stream.hpp)
    size_t bmax = 0, recs = 0, bmin = 0, bcand = 0, bterm = 0, bhead = 0, bstat = 0;
    // multi-workgroup radix select (kernels_bigk.hpp)
    size_t hist = 0, hist_bytes = 0, state = 0, counts = 0, sel = 0, chunkstats = 0;
};

// Launch shape of the multi-workgroup radix select: chunks of 8192 elements.
struct BigKCfg {
    bool ok = false;
    int v = 0;
    uint32_t g = 0, per = 0, kpad = 0;
};

BigKCfg choose_bigk_cfg(const View &v, int k, int dtype) {
    BigKCfg c;
    if (v.g.inner != 1 || v.g.n < 16384 || k < 1 || k > vkop::kMaxK || v.g.outer == 0) return c;
    c.v = dtype == VKOP_HIP_F32 ? 8 : 4;
    c.per = static_cast<uint32_t>(vkop::kBigThreads) * c.v * (dtype == VKOP_HIP_F32 ? 4u : 8u);
    c.g = (v.g.n + c.per - 1) / c.per;
    if (c.g > static_cast<uint32_t>(vkop::kBigThreads) || static_cast<uint64_t>(v.g.outer) * c.g >= (1ull << 31)) return c;
    c.kpad = (static_cast<uint32_t>(k) + 31u) / 32u * 32u;
    c.ok = true;
    return c;
}

// One layout serves the streaming kernel and the general two-kernel path, so
// the size does not depend on which of them a call ends up taking.
// (the arrival counters come first, see kTicketRows)

RowsLayout rows_layout(const View &v, const RowsCfg &c, const BigKCfg &b = BigKCfg{}, const ScanCfg &sc = ScanCfg{}) {
    RowsLayout l;
    const size_t lines = static_cast<size_t>(v.g.outer) * v.g.inner;
    size_t off = 0;
    l.tickets = off;
    off += kTicketBytes;
    l.stats = off;
    off += align_up(lines * sizeof(vkop::LineStats));
    if (sc.ok) {
        l.bmax = off;
        off += align_up(lines * sc.blocks * sizeof(uint32_t));
        l.recs = off;
        off += align_up(lines * sc.g * vkop::kScanWaves * 3 * sizeof(uint64_t));  // (two words a wave, then the waves' third words)
        if (sc.g2 != 0) {
            l.bmin = off;
            off += align_up(lines * sc.blocks * sizeof(uint32_t));
            l.bcand = off;
            off += align_up(lines * vkop::kBigPickLists * vkop::kBigPickListCap * sizeof(uint64_t));
            l.bterm = off;
            off += align_up(lines * vkop::kBigPickLists * vkop::kBigPickListCap * sizeof(float));
            l.bhead = off;
            off += align_up(lines * vkop::kBigPickHeadWords * sizeof(uint32_t));
            l.bstat = off;
            off += align_up(2 * lines * sizeof(double));
        }
    } else if (c.ok) {
        const size_t chunks = lines * c.g;
        l.sums = off;
        off += align_up(chunks * (static_cast<size_t>(c.nt) / 64) * vkop::kRecWords * sizeof(uint64_t));
        l.cand = off;
        off += align_up(chunks * c.cap * sizeof(uint64_t));
    } else if (b.ok) {
        const size_t chunks = lines * b.g;
        l.hist = off;
        l.hist_bytes = align_up(3 * lines * vkop::kBigBins * sizeof(uint32_t));
        off += l.hist_bytes;
        l.state = off;
        off += align_up(lines * 8 * sizeof(uint32_t));
        l.counts = off;
        off += align_up(chunks * 2 * sizeof(uint32_t));
        l.sel = off;
        off += align_up(lines * b.kpad * sizeof(uint64_t));
        l.chunkstats = off;
        off += align_up(chunks * sizeof(vkop::ChunkStat));
    }
    l.total = off;
    return l;
}

template <typename T, bool SOFTMAX>
int launch_bigk(const T *in, T *values, int32_t *indices, const View &v, int k, int largest, const BigKCfg &c, void *ws,
                const RowsLayout &l, hipStream_t st, bool in_order = true) {
    auto *base = static_cast<unsigned char *>(ws);
    vkop::BigKWorkspace w;
    w.hist = reinterpret_cast<uint32_t *>(base + l.hist);
    w.state = reinterpret_cast<uint32_t *>(base + l.state);
    w.counts = reinterpret_cast<uint32_t *>(base + l.counts);
    w.sel = reinterpret_cast<uint64_t *>(base + l.sel);
    auto *stats = reinterpret_cast<vkop::LineStats *>(base + l.stats);
    w.stats = stats;
    w.kpad = c.kpad;
    const uint32_t rows = v.g.outer, n = v.g.n, blocks = rows * c.g;
    const uint32_t flip = largest ? 0u : 0xFFFFFFFFu;
    const uint32_t uk = static_cast<uint32_t>(k);
    const uint32_t vec = 16 / sizeof(T);
    const bool aligned = (reinterpret_cast<uintptr_t>(in) % 16 == 0) && (n % vec == 0);
    constexpr int V = sizeof(T) == 4 ? 8 : 4;
    constexpr int NT = vkop::kBigThreads;
    const size_t words = l.hist_bytes / 4;
    vkop::fill_zero_kernel<<<static_cast<unsigned>((words + 255) / 256), 256, 0, st>>>(w.hist, words);
    auto run = [&](auto al) {
        constexpr bool AL = decltype(al)::value;
        if constexpr (SOFTMAX) {
            auto *cs = reinterpret_cast<vkop::ChunkStat *>(base + l.chunkstats);
            vkop::softmax_stats_kernel<T, NT, V><<<blocks, NT, 0, st>>>(in, cs, n, c.g);
            vkop::bigk_row_stats_kernel<<<rows, vkop::kWave, 0, st>>>(cs, stats, c.g);
        }
        vkop::bigk_hist_kernel<T, V, SOFTMAX, AL, 0><<<blocks, NT, 0, st>>>(in, n, uk, c.g, c.per, flip, w);
        vkop::bigk_hist_kernel<T, V, SOFTMAX, AL, 1><<<blocks, NT, 0, st>>>(in, n, uk, c.g, c.per, flip, w);
        vkop::bigk_hist_kernel<T, V, SOFTMAX, AL, 2><<<blocks, NT, 0, st>>>(in, n, uk, c.g, c.per, flip, w);
        vkop::bigk_count_kernel<T, V, SOFTMAX, AL><<<blocks, NT, 0, st>>>(in, n, c.g, c.per, flip, w);
        vkop::bigk_gather_kernel<T, V, SOFTMAX, AL><<<blocks, NT, 0, st>>>(in, n, uk, c.g, c.per, flip, w);
    };
    if (aligned) run(std::true_type{});
    else run(std::false_type{});
    const uint32_t slices = (uk + vkop::kBigSortSlice - 1) / vkop::kBigSortSlice;
    vkop::bigk_sort_kernel<T, SOFTMAX>
        <<<rows * slices, vkop::kBigSortThreads, 0, st>>>(in, values, indices, n, uk, slices, w, in_order ? 1u : 0u);
    return launched("multi-workgroup radix select");
}

template <typename T, bool SOFTMAX>
int launch_scan(const T *in, T *values, int32_t *indices, const View &v, int k, const ScanCfg &c, void *ws,
                const RowsLayout &l, hipStream_t st, float scale = 1.f, int32_t *counts = nullptr, float top_p = 0.f) {
    auto *base = static_cast<unsigned char *>(ws);
    const uint32_t vec = 16 / sizeof(T);
    vkop::ScanLaunch a;
    a.in = in;
    a.values = values;
    a.indices = indices;
    a.rows = v.g.outer;
    a.n = v.g.n;
    a.k = static_cast<uint32_t>(k);
    a.v = static_cast<uint32_t>(c.v);
    a.g = c.g;
    a.aligned = (reinterpret_cast<uintptr_t>(in) % 16 == 0) && (v.g.n % vec == 0);
    a.stages = measured_stages();
    a.scale = scale;
    a.counts = counts;
    a.top_p = top_p;
    a.ws.bmax = reinterpret_cast<uint32_t *>(base + l.bmax);
    a.ws.recs = reinterpret_cast<uint64_t *>(base + l.recs);
    a.ws.recs2 = a.ws.recs + 2 * static_cast<size_t>(v.g.outer) * c.g * vkop::kScanWaves;
    a.ws.blocks = c.blocks;
    a.ws.bmin = nullptr;
    a.ws.zero = nullptr;
    a.ws.zero_words = 0;
    a.g2 = c.g2;
    a.bw = vkop::BigPickWorkspace{nullptr, nullptr, nullptr, nullptr};
    if (c.g2 != 0) {
        a.bw.cand = reinterpret_cast<uint64_t *>(base + l.bcand);
        a.bw.term = reinterpret_cast<float *>(base + l.bterm);
        a.bw.head = reinterpret_cast<uint32_t *>(base + l.bhead);
        a.bw.stat = reinterpret_cast<double *>(base + l.bstat);
        a.ws.bmin = reinterpret_cast<uint32_t *>(base + l.bmin);
        a.ws.zero = a.bw.head;
        a.ws.zero_words = vkop::kBigPickHeadWords;
    }
    a.stream = st;
    if (!vkop::launch_rows_scan<T, SOFTMAX>(a))
        return fail(VKOP_HIP_ERR_UNSUPPORTED, "no rows_scan_kernel / rows_pick_kernel for %d loads, %u blocks", c.v, c.blocks);
    return launched("rows_scan_kernel / rows_pick_kernel");
}

// Vectors a thread of a workgroup that holds its row: of 512 and 1024 threads, which the plan takes by the places and whose shape
// holds 16384 elements and more, as few as hold this row -- every vector costs its comparisons and counts in every wave, whether
// there are elements in it or not.  us a call, top-k and fused, with eight vectors / these: [16,8400] f32 k = 300 14.5 / 13.4,
// 17.8 / 15.4; [256,8000] k = 300 15.4 / 13.8, 18.6 / 15.8; [64,4000] k = 130 9.5 / 8.8, 11.3 / 9.9; [16,12000] k = 400 13.3 /
// 12.1, 16.2 / 15.0.
int fitted_loads(const RowsCfg &c, uint32_t n, uint32_t vec) {
    if (c.nt < 512 || !c.local() || c.forced) return c.v;
    static const int f32_wide[] = {2, 3, 4}, f32_less[] = {2, 4}, f16[] = {1, 2};
    auto first = [&](const auto &loads) {
        for (const int v : loads)
            if (v < c.v && static_cast<uint64_t>(c.nt) * v * vec >= n) return v;
        return c.v;
    };
    return vec == 8 ? first(f16) : c.nt == 1024 ? first(f32_wide) : first(f32_less);
}

template <typename T, bool SOFTMAX>
int launch_rows(const T *in, T *values, int32_t *indices, const View &v, int k, const RowsCfg &c, void *ws,
                const RowsLayout &l, hipStream_t st, bool sampling = false, float scale = 1.f, int32_t *counts = nullptr,
                float top_p = 0.f) {
    vkop::RowsWorkspace w;
    auto *base = static_cast<unsigned char *>(ws);
    w.tickets = reinterpret_cast<uint32_t *>(base + l.tickets);
    w.sums = reinterpret_cast<uint64_t *>(base + l.sums);
    w.cand = reinterpret_cast<uint64_t *>(base + l.cand);
    w.cap = c.cap;
    w.cap_shift = c.cap_shift;
    const uint32_t vec = 16 / sizeof(T);
    // more rows than arrival counters: the merge runs as a kernel of its own
    const bool by_ticket = g_rows_fused.load() != 0 && v.g.outer <= kTicketRows;
    vkop::RowsLaunch a;
    a.in = in;
    a.values = values;
    a.indices = indices;
    a.rows = v.g.outer;
    a.n = v.g.n;
    a.k = static_cast<uint32_t>(k);
    a.nt = static_cast<uint32_t>(c.nt);
    a.v = static_cast<uint32_t>(c.v);
    a.g = c.g;
    a.per = c.per;
    a.aligned = (reinterpret_cast<uintptr_t>(in) % 16 == 0) && (v.g.n % vec == 0);
    a.merge = c.local() ? vkop::kMergeLocal : (c.g == 1 || by_ticket) ? vkop::kMergeByTicket : vkop::kMergeSplit;
    if (a.merge == vkop::kMergeLocal) {
        // the list is in LDS, where the kernel reserves kLocalCap entries whatever k is: all of them are the
        // list (an overflow -- values equal en masse at the cut -- makes the workgroup list a second time)
        w.cap = static_cast<uint32_t>(vkop::kLocalCap);
        w.cap_shift = 0;
        while ((1u << w.cap_shift) < w.cap) w.cap_shift++;
    }
    if (a.merge == vkop::kMergeLocal && !sampling) {
        a.v = static_cast<uint32_t>(fitted_loads(c, v.g.n, vec));
        a.per = a.nt * a.v * vec;
    }
    a.ws = w;
    a.stream = st;
    a.sampling = sampling;
    a.scale = scale;
    a.counts = counts;
    a.top_p = top_p;
    if (sampling && a.merge != vkop::kMergeLocal) return fail(VKOP_HIP_ERR_UNSUPPORTED, "no scaled form of these kernels for this shape");
    const int stages = a.merge != vkop::kMergeSplit ? 1 : measured_stages();
    if (stages & 1) {
        if (!vkop::launch_rows_chunk<T, SOFTMAX>(a))
            return fail(VKOP_HIP_ERR_UNSUPPORTED, "no rows_chunk_kernel for %d threads x %d loads", c.nt, c.v);
        if (int rc = launched("rows_chunk_kernel")) return rc;
    }
    if constexpr (!vkop::kReversed<T>) {
        if (a.merge == vkop::kMergeSplit && (stages & 2)) {
            vkop::launch_rows_merge<T, SOFTMAX>(a);
            return launched("rows_merge_kernel");
        }
    }
    return VKOP_HIP_OK;
}

// ------------------------------------------------------------------ top-k ----
// Rows that one workgroup of the chunk kernel holds, but that a workgroup's exact select (topk_lines_kernel) ranks sooner.
// (vec: elements a vector.)  The line lies where the two were the same, within 10 % on either side, over 375 shapes of normal rows
// (8 to 30000 of 200 to 20000 elements, f32 and f16, 0.4 to 8 vectors a place, either direction); us a call, chunk kernel / select:
//  * about as many vectors as places, or fewer, whose maxima bound nothing, in rows that the list does not hold whole: [8,1500] f16
//    k = 196 29 / 19, [1500,1500] 167 / 28;
//  * smallest first up to two vectors a place, where the select ran before and its time does not depend on the data, and by the
//    thousand of rows just past what 256 threads hold, where they have too few blocks for the scan (choose_rows_cfg): [3300,8196] k = 23 f16 189 / 124, f32 132 / 121, [3300,10094] f16 191 / 161;
//  * 256 threads, short rows by the thousand, which the select reads again from the cache: [6000,400] f32 k = 44 40 / 30, k = 104
//    52 / 36, [30000,800] f16 k = 104 275 / 207; but [300,400] f32 k = 104 9.3 / 10.8, [1500,800] f16 k = 75 18 / 20;
//  * 512 and 1024 threads, more rows than CUs (a workgroup each at a time) of few elements for so many threads, a line for each of the
//    two (with the vectors fitted, fitted_loads): f32 [1200,1100] k = 240 25 / 18, [6000,1500] k = 130 76 / 66, but [700,1500] k = 130
//    13 / 18, [2500,2200] k = 240 32 / 44, [6000,4000] k = 130 71 / 124; f32 [700,3000] k = 300 36 / 30, [1200,4000] 47 / 44,
//    [6000,5500] 229 / 186, but [450,4000] 20 / 33, [700,4400] 30 / 39, [2500,6400] 98 / 105; f16 [700,3000] k = 300 49 / 38,
//    [2500,5500] 125 / 102, but [450,4000] 27 / 42, [1200,6400] 64 / 71.
bool select_is_faster(const View &v, int k, const RowsCfg &c, uint32_t vec, bool largest) {
    const uint32_t n = v.g.n, rows = v.g.outer;
    if (c.g != 1 || c.nt < 256) return false;
    const uint32_t vectors = (n + vec - 1) / vec, places = static_cast<uint32_t>(k) + 1u;
    if (vectors <= places + places / 16 && n > static_cast<uint32_t>(vkop::kLocalCap)) return true;
    if (!largest && vectors < 2u * places) return true;
    if (!largest && c.nt >= 512 && rows > 1024 && n < (vec == 8 && n % 8 == 0 ? 9000u : 11000u)) return true;
    if (c.nt == 256) return rows >= 1024 && n < (vec == 4 || rows >= 4096 ? 1000u : 600u);
    if (rows <= 256) return false;
    if (c.nt == 512) return rows >= 1000 && n <= 1600;
    return n <= (vec == 4 ? 2000u : 2600u) + std::min(rows, 2000u) * 11u / 5u && n <= (vec == 4 && rows < 4000 ? 5500u : 6500u);
}

template <typename T>
int topk_impl(const T *in, T *values, int32_t *indices, const View &v, int k, int largest, int sorted, int dtype, void *ws,
              size_t ws_bytes, hipStream_t st) {
    // (the one-wave kernel serves both directions: it turns its order keys round)
    if (const int tiny = choose_tiny_loads(v, k, dtype)) return launch_tiny<T, false>(in, values, indices, v, k, tiny, st, !largest);
    // Smallest first runs the kernels of the other direction on reversed elements wherever those are the scan
    // kernels or one workgroup a row (with rows.path = 1, which switches the former off: the radix select): two
    // launches or one for the select's seven, one read of the row for five.  [64,32000] f32 k = 40 41 -> 8.8 us,
    // [64,128256] k = 50 61 -> 12.9, [8,262144] k = 1024 46.8 -> 21.2, [1024,4096] k = 64 29.7 -> 10.2.
    // (2^22 rows and more: a grid of a thousand threads a row is more than HIP takes, the select's is not.)
    const bool routed = largest || (g_rows_path.load() != 1 && v.g.outer < (1u << 22));
    ScanCfg sc = routed ? choose_scan_cfg(v, k, dtype, false, kPlainRows) : ScanCfg{};
    // (without an order, the rows of the large-k kernels keep the select and the listing it has always given)
    if (!largest && !sorted && sc.g2 != 0) sc = ScanCfg{};
    RowsCfg c = (routed && !sc.ok) ? choose_rows_cfg(v, k, dtype, false, false, kPlainRows) : RowsCfg{};
    if (!largest && (c.g != 1 || c.nt < 256 || c.cap > static_cast<uint32_t>(vkop::kLocalCap))) c = RowsCfg{};
    if (c.ok && g_rows_path.load() != 1 && select_is_faster(v, k, c, 16 / sizeof(T), largest != 0)) c = RowsCfg{};
    if (routed && !sc.ok && !c.ok && k > kTwoAndHalfListsMaxK && v.g.outer <= 256 && g_rows_path.load() != 1) {
        // A k that the list holds less than 2.5 times, up to a row a CU.  Such a workgroup keeps everything in LDS: the call takes
        // whatever workspace is given, as the kernels below that need none.  us a call, those below / this, f32: [16,16000] k = 500
        // 30.9 / 13.2, of levels 49 / 19, sorted 28.7 / 25.3; [256,8400] k = 420 25.6 / 12.5, smallest first 25.8 / 12.4; [8,5000]
        // k = 450 18.9 / 11.1; f16 [16,16000] k = 500 44.4 / 13.3; but [300,5000] f32 25.3 / 33.9, [300,9000] f16 42.1 / 44.1.
        const RowsCfg full = choose_rows_cfg(v, k, dtype, false, true, kPlainRows);
        if (full.ok && full.g == 1 && !select_is_faster(v, k, full, 16 / sizeof(T), largest != 0)) {
            const RowsLayout none;
            if (largest) return launch_rows<T, false>(in, values, indices, v, k, full, nullptr, none, st);
            using R = vkop::Reversed<T>;
            return launch_rows<R, false>(reinterpret_cast<const R *>(in), reinterpret_cast<R *>(values), indices, v, k, full, nullptr, none, st);
        }
    }
    const BigKCfg b = (c.ok || sc.ok) ? BigKCfg{} : choose_bigk_cfg(v, k, dtype);
    if (sc.ok || c.ok || b.ok) {
        const RowsLayout l = rows_layout(v, c, b, sc);
        if (ws == nullptr || ws_bytes < l.total)
            return fail(VKOP_HIP_ERR_WORKSPACE, "workspace of %zu bytes given, %zu needed", ws_bytes, l.total);
        if ((reinterpret_cast<uintptr_t>(ws) & (kAlign - 1)) != 0)
            return fail(VKOP_HIP_ERR_WORKSPACE, "workspace must be %zu-byte aligned", kAlign);
        if (sc.ok && largest) return launch_scan<T, false>(in, values, indices, v, k, sc, ws, l, st);
        if (c.ok && largest) return launch_rows<T, false>(in, values, indices, v, k, c, ws, l, st);
        if (sc.ok || c.ok) {
            using R = vkop::Reversed<T>;
            const R *rin = reinterpret_cast<const R *>(in);
            R *rvalues = reinterpret_cast<R *>(values);
            if (sc.ok) return launch_scan<R, false>(rin, rvalues, indices, v, k, sc, ws, l, st);
            return launch_rows<R, false>(rin, rvalues, indices, v, k, c, ws, l, st);
        }
        // (sorted == 0: the one route where an order costs a step of its own leaves it out; every other route's
        // result is in order by construction, which satisfies "any order" too)
        return launch_bigk<T, false>(in, values, indices, v, k, largest, b, ws, l, st, sorted != 0);
    }
    const uint32_t lines = v.g.outer * v.g.inner;
    // one workgroup per line: a big one when the line is long and lines are few
    if (v.g.n >= 4096 && lines <= 1024)
        vkop::topk_lines_kernel<T, 1024><<<lines, 1024, 0, st>>>(in, values, indices, v.g, static_cast<uint32_t>(k), largest);
    else
        vkop::topk_lines_kernel<T, kLineThreads>
            <<<lines, kLineThreads, 0, st>>>(in, values, indices, v.g, static_cast<uint32_t>(k), largest);
    return launched("topk_lines_kernel");
}

// ------------------------------------------------------------------ fused ----
// Which route a fused call takes; the workspace size follows from it.
struct FusedPlan {
    ScanCfg scan;
    RowsCfg rows;
    BigKCfg big;
};
FusedPlan plan_fused(const View &v, int k, int dtype, int largest, bool want_probs) {
    FusedPlan p;
    if (want_probs) return p;  // the softmax tensor is written by the general kernels
    if (largest) p.scan = choose_scan_cfg(v, k, dtype);
    if (largest && !p.scan.ok) p.rows = choose_rows_cfg(v, k, dtype);
    // A k whose places are about as many as a row's vectors, on more rows than CUs or in rows that the list does not hold whole:
    // every row would take the one-workgroup kernel's second list; the general kernels (line statistics, an exact select of probabilities) rank it sooner.  us a call:
    // [300,1500] f32 k = 393 76 / 26, f16 k = 196 62 / 35, [1500,800] f32 k = 209 74 / 27, [8,1500] f32 k = 393 38 / 24; but at
    // 1.3 vectors a place [300,2400] f16 k = 229 30 / 48, and [64,800] f32 k = 209 14 / 18.
    const uint32_t vec = dtype == VKOP_HIP_F32 ? 4u : 8u, places = static_cast<uint32_t>(k) + 1u;
    if (p.rows.ok && g_rows_path.load() != 1 && p.rows.nt >= 512 && p.rows.g == 1 &&
        (v.g.outer > 256 || v.g.n > static_cast<uint32_t>(vkop::kLocalCap)) &&
        (v.g.n + vec - 1) / vec <= places + places / 16)
        p.rows = RowsCfg{};
    if (!p.scan.ok && !p.rows.ok) p.big = choose_bigk_cfg(v, k, dtype);
    return p;
}

template <typename T>
int fused_impl(const T *in, T *probs, T *values, int32_t *indices, const View &v, int k, int largest, int dtype,
               void *ws, hipStream_t st, size_t ws_limit = ~static_cast<size_t>(0)) {
    if (const int tiny = (largest && probs == nullptr) ? choose_tiny_loads(v, k, dtype) : 0)
        return launch_tiny<T, true>(in, values, indices, v, k, tiny, st);
    const FusedPlan p = plan_fused(v, k, dtype, largest, probs != nullptr);
    const RowsLayout l = rows_layout(v, p.rows, p.big, p.scan);
    // (the layout the kernels are given is the one checked here: a tuning change between a caller's
    // size query and this call cannot put it past the end of what the caller holds)
    if (l.total > ws_limit)
        return fail(VKOP_HIP_ERR_WORKSPACE, "this call's scratch layout takes %zu bytes, %zu are there", l.total, ws_limit);
    if (p.scan.ok) return launch_scan<T, true>(in, values, indices, v, k, p.scan, ws, l, st);
    if (p.rows.ok) return launch_rows<T, true>(in, values, indices, v, k, p.rows, ws, l, st);
    if (p.big.ok) return launch_bigk<T, true>(in, values, indices, v, k, largest, p.big, ws, l, st);
    // general path: line statistics (and the softmax tensor when asked for), then
    // an exact select keyed by the probabilities those statistics define
    const uint32_t lines = v.g.outer * v.g.inner;
    auto *stats = reinterpret_cast<vkop::LineStats *>(static_cast<unsigned char *>(ws) + l.stats);
    vkop::softmax_lines_kernel<T, kLineThreads><<<lines, kLineThreads, 0, st>>>(in, probs, v.g, 0, 0.f, stats);
    if (int rc = launched("softmax_lines_kernel")) return rc;
    vkop::softmax_topk_lines_kernel<T, kLineThreads>
        <<<lines, kLineThreads, 0, st>>>(in, stats, values, indices, v.g, static_cast<uint32_t>(k), largest);
    return launched("softmax_topk_lines_kernel");
}

// Workspace that serves whichever route a top-k or fused call on this tensor can
// take (largest or smallest, with or without the softmax tensor).
size_t selection_workspace(const View &v, int k, int dtype) {
    const size_t a = rows_layout(v, choose_rows_cfg(v, k, dtype, true)).total;
    const size_t b = rows_layout(v, RowsCfg{}, choose_bigk_cfg(v, k, dtype)).total;
    const size_t c = rows_layout(v, RowsCfg{}, BigKCfg{}, choose_scan_cfg(v, k, dtype, true)).total;
    return a > b ? (a > c ? a : c) : (b > c ? b : c);
}

// max over `axis` of the softmax along `axis`, without the softmax tensor
template <typename T>
int softmax_reduce_max_impl(const T *in, T *out, const View &v, void *ws, size_t ws_bytes, hipStream_t st) {
    const uint32_t lines = v.g.outer * v.g.inner;
    const SoftmaxPlan p = plan_softmax(v, sizeof(T) == 4 ? VKOP_HIP_F32 : VKOP_HIP_F16);
    if (p.kind == SoftmaxPlan::kLinesRegs) {
        return launch_lines(in, out, v, p, true, 0, 0.f, st);
    }
    if (v.g.inner == 1 && p.kind != SoftmaxPlan::kGeneralLines) return softmax_rows<T, true>(in, out, v, p, 0, 0.f, ws, ws_bytes, st);
    if (p.kind == SoftmaxPlan::kStridedRegs) {
        launch_strided_reg<T, true>(in, out, v, 0, 0.f, st);
        return launched("softmax_strided_reg_kernel");
    }
    if (v.g.inner != 1) {
        // long lines along a non-last axis: the statistics of the tile kernel, as the softmax itself takes them
        const uint32_t tiles = v.g.outer * ((v.g.inner + (1u << p.ti_shift) - 1) >> p.ti_shift);
        if (p.g == 1) {
            vkop::softmax_strided_tile_kernel<T, vkop::kTileWholeMax>
                <<<tiles, vkop::kStridedTileThreads, 0, st>>>(in, out, nullptr, v.g, p.ti_shift, 1, v.g.n, 0, 0.f);
            return launched("softmax_strided_tile_kernel (max)");
        }
        if (ws == nullptr || ws_bytes < p.workspace)
            return fail(VKOP_HIP_ERR_WORKSPACE, "workspace of %zu bytes given, %zu needed", ws_bytes, p.workspace);
        auto *cstats = reinterpret_cast<vkop::ChunkStat *>(static_cast<unsigned char *>(ws) + kTicketBytes);
        vkop::softmax_strided_tile_kernel<T, vkop::kTileStats>
            <<<tiles * p.g, vkop::kStridedTileThreads, 0, st>>>(in, out, cstats, v.g, p.ti_shift, p.g, p.per, 0, 0.f);
        vkop::softmax_strided_tile_kernel<T, vkop::kTileFoldMax>
            <<<tiles * p.g, vkop::kStridedTileThreads, 0, st>>>(in, out, cstats, v.g, p.ti_shift, p.g, p.per, 0, 0.f);
        return launched("softmax_strided_tile_kernel (split, max)");
    }
    // rows of more than 2^25 elements: the line statistics, then exp_accurate(0) / S per line
    const size_t need = kTicketBytes + align_up(static_cast<size_t>(lines) * sizeof(vkop::LineStats));
    if (ws == nullptr || ws_bytes < need)
        return fail(VKOP_HIP_ERR_WORKSPACE, "workspace of %zu bytes given, %zu needed", ws_bytes, need);
    auto *stats = reinterpret_cast<vkop::LineStats *>(static_cast<unsigned char *>(ws) + kTicketBytes);
    vkop::softmax_lines_kernel<T, kLineThreads>
        <<<lines, kLineThreads, 0, st>>>(in, static_cast<T *>(nullptr), v.g, 0, 0.f, stats);
    vkop::stats_to_max_kernel<T><<<(lines + 255) / 256, 256, 0, st>>>(stats, out, lines);
    return launched("softmax_lines_kernel / stats_to_max_kernel");
}

template <typename T> int reduce_max_impl(const T *in, T *out, const View &v, hipStream_t st) {
    const uint32_t lines = v.g.outer * v.g.inner;
    if (v.g.inner == 1) {
        vkop::reduce_max_lines_kernel<T, kLineThreads><<<lines, kLineThreads, 0, st>>>(in, out, v.g);
        return launched("reduce_max_lines_kernel");
    }
    const uint32_t per_block = kLineThreads / 4;  // four lanes per line
    const uint32_t blocks = (lines + per_block - 1) / per_block;
    vkop::reduce_max_strided_kernel<T, kLineThreads><<<blocks, kLineThreads, 0, st>>>(in, out, v.g);
    return launched("reduce_max_strided_kernel");
}

// ---------------------------------------------------------------- nms ----
uint32_t nms_max_sel(int N, int max_per_class) {
    uint32_t m = static_cast<uint32_t>(N) < static_cast<uint32_t>(vkop::kNmsMaxCandidates)
                     ? static_cast<uint32_t>(N) : static_cast<uint32_t>(vkop::kNmsMaxCandidates);
    if (max_per_class > 0 && static_cast<uint32_t>(max_per_class) < m) m = static_cast<uint32_t>(max_per_class);
    return m < 1 ? 1 : m;
}
size_t nms_workspace(int B, int C, int N, int max_per_class) {
    const size_t pairs = static_cast<size_t>(B) * C;
    return kTicketBytes + align_up(2 * pairs * sizeof(uint32_t)) + align_up(pairs * nms_max_sel(N, max_per_class) * sizeof(int32_t));
}
// With the words of the one launch (in a workspace of the size above, without them, a call takes the two, as a recorded one does).
size_t nms_joined_workspace(int B, int C, int N, int max_per_class) {
    const uint64_t pairs = static_cast<uint64_t>(B) * C;
    const size_t two = nms_workspace(B, C, N, max_per_class);
    return pairs > vkop::kNmsHeldNarrow ? two : two + align_up(vkop::nms_words(static_cast<uint32_t>(pairs)) * sizeof(uint64_t));
}

// A tag of the one launch: not 0, and no two of 2^37 calls in a row have the same (N of the golden ratio's multiples lie 2^64 / (sqrt(5) N)
// apart at least, and a tag tells 2^25 apart).  Another process that has had the workspace, or another build of
// the library in this one, starts somewhere else.
uint64_t nms_call_tag() {
    static std::atomic<uint64_t> calls{(static_cast<uint64_t>(std::chrono::system_clock::now().time_since_epoch().count()) ^
                                        reinterpret_cast<uintptr_t>(&g_nms_threads)) * 0xD6E8FEB86659FD93ull};
    return ((calls.fetch_add(1, std::memory_order_relaxed) * 0x9E3779B97F4A7C15ull) >> 24) | 1ull;
}
// Whether calls on the stream are being recorded, or the runtime does not say.
bool recorded(hipStream_t st) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &status) == hipSuccess) return status != hipStreamCaptureStatusNone;
    (void)hipGetLastError();
    return true;
}

template <typename T>
int nms_impl(const T *boxes, const T *scores, int32_t *out, int out_capacity, int32_t *out_count, int B, int C, int N,
             int center_point_box, int max_per_class, float iou_threshold, float score_threshold, void *ws, size_t ws_bytes,
             hipStream_t st) {
    const uint32_t pairs = static_cast<uint32_t>(B) * static_cast<uint32_t>(C);
    auto *base = static_cast<unsigned char *>(ws) + kTicketBytes;
    auto *counts = reinterpret_cast<uint32_t *>(base);
    auto *selected = reinterpret_cast<int32_t *>(base + align_up(2 * static_cast<size_t>(pairs) * sizeof(uint32_t)));
    const uint32_t max_sel = nms_max_sel(N, max_per_class);
    const uint32_t per = max_per_class > 0 ? static_cast<uint32_t>(max_per_class) : 0u;
    const int knob = g_nms_threads;  // 0: by the number of pairs
    const bool narrow = knob > 0 ? knob == vkop::kNmsThreadsNarrow : pairs >= static_cast<uint32_t>(vkop::kNmsNarrowMinPairs);
    const bool one_launch = pairs <= (narrow ? vkop::kNmsHeldNarrow : vkop::kNmsHeldWide) && ws_bytes >= nms_joined_workspace(B, C, N, max_per_class) &&
                            reinterpret_cast<uintptr_t>(ws) % sizeof(uint64_t) == 0 && !recorded(st);
    auto *words = reinterpret_cast<uint64_t *>(static_cast<unsigned char *>(ws) + nms_workspace(B, C, N, max_per_class));
    const vkop::NmsJoined joined{one_launch ? words : nullptr, out, out_count, static_cast<uint32_t>(out_capacity), nms_polls(),
                                 one_launch ? nms_call_tag() : 0u};
#define VKOP_NMS_LAUNCH(NT, WHOLE, JOINED)                                                                                 \
    vkop::nms_kernel<T, NT, WHOLE, JOINED><<<pairs, NT, 0, st>>>(boxes, scores, selected, counts, pairs,                   \
                                                                 static_cast<uint32_t>(C), static_cast<uint32_t>(N),       \
                                                                 center_point_box, per, iou_threshold, score_threshold,    \
                                                                 max_sel, joined)
#define VKOP_NMS_FORM(NT, WHOLE)                            \
    if (one_launch) VKOP_NMS_LAUNCH(NT, WHOLE, true);       \
    else VKOP_NMS_LAUNCH(NT, WHOLE, false)
    if (narrow && N % 4 == 0) {
        VKOP_NMS_FORM(vkop::kNmsThreadsNarrow, true);
    } else if (narrow) {
        VKOP_NMS_FORM(vkop::kNmsThreadsNarrow, false);
    } else if (N % 4 == 0) {
        VKOP_NMS_FORM(vkop::kNmsThreadsWide, true);
    } else {
        VKOP_NMS_FORM(vkop::kNmsThreadsWide, false);
    }
#undef VKOP_NMS_FORM
#undef VKOP_NMS_LAUNCH
    if (int rc = launched("nms_kernel"); rc != VKOP_HIP_OK || one_launch) return rc;
    const uint32_t packers = (pairs + vkop::kNmsPackPairs - 1) / vkop::kNmsPackPairs;
    vkop::nms_pack_kernel<<<packers, 256, 0, st>>>(selected, counts, out, out_count, pairs, static_cast<uint32_t>(C), max_sel,
                                                   static_cast<uint32_t>(out_capacity));
    return launched("nms_pack_kernel");
}

}  // namespace

extern "C" {

const char *vkop_hip_last_error(void) { return g_err; }

int vkop_hip_init(int device) {
    int count = 0;
    VKOP_HIP_TRY(hipGetDeviceCount(&count));
    if (device < 0 || device >= count) return fail(VKOP_HIP_ERR_INVALID, "device %d of %d", device, count);
    VKOP_HIP_TRY(hipSetDevice(device));
    hipDeviceProp_t prop;
    VKOP_HIP_TRY(hipGetDeviceProperties(&prop, device));
    if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0)
        return fail(VKOP_HIP_ERR_UNSUPPORTED, "device %d is %s; this library is built for gfx950 only", device,
                    prop.gcnArchName);
    VKOP_HIP_TRY(hipFree(nullptr));  // force context creation here, not inside the first timed call
    // the address of this device's static scratch, for vkop_hip_softmax_topk_static
    void *sp = nullptr;
    int dev = 0;
    if (int rc = resolve_static_scratch(&sp, &dev)) return rc;
    return VKOP_HIP_OK;
}

int vkop_hip_shutdown(void) {
    VKOP_HIP_TRY(hipDeviceSynchronize());
    return VKOP_HIP_OK;
}

int vkop_hip_device_info(char *name, size_t name_len, int *compute_units, size_t *memory_bytes) {
    int dev = 0;
    VKOP_HIP_TRY(hipGetDevice(&dev));
    hipDeviceProp_t prop;
    VKOP_HIP_TRY(hipGetDeviceProperties(&prop, dev));
    if (name != nullptr && name_len > 0) std::snprintf(name, name_len, "%s (%s)", prop.name, prop.gcnArchName);
    if (compute_units != nullptr) *compute_units = prop.multiProcessorCount;
    if (memory_bytes != nullptr) *memory_bytes = prop.totalGlobalMem;
    return VKOP_HIP_OK;
}

int vkop_hip_malloc(void **ptr, size_t bytes) {
    if (ptr == nullptr) return fail(VKOP_HIP_ERR_INVALID, "ptr is null");
    *ptr = nullptr;
    if (bytes == 0) return VKOP_HIP_OK;
    VKOP_HIP_TRY(hipMalloc(ptr, bytes));
    return VKOP_HIP_OK;
}

int vkop_hip_free(void *ptr) {
    if (ptr == nullptr) return VKOP_HIP_OK;
    VKOP_HIP_TRY(hipFree(ptr));
    return VKOP_HIP_OK;
}

int vkop_hip_memcpy_h2d(void *dst, const void *src, size_t bytes, void *stream) {
    if (bytes == 0) return VKOP_HIP_OK;
    if (dst == nullptr || src == nullptr) return fail(VKOP_HIP_ERR_INVALID, "null pointer in h2d copy");
    VKOP_HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, as_stream(stream)));
    VKOP_HIP_TRY(hipStreamSynchronize(as_stream(stream)));
    return VKOP_HIP_OK;
}

int vkop_hip_memcpy_d2h(void *dst, const void *src, size_t bytes, void *stream) {
    if (bytes == 0) return VKOP_HIP_OK;
    if (dst == nullptr || src == nullptr) return fail(VKOP_HIP_ERR_INVALID, "null pointer in d2h copy");
    VKOP_HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, as_stream(stream)));
    VKOP_HIP_TRY(hipStreamSynchronize(as_stream(stream)));
    return VKOP_HIP_OK;
}

int vkop_hip_memcpy_d2d(void *dst, const void *src, size_t bytes, void *stream) {
    if (bytes == 0) return VKOP_HIP_OK;
    if (dst == nullptr || src == nullptr) return fail(VKOP_HIP_ERR_INVALID, "null pointer in d2d copy");
    VKOP_HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, as_stream(stream)));
    return VKOP_HIP_OK;
}

int vkop_hip_stream_create(void **stream) {
    if (stream == nullptr) return fail(VKOP_HIP_ERR_INVALID, "stream is null");
    hipStream_t s;
    VKOP_HIP_TRY(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));  // default priority
    *stream = s;
    return VKOP_HIP_OK;
}

int vkop_hip_stream_destroy(void *stream) {
    if (stream == nullptr) return VKOP_HIP_OK;
    VKOP_HIP_TRY(hipStreamDestroy(as_stream(stream)));
    return VKOP_HIP_OK;
}

int vkop_hip_stream_sync(void *stream) {
    VKOP_HIP_TRY(hipStreamSynchronize(as_stream(stream)));
    return VKOP_HIP_OK;
}

int vkop_hip_event_create(void **event) {
    if (event == nullptr) return fail(VKOP_HIP_ERR_INVALID, "event is null");
    hipEvent_t e;
    VKOP_HIP_TRY(hipEventCreate(&e));
    *event = e;
    return VKOP_HIP_OK;
}

int vkop_hip_event_destroy(void *event) {
    if (event == nullptr) return VKOP_HIP_OK;
    VKOP_HIP_TRY(hipEventDestroy(static_cast<hipEvent_t>(event)));
    return VKOP_HIP_OK;
}

int vkop_hip_event_record(void *event, void *stream) {
    if (event == nullptr) return fail(VKOP_HIP_ERR_INVALID, "event is null");
    VKOP_HIP_TRY(hipEventRecord(static_cast<hipEvent_t>(event), as_stream(stream)));
    return VKOP_HIP_OK;
}

int vkop_hip_event_sync(void *event) {
    if (event == nullptr) return fail(VKOP_HIP_ERR_INVALID, "event is null");
    VKOP_HIP_TRY(hipEventSynchronize(static_cast<hipEvent_t>(event)));
    return VKOP_HIP_OK;
}

int vkop_hip_stream_wait_event(void *stream, void *event) {
    if (event == nullptr) return fail(VKOP_HIP_ERR_INVALID, "event is null");
    VKOP_HIP_TRY(hipStreamWaitEvent(as_stream(stream), static_cast<hipEvent_t>(event), 0));
    return VKOP_HIP_OK;
}

int vkop_hip_event_elapsed_ms(void *start, void *stop, float *ms) {
    if (start == nullptr || stop == nullptr || ms == nullptr) return fail(VKOP_HIP_ERR_INVALID, "null argument");
    VKOP_HIP_TRY(hipEventElapsedTime(ms, static_cast<hipEvent_t>(start), static_cast<hipEvent_t>(stop)));
    return VKOP_HIP_OK;
}

int vkop_hip_graph_begin(void *stream) {
    if (stream == nullptr) return fail(VKOP_HIP_ERR_INVALID, "recording needs a stream created by vkop_hip_stream_create");
    VKOP_HIP_TRY(hipStreamBeginCapture(as_stream(stream), hipStreamCaptureModeThreadLocal));
    return VKOP_HIP_OK;
}

int vkop_hip_graph_end(void *stream, void **graph) {
    if (stream == nullptr || graph == nullptr) return fail(VKOP_HIP_ERR_INVALID, "null argument");
    *graph = nullptr;
    hipGraph_t g = nullptr;
    VKOP_HIP_TRY(hipStreamEndCapture(as_stream(stream), &g));
    hipGraphExec_t exec = nullptr;
    hipError_t e = hipGraphInstantiate(&exec, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (e != hipSuccess) return fail(VKOP_HIP_ERR_DEVICE, "hipGraphInstantiate: %s", hipGetErrorString(e));
    *graph = exec;
    return VKOP_HIP_OK;
}

int vkop_hip_graph_launch(void *graph, void *stream) {
    if (graph == nullptr) return fail(VKOP_HIP_ERR_INVALID, "graph is null");
    VKOP_HIP_TRY(hipGraphLaunch(static_cast<hipGraphExec_t>(graph), as_stream(stream)));
    return VKOP_HIP_OK;
}

int vkop_hip_graph_destroy(void *graph) {
    if (graph == nullptr) return VKOP_HIP_OK;
    VKOP_HIP_TRY(hipGraphExecDestroy(static_cast<hipGraphExec_t>(graph)));
    return VKOP_HIP_OK;
}

int vkop_hip_workspace_init(void *workspace, size_t bytes, void *stream) {
    if (bytes == 0) return VKOP_HIP_OK;
    if (workspace == nullptr) return fail(VKOP_HIP_ERR_INVALID, "workspace is null");
    if ((reinterpret_cast<uintptr_t>(workspace) & 3u) != 0 || (bytes & 3u) != 0)
        return fail(VKOP_HIP_ERR_INVALID, "workspace address and size must be multiples of 4");
    const size_t words = bytes / 4;
    const unsigned blocks = static_cast<unsigned>((words + 255) / 256);
    vkop::fill_zero_kernel<<<blocks, 256, 0, as_stream(stream)>>>(static_cast<uint32_t *>(workspace), words);
    return launched("fill_zero_kernel");
}

size_t vkop_hip_softmax_workspace_bytes(int dtype, const int *shape, int ndim, int axis) {
    View v;
    if (check_dtype(dtype) || make_view(shape, ndim, axis, &v)) return 0;
    return plan_softmax(v, dtype).workspace;
}

int vkop_hip_softmax(const void *in, void *out, int dtype, const int *shape, int ndim, int axis, int nan_where,
                     float nan_value, void *workspace, size_t workspace_bytes, void *stream) {
    View v;
    if (int rc = check_dtype(dtype)) return rc;
    if (int rc = make_view(shape, ndim, axis, &v)) return rc;
    if (v.elems == 0) return VKOP_HIP_OK;
    if (in == nullptr || out == nullptr) return fail(VKOP_HIP_ERR_INVALID, "null tensor pointer");
    if (dtype == VKOP_HIP_F32)
        return softmax_impl(static_cast<const float *>(in), static_cast<float *>(out), v, dtype, nan_where, nan_value,
                            workspace, workspace_bytes, as_stream(stream));
    return softmax_impl(static_cast<const uint16_t *>(in), static_cast<uint16_t *>(out), v, dtype, nan_where,
                        nan_value, workspace, workspace_bytes, as_stream(stream));
}

size_t vkop_hip_topk_workspace_bytes(int dtype, const int *shape, int ndim, int axis, int k) {
    View v;
    if (check_dtype(dtype) || make_view(shape, ndim, axis, &v) || k < 1) return 0;
    return selection_workspace(v, k, dtype);
}

int vkop_hip_topk(const void *in, void *out_values, int32_t *out_indices, int dtype, const int *shape, int ndim,
                  int axis, int k, int largest, int sorted, void *workspace, size_t workspace_bytes, void *stream) {
    View v;
    if (int rc = check_dtype(dtype)) return rc;
    if (int rc = make_view(shape, ndim, axis, &v)) return rc;
    if (v.elems == 0 && k == 0) return VKOP_HIP_OK;
    if (int rc = check_k(v, k)) return rc;
    if (v.g.outer == 0 || v.g.inner == 0) return VKOP_HIP_OK;
    if (in == nullptr || out_values == nullptr || out_indices == nullptr)
        return fail(VKOP_HIP_ERR_INVALID, "null tensor pointer");
    if (dtype == VKOP_HIP_F32)
        return topk_impl(static_cast<const float *>(in), static_cast<float *>(out_values), out_indices, v, k, largest,
                         sorted, dtype, workspace, workspace_bytes, as_stream(stream));
    return topk_impl(static_cast<const uint16_t *>(in), static_cast<uint16_t *>(out_values), out_indices, v, k,
                     largest, sorted, dtype, workspace, workspace_bytes, as_stream(stream));
}

size_t vkop_hip_softmax_topk_workspace_bytes(int dtype, const int *shape, int ndim, int axis, int k) {
    View v;
    if (check_dtype(dtype) || make_view(shape, ndim, axis, &v) || k < 1) return 0;
    return selection_workspace(v, k, dtype);
}

int vkop_hip_softmax_topk(const void *in, void *out_probs, void *out_values, int32_t *out_indices, int dtype,
                          const int *shape, int ndim, int axis, int k, int largest, void *workspace,
                          size_t workspace_bytes, void *stream) {
    View v;
    if (int rc = check_dtype(dtype)) return rc;
    if (int rc = make_view(shape, ndim, axis, &v)) return rc;
    if (v.elems == 0 && k == 0) return VKOP_HIP_OK;
    if (int rc = check_k(v, k)) return rc;
    if (v.g.outer == 0 || v.g.inner == 0) return VKOP_HIP_OK;
    if (in == nullptr || out_values == nullptr || out_indices == nullptr)
        return fail(VKOP_HIP_ERR_INVALID, "null tensor pointer");
    const FusedPlan plan = plan_fused(v, k, dtype, largest, out_probs != nullptr);
    const size_t need = rows_layout(v, plan.rows, plan.big, plan.scan).total;
    if (workspace == nullptr || workspace_bytes < need)
        return fail(VKOP_HIP_ERR_WORKSPACE, "workspace of %zu bytes given, %zu needed", workspace_bytes, need);
    if ((reinterpret_cast<uintptr_t>(workspace) & (kAlign - 1)) != 0)
        return fail(VKOP_HIP_ERR_WORKSPACE, "workspace must be %zu-byte aligned", kAlign);
    if (dtype == VKOP_HIP_F32)
        return fused_impl(static_cast<const float *>(in), static_cast<float *>(out_probs),
                          static_cast<float *>(out_values), out_indices, v, k, largest, dtype, workspace,
                          as_stream(stream), workspace_bytes);
    return fused_impl(static_cast<const uint16_t *>(in), static_cast<uint16_t *>(out_probs),
                      static_cast<uint16_t *>(out_values), out_indices, v, k, largest, dtype, workspace,
                      as_stream(stream), workspace_bytes);
}

int vkop_hip_softmax_topk_sampling(const void *in, void *out_values, int32_t *out_indices, int32_t *out_counts, int dtype,
                                   const int *shape, int ndim, int axis, int k, float scale, float top_p, void *workspace,
                                   size_t workspace_bytes, void *stream) {
    View v;
    if (int rc = check_dtype(dtype)) return rc;
    if (int rc = make_view(shape, ndim, axis, &v)) return rc;
    if (!(scale > 0.f) || !(scale < INFINITY)) return fail(VKOP_HIP_ERR_INVALID, "scale must be positive and finite");
    if (v.elems == 0 && k == 0) return VKOP_HIP_OK;
    if (int rc = check_k(v, k)) return rc;
    if (v.g.outer == 0 || v.g.inner == 0) return VKOP_HIP_OK;
    if (in == nullptr || out_values == nullptr || out_indices == nullptr)
        return fail(VKOP_HIP_ERR_INVALID, "null tensor pointer");
    if (out_counts != nullptr && v.g.inner != 1)
        return fail(VKOP_HIP_ERR_UNSUPPORTED, "the nucleus count is defined along the last axis only");
    const size_t need = selection_workspace(v, k, dtype);
    if (workspace == nullptr || workspace_bytes < need)
        return fail(VKOP_HIP_ERR_WORKSPACE, "workspace of %zu bytes given, %zu needed", workspace_bytes, need);
    if ((reinterpret_cast<uintptr_t>(workspace) & (kAlign - 1)) != 0)
        return fail(VKOP_HIP_ERR_WORKSPACE, "workspace must be %zu-byte aligned", kAlign);
    const hipStream_t st = as_stream(stream);
    const ScanCfg sc = choose_scan_cfg(v, k, dtype, false, kScaledRows);
    auto run = [&](auto tag) -> int {
        using T = decltype(tag);
        const T *x = static_cast<const T *>(in);
        T *values = static_cast<T *>(out_values);
        if (sc.ok && sc.g2 == 0) {
            const RowsLayout l = rows_layout(v, RowsCfg{}, BigKCfg{}, sc);
            return launch_scan<T, true>(x, values, out_indices, v, k, sc, workspace, l, st, scale, out_counts, top_p);
        }
        // short rows and a small k: one wave per row, in the scaled form
        if (const int tiny = choose_tiny_loads(v, k, dtype))
            return launch_tiny<T, true>(x, values, out_indices, v, k, tiny, st, false, true, scale, out_counts, top_p);
        // a row that one workgroup holds: its kernel in the scaled form
        if (!sc.ok) {
            const RowsCfg rc = choose_rows_cfg(v, k, dtype, false, false, kScaledRows);
            if (rc.ok && rc.g == 1 && rows_cap(k) <= static_cast<uint32_t>(vkop::kLocalCap) && g_rows_fused.load() == 0) {
                const RowsLayout lr = rows_layout(v, rc);
                return launch_rows<T, true>(x, values, out_indices, v, k, rc, workspace, lr, st, true, scale, out_counts, top_p);
            }
        }
        // every other shape: the line kernels on the scaled elements, then the count on their sorted result
        const RowsLayout l = rows_layout(v, RowsCfg{}, BigKCfg{});
        const uint32_t lines = v.g.outer * v.g.inner;
        auto *stats = reinterpret_cast<vkop::LineStats *>(static_cast<unsigned char *>(workspace) + l.stats);
        vkop::softmax_lines_kernel<T, kLineThreads>
            <<<lines, kLineThreads, 0, st>>>(x, static_cast<T *>(nullptr), v.g, 0, 0.f, stats, scale);
        vkop::softmax_topk_lines_kernel<T, kLineThreads>
            <<<lines, kLineThreads, 0, st>>>(x, stats, values, out_indices, v.g, static_cast<uint32_t>(k), 1, scale);
        if (out_counts != nullptr)
            vkop::topp_count_kernel<T><<<lines, vkop::kWave, 0, st>>>(values, out_counts, static_cast<uint32_t>(k),
                                                                      static_cast<size_t>(k), top_p);
        return launched("softmax_lines_kernel / softmax_topk_lines_kernel / topp_count_kernel");
    };
    if (dtype == VKOP_HIP_F32) return run(float{});
    return run(uint16_t{});
}

int vkop_hip_softmax_topk_static(const void *in, void *out_values, int32_t *out_indices, int dtype, const int *shape,
                                 int ndim, int axis, int k, int largest, void *stream) {
    View v;
    if (int rc = check_dtype(dtype)) return rc;
    if (int rc = make_view(shape, ndim, axis, &v)) return rc;
    if (v.elems == 0 && k == 0) return VKOP_HIP_OK;
    if (int rc = check_k(v, k)) return rc;
    if (v.g.outer == 0 || v.g.inner == 0) return VKOP_HIP_OK;
    if (in == nullptr || out_values == nullptr || out_indices == nullptr)
        return fail(VKOP_HIP_ERR_INVALID, "null tensor pointer");
    const FusedPlan plan = plan_fused(v, k, dtype, largest, false);
    const size_t need = rows_layout(v, plan.rows, plan.big, plan.scan).total;
    if (need > static_cast<size_t>(VKOP_HIP_STATIC_SCRATCH_BYTES))
        return fail(VKOP_HIP_ERR_WORKSPACE,
                    "this tensor needs %zu bytes of scratch, the static array holds %zu: use vkop_hip_softmax_topk with a workspace",
                    need, static_cast<size_t>(VKOP_HIP_STATIC_SCRATCH_BYTES));
    void *sp = nullptr;
    int dev = 0;
    {
        // the stream belongs to the current device (each device has its own copy of the array), and the
        // array's address is looked up outside a recording (vkop_hip_init does it)
        int cur = 0;
        VKOP_HIP_TRY(hipGetDevice(&cur));
        if (stream != nullptr) {
            int sdev = cur;
            VKOP_HIP_TRY(hipStreamGetDevice(as_stream(stream), &sdev));
            if (sdev != cur)
                return fail(VKOP_HIP_ERR_INVALID, "the stream belongs to device %d, the current device is %d", sdev, cur);
        }
        if (cur >= 0 && cur < kMaxDevices && g_scratch_ptr[cur].load(std::memory_order_acquire) == nullptr) {
            hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
            VKOP_HIP_TRY(hipStreamIsCapturing(as_stream(stream), &cs));
            if (cs != hipStreamCaptureStatusNone)
                return fail(VKOP_HIP_ERR_INVALID, "the static scratch of device %d is not resolved yet and the stream is recording: "
                                                  "call vkop_hip_init(%d) before recording", cur, cur);
        }
    }
    if (int rc = resolve_static_scratch(&sp, &dev)) return rc;
    // The array keeps what the last call left.  All a call needs to find at zero
    // are the per-row arrival counters, which every call that completes returns
    // to zero; after a call that failed half way they are cleared here (a fill
    // kernel, not a memset, so that the call may be recorded).
    if (g_scratch_dirty[dev].exchange(0) != 0) {
        const size_t words = kTicketBytes / 4;
        vkop::fill_zero_kernel<<<static_cast<unsigned>((words + 255) / 256), 256, 0, as_stream(stream)>>>(
            static_cast<uint32_t *>(sp), words);
        if (int rc = launched("fill_zero_kernel")) {
            g_scratch_dirty[dev].store(1);
            return rc;
        }
    }
    int rc;
    if (dtype == VKOP_HIP_F32)
        rc = fused_impl(static_cast<const float *>(in), static_cast<float *>(nullptr), static_cast<float *>(out_values),
                        out_indices, v, k, largest, dtype, sp, as_stream(stream), static_cast<size_t>(VKOP_HIP_STATIC_SCRATCH_BYTES));
    else
        rc = fused_impl(static_cast<const uint16_t *>(in), static_cast<uint16_t *>(nullptr),
                        static_cast<uint16_t *>(out_values), out_indices, v, k, largest, dtype, sp, as_stream(stream),
                        static_cast<size_t>(VKOP_HIP_STATIC_SCRATCH_BYTES));
    if (rc != VKOP_HIP_OK) g_scratch_dirty[dev].store(1);
    return rc;
}

int vkop_hip_reduce_max(const void *in, void *out, int dtype, const int *shape, int ndim, int axis, void *stream) {
    View v;
    if (int rc = check_dtype(dtype)) return rc;
    if (int rc = make_view(shape, ndim, axis, &v)) return rc;
    if (v.g.outer == 0 || v.g.inner == 0) return VKOP_HIP_OK;
    if (v.g.n == 0) return fail(VKOP_HIP_ERR_INVALID, "max over an empty axis");
    if (in == nullptr || out == nullptr) return fail(VKOP_HIP_ERR_INVALID, "null tensor pointer");
    if (dtype == VKOP_HIP_F32)
        return reduce_max_impl(static_cast<const float *>(in), static_cast<float *>(out), v, as_stream(stream));
    return reduce_max_impl(static_cast<const uint16_t *>(in), static_cast<uint16_t *>(out), v, as_stream(stream));
}

int vkop_hip_topp_count(const void *values, int32_t *counts, int dtype, int rows, int k, int row_stride, float p, void *stream) {
    if (int rc = check_dtype(dtype)) return rc;
    if (rows < 0 || k < 1 || row_stride < k) return fail(VKOP_HIP_ERR_INVALID, "rows %d, k %d, row stride %d", rows, k, row_stride);
    if (rows == 0) return VKOP_HIP_OK;
    if (values == nullptr || counts == nullptr) return fail(VKOP_HIP_ERR_INVALID, "null tensor pointer");
    if (dtype == VKOP_HIP_F32)
        vkop::topp_count_kernel<float><<<rows, vkop::kWave, 0, as_stream(stream)>>>(static_cast<const float *>(values), counts,
                                                                                static_cast<uint32_t>(k), static_cast<size_t>(row_stride), p);
    else
        vkop::topp_count_kernel<uint16_t><<<rows, vkop::kWave, 0, as_stream(stream)>>>(static_cast<const uint16_t *>(values), counts,
                                                                                   static_cast<uint32_t>(k), static_cast<size_t>(row_stride), p);
    return launched("topp_count_kernel");
}

int vkop_hip_tune(const char *name, int value) {
    if (name == nullptr) return fail(VKOP_HIP_ERR_INVALID, "name is null");
    if (std::strcmp(name, "rows.threads") == 0) g_rows_threads = value;
    else if (std::strcmp(name, "rows.loads") == 0) g_rows_loads = value;
    else if (std::strcmp(name, "rows.chunks") == 0) g_rows_chunks = value;
    else if (std::strcmp(name, "rows.fused") == 0) g_rows_fused = value != 0;
    else if (std::strcmp(name, "rows.path") == 0) {
        if (value != 0 && value != 1) return fail(VKOP_HIP_ERR_INVALID, "rows.path must be 0 or 1");
        g_rows_path = value;
    }
    else if (std::strcmp(name, "nms.threads") == 0) {
        if (value != 0 && value != vkop::kNmsThreadsNarrow && value != vkop::kNmsThreadsWide)
            return fail(VKOP_HIP_ERR_INVALID, "nms.threads must be 0, %d or %d", vkop::kNmsThreadsNarrow, vkop::kNmsThreadsWide);
        g_nms_threads = value;
    }
    else return fail(VKOP_HIP_ERR_INVALID, "unknown tuning name '%s'", name);
    return VKOP_HIP_OK;
}

int vkop_hip_measure_path(int dtype, const int *shape, int ndim, int axis, int k) {
    View v;
    if (check_dtype(dtype) || make_view(shape, ndim, axis, &v) || k < 1) return -1;
    if (choose_tiny_loads(v, k, dtype) != 0) return 4;
    const ScanCfg sc = choose_scan_cfg(v, k, dtype);
    if (sc.ok) return sc.g2 != 0 ? 3 : 2;
    if (plan_fused(v, k, dtype, 1, false).rows.ok) return 1;
    return 0;
}

#ifdef VKOP_BENCH_HOOKS
int vkop_hip_measure_stages(int stages) {
    if (stages < 1 || stages > 3) return fail(VKOP_HIP_ERR_INVALID, "stages must be 1, 2 or 3");
    g_rows_stages = stages;
    return VKOP_HIP_OK;
}

int vkop_hip_measure_polls(int polls) {
    if (polls < 0) return fail(VKOP_HIP_ERR_INVALID, "polls must not be negative");
    g_joined_polls = static_cast<uint32_t>(polls);
    return VKOP_HIP_OK;
}

int vkop_hip_measure_tags(unsigned first, unsigned count, unsigned *tags) {
    if (tags == nullptr) return fail(VKOP_HIP_ERR_INVALID, "tags is null");
    for (size_t i = 0; i < count; i++)
        for (int w = 0; w < vkop::kJoinedWords; w++)
            tags[i * vkop::kJoinedWords + w] = vkop::word_tag(vkop::launch_tag(first + static_cast<unsigned>(i)), w);
    return VKOP_HIP_OK;
}
#endif

int vkop_hip_rows_plan(int dtype, const int *shape, int ndim, int axis, int k, int *threads, int *loads,
                       int *chunks) {
    View v;
    if (int rc = check_dtype(dtype)) return rc;
    if (int rc = make_view(shape, ndim, axis, &v)) return rc;
    if (const int tiny = choose_tiny_loads(v, k, dtype)) {
        if (threads != nullptr) *threads = vkop::kWave;
        if (loads != nullptr) *loads = tiny;
        if (chunks != nullptr) *chunks = 1;
        return VKOP_HIP_OK;
    }
    const ScanCfg sc = k >= 1 ? choose_scan_cfg(v, k, dtype) : ScanCfg{};
    if (sc.ok) {
        if (threads != nullptr) *threads = vkop::kScanThreads;
        if (loads != nullptr) *loads = sc.v;
        if (chunks != nullptr) *chunks = static_cast<int>(sc.g);
        return VKOP_HIP_OK;
    }
    const RowsCfg c = k >= 1 ? plan_fused(v, k, dtype, 1, false).rows : RowsCfg{};
    if (threads != nullptr) *threads = c.ok ? c.nt : 0;
    if (loads != nullptr) *loads = c.ok ? fitted_loads(c, v.g.n, dtype == VKOP_HIP_F32 ? 4u : 8u) : 0;
    if (chunks != nullptr) *chunks = c.ok ? static_cast<int>(c.g) : 0;
    return VKOP_HIP_OK;
}

size_t vkop_hip_softmax_reduce_max_workspace_bytes(int dtype, const int *shape, int ndim, int axis) {
    View v;
    if (check_dtype(dtype) || make_view(shape, ndim, axis, &v)) return 0;
    if (v.elems == 0) return 0;
    const SoftmaxPlan p = plan_softmax(v, dtype);
    if (p.kind != SoftmaxPlan::kGeneralLines) return p.workspace;
    return kTicketBytes + align_up(static_cast<size_t>(v.g.outer) * sizeof(vkop::LineStats));
}

int vkop_hip_softmax_reduce_max(const void *in, void *out, int dtype, const int *shape, int ndim, int axis,
                                void *workspace, size_t workspace_bytes, void *stream) {
    View v;
    if (int rc = check_dtype(dtype)) return rc;
    if (int rc = make_view(shape, ndim, axis, &v)) return rc;
    if (v.g.outer == 0 || v.g.inner == 0) return VKOP_HIP_OK;
    if (v.g.n == 0) return fail(VKOP_HIP_ERR_INVALID, "max over an empty axis");
    if (in == nullptr || out == nullptr) return fail(VKOP_HIP_ERR_INVALID, "null tensor pointer");
    if (dtype == VKOP_HIP_F32)
        return softmax_reduce_max_impl(static_cast<const float *>(in), static_cast<float *>(out), v, workspace,
                                       workspace_bytes, as_stream(stream));
    return softmax_reduce_max_impl(static_cast<const uint16_t *>(in), static_cast<uint16_t *>(out), v, workspace,
                                   workspace_bytes, as_stream(stream));
}

size_t vkop_hip_nms_workspace_bytes(int B, int C, int N, int max_output_boxes_per_class) {
    if (B < 0 || C < 0 || N < 0) return 0;
    return nms_joined_workspace(B, C, N, max_output_boxes_per_class);
}

int vkop_hip_nms(const void *boxes, const void *scores, int32_t *out, int out_capacity, int32_t *out_count, int dtype, int B,
                 int C, int N, int center_point_box, int max_output_boxes_per_class, float iou_threshold,
                 float score_threshold, void *workspace, size_t workspace_bytes, void *stream) {
    if (int rc = check_dtype(dtype)) return rc;
    if (B < 0 || C < 0 || N < 0 || out_capacity < 0) return fail(VKOP_HIP_ERR_INVALID, "negative extent");
    if (static_cast<uint64_t>(B) * static_cast<uint64_t>(C) >= (1ull << 31) || static_cast<uint64_t>(N) >= (1ull << 31) / 4)
        return fail(VKOP_HIP_ERR_UNSUPPORTED, "too many (batch, class) pairs or boxes");
    if (out_count == nullptr) return fail(VKOP_HIP_ERR_INVALID, "out_count is null");
    if (B == 0 || C == 0) {
        vkop::fill_zero_kernel<<<1, 64, 0, as_stream(stream)>>>(reinterpret_cast<uint32_t *>(out_count), 2);  // (no memset: capture-safe)
        return launched("fill_zero_kernel");
    }
    if (boxes == nullptr || scores == nullptr || (out == nullptr && out_capacity > 0))
        return fail(VKOP_HIP_ERR_INVALID, "null tensor pointer");
    const size_t need = nms_workspace(B, C, N, max_output_boxes_per_class);
    if (workspace == nullptr || workspace_bytes < need)
        return fail(VKOP_HIP_ERR_WORKSPACE, "workspace of %zu bytes given, %zu needed", workspace_bytes, need);
    if ((reinterpret_cast<uintptr_t>(workspace) & (kAlign - 1)) != 0)
        return fail(VKOP_HIP_ERR_WORKSPACE, "workspace must be %zu-byte aligned", kAlign);
    if (dtype == VKOP_HIP_F32)
        return nms_impl(static_cast<const float *>(boxes), static_cast<const float *>(scores), out, out_capacity, out_count,
                        B, C, N, center_point_box, max_output_boxes_per_class, iou_threshold, score_threshold, workspace,
                        workspace_bytes, as_stream(stream));
    return nms_impl(static_cast<const uint16_t *>(boxes), static_cast<const uint16_t *>(scores), out, out_capacity, out_count,
                    B, C, N, center_point_box, max_output_boxes_per_class, iou_threshold, score_threshold, workspace,
                    workspace_bytes, as_stream(stream));
}

}  // extern "C"
