// Throughput kernels for the plain softmax operator.
//
// Contiguous rows (the reduced axis is the last one):
//   softmax_group_kernel    rows of up to a wave's registers: 8 to 64 lanes a row.
//   softmax_row_kernel      one workgroup holds a whole row in registers: one
//                           read, one write.
//   softmax_stats_kernel +  long rows, or too few rows to fill the chip: a row
//   softmax_scale_kernel    is split into chunks, one workgroup each.  The first
//                           kernel leaves (maximum, sum of exp(x - maximum)) per
//                           chunk, the second combines a row's chunk results and
//                           writes exp(x - M) / S for its chunk.  The second
//                           read of the input comes from the Infinity Cache for
//                           tensors that fit it.  (Most such tensors: both in
//                           one launch and one read, kernels_joined.hpp.)
//   softmax_thread_kernel   rows of fewer elements than a vector.
//   (each also without the tensor: the row's largest probability alone, from the same sum)
// Strided lines (another axis, long lines):
//   softmax_strided_tile_kernel  a tile of up to 64 neighbouring lines per workgroup of 16 waves,
//                           rows dealt to the waves, three passes over the tile; with few
//                           tiles, the tile's rows split over several workgroups (two launches).
// Strided lines (another axis, short lines):
//   softmax_strided_reg_kernel  one thread per line, threads along the
//                           contiguous inner axis; the line's elements stay in
//                           registers, so the input is read once.
// All of them produce what kernels_general.hpp defines: terms exp_accurate(x - M),
// the sum in double, one rounding of term * (1 / sum).  The chunked variants sum
// hardware-exp terms (argument scaled with a two-part log2 e, so the scaling adds
// no bias); the sum's relative error of ~1e-8 is far below a float ulp.
#pragma once

#include "device_utils.hpp"
#include "kernels_general.hpp"
#include "kernels_rows.hpp"

namespace vkop {

// exp(x - m) on the hardware unit with an unbiased argument: (x - m) * log2 e
// evaluated with log2 e split in two floats.
__device__ __forceinline__ float fast_term_unbiased(float x, float m) {
    const float d = x - m;
    constexpr float kHi = 1.44269502162933349609375f;    // float(log2 e)
    constexpr float kLo = 1.925963033500011e-8f;         // log2 e - kHi
    return __builtin_amdgcn_exp2f(fmaf(d, kHi, d * kLo));
}

struct ChunkStat {
    double s;       // sum of exp(x - ref) over the chunk (softmax_stats_kernel: without the copies of its minimum)
    float m;        // maximum of the chunk (NaN ignored; -inf for an empty chunk)
    float ref;      // reference of the sum: m, or 0 when m is not finite
    float vmin;     // the value whose copies the sum leaves out (softmax_stats_kernel: the chunk's minimum; the
                    // strided tiles: the line's first element in the chunk) ...
    uint32_t nmin;  // ... and how many elements equal it (0: none set apart)
};

// ---- short rows, many of them: G lanes a row, 128-bit loads ---------------------------------
// Rows of VEC to 64 * V * VEC elements, at any alignment.  G lanes of a wave share a row (64 / G
// rows a wave), lane l of them holds vectors l, l + G, ..., V of them; maximum and sum cross the G
// lanes without LDS or a barrier.  A row that is no whole number of vectors has its last vector
// moved back to end with the row: the elements it shares with the vector before are loaded twice,
// left out of the sum once, and stored twice with the same bits (the launch makes every slot but a
// lane's last a full vector: (V - 1) * G * VEC < n).
// What bounds it is the memory system, once the arithmetic is out of its way: large tensors' loads and stores are
// non-temporal (CACHE: softmax_caching), halves' terms have the fewest instructions (below: half_minus, half2_of_products), NaN shows
// in the row's maximum instead of in every term, a thread keeps few vectors, and a wave takes its rows and ends -- a loop over rows
// with the next one's loads in flight, the form before, copies at 4.8 to 5.7 TB/s where waves that
// end copy at 6.2 to 6.6.  [524288,1024] f16 422 -> 343 us (6.3 TB/s), f32 827 -> 728; [302592,197]
// f16 83 -> 48 us (element by element before), f32 133 -> 102 -> 84; [65536,64] f32 13.7 -> 7.2 us; with ordinary accesses
// [165000,50] f32 19.7 -> 12.6, [300000,100] f32 64 -> 43.  By the terms f16 [304568,197] 48.4 -> 43.8, [83756,197] 14.9 -> 12.9,
// [2441,8192] 14.1 -> 13.1, [8,1000,8000] axis 1 73 -> 68, f32 [64,128256] 15.7 -> 15.2.
template <int CTRL> __device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
    return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), CTRL, 0xF, 0xF, true));
}
template <int G, typename F> __device__ __forceinline__ uint32_t group_join(uint32_t v, F op) {
    static_assert(G >= 8 && G <= kWave, "lanes a row");
    v = op(v, dpp_u32<0xB1>(v));   // lane ^ 1
    v = op(v, dpp_u32<0x4E>(v));   // lane ^ 2
    v = op(v, dpp_u32<0x141>(v));  // the other four of eight
    if constexpr (G >= 16) v = op(v, dpp_u32<0x140>(v));  // the other eight of sixteen
    if constexpr (G >= 32) {
        const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
        v = op(r[0], r[1]);
    }
    if constexpr (G >= 64) {
        const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
        v = op(r[0], r[1]);
    }
    return v;
}
template <int G> __device__ __forceinline__ float group_max(float v) {
    return __uint_as_float(group_join<G>(__float_as_uint(v), [](uint32_t a, uint32_t b) { return __float_as_uint(fmaxf(__uint_as_float(a), __uint_as_float(b))); }));
}
// (NaN where a lane has NaN)
template <int G> __device__ __forceinline__ float group_maximum(float v) {
    return __uint_as_float(group_join<G>(__float_as_uint(v), [](uint32_t a, uint32_t b) { return __float_as_uint(maximum(__uint_as_float(a), __uint_as_float(b), __uint_as_float(b))); }));
}
template <int G> __device__ __forceinline__ double group_sum(double v) {
    auto join = [](uint32_t lo, uint32_t hi) { return __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(hi) << 32) | lo)); };
    auto step = [&](double a, auto tag) {
        constexpr int ctrl = decltype(tag)::value;
        const uint64_t u = static_cast<uint64_t>(__double_as_longlong(a));
        return a + join(dpp_u32<ctrl>(static_cast<uint32_t>(u)), dpp_u32<ctrl>(static_cast<uint32_t>(u >> 32)));
    };
    v = step(v, std::integral_constant<int, 0xB1>{});
    v = step(v, std::integral_constant<int, 0x4E>{});
    v = step(v, std::integral_constant<int, 0x141>{});
    if constexpr (G >= 16) v = step(v, std::integral_constant<int, 0x140>{});
    if constexpr (G >= 32) {
        const uint64_t u = static_cast<uint64_t>(__double_as_longlong(v));
        const auto lo = __builtin_amdgcn_permlane16_swap(static_cast<uint32_t>(u), static_cast<uint32_t>(u), false, false);
        const auto hi = __builtin_amdgcn_permlane16_swap(static_cast<uint32_t>(u >> 32), static_cast<uint32_t>(u >> 32), false, false);
        v = join(lo[0], hi[0]) + join(lo[1], hi[1]);
    }
    if constexpr (G >= 64) {
        const uint64_t u = static_cast<uint64_t>(__double_as_longlong(v));
        const auto lo = __builtin_amdgcn_permlane32_swap(static_cast<uint32_t>(u), static_cast<uint32_t>(u), false, false);
        const auto hi = __builtin_amdgcn_permlane32_swap(static_cast<uint32_t>(u >> 32), static_cast<uint32_t>(u >> 32), false, false);
        v = join(lo[0], hi[0]) + join(lo[1], hi[1]);
    }
    return v;
}
// 1 / s for a row's sum (1 <= s < 2^32, or NaN): the hardware reciprocal (about 2^-22) and two Newton steps, the second of
// which rounds once from a residual that is exact to 2^-84: the quotient a division gives, in half its instructions, which a
// wave of short rows pays once per handful of elements (none of 2.7e8 sums over that range differed).
__device__ __forceinline__ double reciprocal_of_sum(double s) {
    double y = __builtin_amdgcn_rcp(s);
    y = fma(fma(-s, y, 1.0), y, y);
    return fma(fma(-s, y, 1.0), y, y);
}
// 1 / s where the row's maximum m is a number; NaN, which every probability then is, where an element is NaN or the maximum infinite.
__device__ __forceinline__ double row_reciprocal(double s, float m) {
    return reciprocal_of_sum(m > -INFINITY && m < INFINITY ? s : __longlong_as_double(0x7FF8000000000000ll));
}
// The term of element c of a vector, softmax_term_as without its step for NaN: where the row's maximum or sum makes NaN of all.
__device__ __forceinline__ float term_of_row(const Vec128<float> &q, int c, float m) { return exp_accurate<false>(q.get(c) - m); }
__device__ __forceinline__ float term_of_row(const Vec128<uint16_t> &q, int c, float m) {
    return exp_half_grade<false>(half_minus(c < 2 ? q.v.x : c < 4 ? q.v.y : c < 6 ? q.v.z : q.v.w, c & 1, m));
}
// A vector of probabilities as they are stored, the term of element c over the sum that over(c) stands for.
template <typename T, typename F>
__device__ __forceinline__ Vec128<T> probabilities(const float (&e)[Vec128<T>::N], F &&over, int nan_where, float nan_value) {
    Vec128<T> r;
    if constexpr (sizeof(T) == 2) {
        auto pair = [&](int c) { return half2_of_products(e[c], over(c).high, e[c + 1], over(c + 1).high); };
        r.v = make_uint4(pair(0), pair(2), pair(4), pair(6));
    } else {
        r.v = make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int c = 0; c < Vec128<T>::N; c++) r.set(c, over(c)(e[c]));
    }
    if (nan_where) {  // (the same in every thread)
#pragma unroll
        for (int c = 0; c < Vec128<T>::N; c++) {
            const float p = r.get(c);
            if (p != p) r.set(c, nan_value);
        }
    }
    return r;
}
// What a lane of a row does with its V vectors, in the group kernel and in the row kernel: `stride`
// vectors lie between two of them, `at` is the first one's number in the row.  Only the last may
// reach the row's end.
template <typename T, int V, int CACHE> struct RowPiece {
    static constexpr int VEC = Vec128<T>::N;
    Vec128<T> q[V];
    float e[V][VEC];
    uint32_t first[V];  // where in the row each vector was loaded from
    uint32_t dup;       // leading elements of the last vector that another vector holds too (VEC: all of them)
    __device__ __forceinline__ void load(const T *rowp, uint32_t n, uint32_t at, uint32_t stride) {
#pragma unroll
        for (int i = 0; i < V; i++) {
            const uint32_t e0 = (static_cast<uint32_t>(i) * stride + at) * VEC;
            first[i] = i == V - 1 ? min(e0, n - VEC) : e0;
            q[i].v = load16<CACHE>(rowp + first[i]);
        }
        const uint32_t e_last = (static_cast<uint32_t>(V - 1) * stride + at) * VEC;
        dup = e_last > n - VEC ? min(e_last - (n - VEC), static_cast<uint32_t>(VEC)) : 0u;
    }
    // The largest of the G lanes' elements, NaN where one of them is NaN.
    template <int G> __device__ __forceinline__ float largest() const {
        if constexpr (sizeof(T) == 2) {
            uint32_t pk = maximum_half2(q[0].v.x, q[0].v.y, q[0].v.z);
#pragma unroll
            for (int i = 1; i < V; i++) pk = maximum_half2(maximum_half2(pk, q[i - 1].v.w, q[i].v.x), q[i].v.y, q[i].v.z);
            pk = maximum_half2(pk, q[V - 1].v.w, q[V - 1].v.w);
            pk = group_join<G>(pk, [](uint32_t a, uint32_t b) { return maximum_half2(a, b, b); });
            const float other = __half2float(__ushort_as_half(static_cast<uint16_t>(pk >> 16)));
            return maximum(__half2float(__ushort_as_half(static_cast<uint16_t>(pk & 0xFFFFu))), other, other);
        } else {
            float m = maximum(q[0].get(0), q[0].get(1), q[0].get(2));
#pragma unroll
            for (int i = 1; i < V; i++) m = maximum(maximum(m, q[i - 1].get(3), q[i].get(0)), q[i].get(1), q[i].get(2));
            m = maximum(m, q[V - 1].get(3), q[V - 1].get(3));
            return group_maximum<G>(m);
        }
    }
    // The terms, and their sum over this lane's elements: halves' terms added in float SUM at a time (TermSum).  (Numbers, whatever
    // the elements: a row with NaN, or whose maximum is not finite, shows in m -- row_reciprocal.)  n: the row's length.
    template <int SUM> __device__ __forceinline__ double terms(float m, uint32_t n) {
        static_assert(VEC % SUM == 0, "a vector's terms in equal parts");
        double acc = 0.0;
#pragma unroll
        for (int i = 0; i < V; i++) {
#pragma unroll
            for (int c = 0; c < VEC; c++) e[i][c] = term_of_row(q[i], c, m);
            if constexpr (sizeof(T) == 4) {
#pragma unroll
                for (int c = 0; c < VEC; c++) acc += static_cast<double>(i < V - 1 || static_cast<uint32_t>(c) >= dup ? e[i][c] : 0.f);
            } else {
                // The last vector repeats none of its elements (dup = 0), all of them, or, in one lane of a row, as many as
                // n says: the same number in every row, so that lane's sum has weights that are the same in every lane
                // (by a condition an element 16 instructions, which issue in 4.4 cycles, not 8 in 2.4).
                const uint32_t some = (0u - n) % VEC;
                auto weight = [&](int c) {  // (a scalar register's)
                    return __int_as_float(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(c) >= some ? 0x3F800000 : 0));
                };
#pragma unroll
                for (int c0 = 0; c0 < VEC; c0 += SUM) {
                    float part = e[i][c0];
#pragma unroll
                    for (int c = c0 + 1; c < c0 + SUM; c++) part += e[i][c];
                    if (i == V - 1) {
                        float rest = e[i][c0] * weight(c0);
#pragma unroll
                        for (int c = c0 + 1; c < c0 + SUM; c++) rest = fmaf(e[i][c], weight(c), rest);
                        part = dup == 0u ? part : dup < static_cast<uint32_t>(VEC) ? rest : 0.f;
                    }
                    acc += static_cast<double>(part);
                }
            }
        }
        return acc;
    }
    __device__ __forceinline__ void store(T *orow, double rinv, bool live, int nan_where, float nan_value) {
        const Quotient<T> over_sum(rinv);
#pragma unroll
        for (int i = 0; i < V; i++) {
            const Vec128<T> r = probabilities<T>(e[i], [&](int) { return over_sum; }, nan_where, nan_value);
            if (live && (i < V - 1 || dup < static_cast<uint32_t>(VEC))) store16<CACHE>(orow + first[i], r.v);
        }
    }
};
// The MAX_ONLY forms below write, instead of the tensor, each row's largest probability to out[row]: the term of the row's
// maximum over the same sum, so bit for bit the maximum of what the other form writes (NaN where that is NaN).
template <typename T> __device__ __forceinline__ void store_largest(T *out, size_t row, float m, double rinv) {
    store_elem(out, row, round_to_storage<T>(scale_term<T>(softmax_term_as<T>(m, m), rinv)));
}

constexpr int kSoftmaxGroupThreads = 256;
template <typename T, int G, int V, bool MAX_ONLY, int CACHE>
__global__ __launch_bounds__(kSoftmaxGroupThreads) void softmax_group_kernel(const T *in, T *out, uint32_t rows, uint32_t n,
                                                                            int nan_where, float nan_value) {
    const uint32_t row = blockIdx.x * (kSoftmaxGroupThreads / G) + threadIdx.x / G;
    const bool live = row < rows;
    const size_t row0 = static_cast<size_t>(live ? row : rows - 1u) * n;  // (lanes past the last row shadow it and store nothing)
    RowPiece<T, V, CACHE> p;
    p.load(in + row0, n, threadIdx.x % G, G);
    const float m = p.template largest<G>();
    // (halves: the shorter the row, the fewer terms are added in float -- n up to 64: 1, 128: 2, 256: 4, else 8)
    constexpr int SUM = G == 8 ? (V == 1 ? 1 : V == 2 ? 2 : 4) : G == 16 && V <= 2 ? 4 : 8;
    const double rinv = row_reciprocal(group_sum<G>(p.template terms<SUM < Vec128<T>::N ? SUM : Vec128<T>::N>(m, n)), m);
    if constexpr (MAX_ONLY) {
        if (live && threadIdx.x % G == 0) store_largest(out, row, m, rinv);
    } else {
        p.store(out + row0, rinv, live, nan_where, nan_value);
    }
}

// ---- a row per workgroup ----------------------------------------------------------------------
// Rows that a workgroup holds in registers, V vectors a thread; the workgroup has as many waves as
// the row needs (blockDim.x: at most 1024), so that a row just past a power of two does not leave
// half of it idle.  One read, one write, two barriers.  [9872,8296] f32 241 -> 114 us, f16 88 -> 61;
// [2000,20001] f32 225 -> 60 us, f16 133 -> 39 (element by element before); [256,8192] f32 8.4 -> 5.5.
constexpr int kSoftmaxRowWavesMax = 16;
template <typename T, int V, bool MAX_ONLY, int CACHE>
__global__ __launch_bounds__(kSoftmaxRowWavesMax *kWave) void softmax_row_kernel(const T *in, T *out, uint32_t n, int nan_where,
                                                                                float nan_value) {
    __shared__ float fscratch[kSoftmaxRowWavesMax];
    __shared__ double dscratch[kSoftmaxRowWavesMax];
    const uint32_t tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave, waves = blockDim.x / kWave;
    const size_t row0 = static_cast<size_t>(blockIdx.x) * n;
    RowPiece<T, V, CACHE> p;
    p.load(in + row0, n, tid, blockDim.x);
    float m = p.template largest<kWave>();
    if (waves > 1) {
        if (lane == 0) fscratch[wave] = m;
        __syncthreads();
        const uint32_t w = lane & (kSoftmaxRowWavesMax - 1);
        m = group_maximum<kSoftmaxRowWavesMax>(w < waves ? fscratch[w] : -INFINITY);
    }
    double s = group_sum<kWave>(p.template terms<Vec128<T>::N>(m, n));
    if (waves > 1) {
        if (lane == 0) dscratch[wave] = s;
        __syncthreads();
        const uint32_t w = lane & (kSoftmaxRowWavesMax - 1);
        s = group_sum<kSoftmaxRowWavesMax>(w < waves ? dscratch[w] : 0.0);
    }
    if constexpr (MAX_ONLY) {
        if (tid == 0) store_largest(out, blockIdx.x, m, row_reciprocal(s, m));
    } else {
        p.store(out + row0, row_reciprocal(s, m), true, nan_where, nan_value);
    }
}

// ---- rows shorter than a vector: a thread each ------------------------------------------------
// MAX_ONLY: rows of up to 16 elements, where a thread a row is still the faster one ([200000,13] f16 5.5 us, by the group
// kernel 9.8; f32 7.8 / 9.0).  The sum is taken as the kernel that writes the tensor takes it: rows longer than a vector a
// vector at a time, and those as the group kernel's lanes join (V = 1, terms in double).
constexpr uint32_t kSoftmaxThreadMaxN = 16;
template <typename T, bool MAX_ONLY>
__global__ __launch_bounds__(kSoftmaxGroupThreads) void softmax_thread_kernel(const T *in, T *out, uint32_t rows, uint32_t n,
                                                                             int nan_where, float nan_value) {
    constexpr uint32_t VEC = Vec128<T>::N, NMAX = MAX_ONLY ? kSoftmaxThreadMaxN : VEC - 1;
    static_assert(kSoftmaxThreadMaxN <= 4 * VEC, "vectors' sums");
    const uint32_t row = blockIdx.x * kSoftmaxGroupThreads + threadIdx.x;
    if (row >= rows) return;
    const T *rowp = in + static_cast<size_t>(row) * n;
    float x[NMAX], m = -INFINITY;
#pragma unroll
    for (uint32_t j = 0; j < NMAX; j++) {
        x[j] = load_elem(rowp, j < n ? j : 0u);
        if (j < n) m = fmaxf(m, x[j]);
    }
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (uint32_t j = 0; j < NMAX; j++) {
        x[j] = j < n ? softmax_term_as<T>(x[j], m) : 0.f;
        acc[j / VEC] += static_cast<double>(x[j]);
    }
    const double rinv = reciprocal_of_sum((acc[0] + acc[1]) + (acc[2] + acc[3]));
    if constexpr (MAX_ONLY) {
        store_largest(out, row, m, rinv);
    } else {
        T *orow = out + static_cast<size_t>(row) * n;
#pragma unroll
        for (uint32_t j = 0; j < NMAX; j++) {
            float p = round_to_storage<T>(scale_term<T>(x[j], rinv));
            if (nan_where && p != p) p = nan_value;
            if (j < n) store_elem(orow, j, p);
        }
    }
}

// ---- chunked rows: statistics ---------------------------------------------------------
// A chunk is NT * V * VEC elements of a row, what a workgroup of NT threads holds: vector i of thread tid is elements
// ((chunk * V + i) * NT + tid) * VEC and on, from any element (n >= VEC).  A row that is no whole
// number of vectors has its last one moved back to end with the row; the leading elements it repeats -- of the chunk
// before, possibly -- count for the chunk's maximum and minimum, which does no harm, and for nothing else.
template <typename T, int NT, int V> struct Chunk {
    static constexpr uint32_t VEC = Vec128<T>::N;
    Vec128<T> q[V];
    static __device__ __forceinline__ uint32_t first(uint32_t chunk) { return (chunk * (V * NT) + threadIdx.x) * VEC; }
    template <int CACHE> __device__ __forceinline__ void load(const T *rowp, uint32_t chunk, uint32_t n) {
        const uint32_t e_first = first(chunk);
#pragma unroll
        for (int i = 0; i < V; i++) {
            const uint32_t at = min(e_first + static_cast<uint32_t>(i) * (NT * VEC), n - VEC) * static_cast<uint32_t>(sizeof(T));  // (bytes: below 2^27)
            q[i].v = load16<CACHE>(reinterpret_cast<const T *>(reinterpret_cast<const char *>(rowp) + at));
        }
    }
};
template <int NT> struct ChunkScratch {
    static constexpr int NW = NT / kWave;
    static_assert(NW <= kSoftmaxRowWavesMax && kSoftmaxRowWavesMax % NW == 0, "waves a workgroup");
    float m[NW], mn[NW];
    double s[NW];
    uint32_t n[NW];
};
// The chunk's statistics, in every lane of the first wave.  All threads call; two barriers.
template <typename T, int NT, int V>
__device__ __forceinline__ ChunkStat chunk_stats(const Chunk<T, NT, V> &ch, uint32_t chunk, uint32_t n, ChunkScratch<NT> &sh) {
    constexpr uint32_t VEC = Vec128<T>::N;
    constexpr int NW = NT / kWave;
    const uint32_t tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    const uint32_t e_first = ch.first(chunk);
    // Maximum and minimum in one pass and one reduction.
    float m = -INFINITY, mn = INFINITY;  // (NaN is dropped)
    if constexpr (sizeof(T) == 2) {
        uint32_t pm = 0xFC00FC00u, pn = 0x7C007C00u;
#pragma unroll
        for (int i = 0; i < V; i++) {
            const uint4 &v = ch.q[i].v;
            pm = max_half2(max_half2(pm, max_half2(v.x, v.y)), max_half2(v.z, v.w));
            pn = min_half2(min_half2(pn, min_half2(v.x, v.y)), min_half2(v.z, v.w));
        }
        auto half = [](uint32_t h) { return __half2float(__ushort_as_half(static_cast<uint16_t>(h))); };
        m = fmaxf(half(pm & 0xFFFFu), half(pm >> 16));
        mn = fminf(half(pn & 0xFFFFu), half(pn >> 16));
    } else {
#pragma unroll
        for (int i = 0; i < V; i++) {
            m = max3(max3(m, ch.q[i].get(0), ch.q[i].get(1)), ch.q[i].get(2), ch.q[i].get(3));
            mn = min3(min3(mn, ch.q[i].get(0), ch.q[i].get(1)), ch.q[i].get(2), ch.q[i].get(3));
        }
    }
    const float own_min = mn;
    m = group_max<kWave>(m);
    mn = -group_max<kWave>(-mn);
    if (lane == 0) {
        sh.m[wave] = m;
        sh.mn[wave] = mn;
    }
    __syncthreads();
    m = group_max<kSoftmaxRowWavesMax>(sh.m[lane % NW]);
    mn = -group_max<kSoftmaxRowWavesMax>(-sh.mn[lane % NW]);
    // reference of the chunk's sum: its maximum, or 0 when that is not finite
    // (then every term is 0, inf or NaN, and NaN / inf must reach the sum)
    const float ref = (m > -INFINITY && m < INFINITY) ? m : 0.f;
    // The copies of the chunk's smallest value are set apart and counted: a value that fills most
    // of a row (padding, a floor, zeros) is usually its smallest, every copy of it has the same
    // term, and that term's error would go into the sum thousands of times over -- the row's sum
    // is DEFINED with exp_accurate(fl(x - M)) for each, which only the kernel that knows M can
    // count (4 ulp on rows of one value and a few peaks otherwise).  A wave without a copy has nothing to
    // set apart and saves two instructions an element.
    const bool apart = mn > -INFINITY && mn < INFINITY && __ballot(own_min == mn) != 0ull;  // (copies of -inf count for nothing either way)
    double acc = 0.0;
    uint32_t copies = 0;
    auto sum = [&](auto full_tag) {
#pragma unroll
        for (int i = 0; i < V; i++) {
            const uint32_t e0 = e_first + static_cast<uint32_t>(i) * (NT * VEC);
            const uint32_t dup = decltype(full_tag)::value || e0 <= n - VEC ? 0u : min(e0 - (n - VEC), VEC);
#pragma unroll
            for (int c = 0; c < static_cast<int>(VEC); c++) {
                const float x = ch.q[i].get(c);
                const double t = static_cast<double>(fast_term_unbiased(x, ref));
                const bool counts = decltype(full_tag)::value || static_cast<uint32_t>(c) >= dup;
                acc += counts ? t : 0.0;
                if (apart) copies += (counts && x == mn) ? 1u : 0u;  // (wave-uniform)
            }
        }
    };
    if ((chunk + 1u) * (NT * V * VEC) <= n) sum(std::true_type{});
    else sum(std::false_type{});
    // (every copy added the same float: taking them out again is exact to the sum's own rounding)
    if (apart) acc -= static_cast<double>(copies) * static_cast<double>(fast_term_unbiased(mn, ref));
    acc = group_sum<kWave>(acc);
    copies = wave_sum(copies);
    if (lane == 0) {
        sh.s[wave] = acc;
        sh.n[wave] = copies;
    }
    __syncthreads();
    if (tid < static_cast<uint32_t>(kWave)) {
        acc = sh.s[0];
        copies = sh.n[0];
#pragma unroll
        for (int w = 1; w < NW; w++) {  // fixed order: run-to-run stable
            acc += sh.s[w];
            copies += sh.n[w];
        }
    }
    return ChunkStat{acc, m, ref, mn, copies};
}

// Launch: rows * G workgroups.  The scale kernel reads the same bytes again and finds them in the Infinity Cache.
template <typename T, int NT, int V>
__global__ __launch_bounds__(NT) void softmax_stats_kernel(const T *__restrict__ in, ChunkStat *__restrict__ stats, uint32_t n,
                                                           uint32_t G) {
    __shared__ ChunkScratch<NT> sh;
    const uint32_t row = blockIdx.x / G, chunk = blockIdx.x - row * G;
    Chunk<T, NT, V> ch;
    ch.template load<kCacheLoads>(in + static_cast<size_t>(row) * n, chunk, n);
    const ChunkStat st = chunk_stats(ch, chunk, n, sh);
    if (threadIdx.x == 0) stats[blockIdx.x] = st;
}

// A row's maximum and the reciprocal of its sum (in thread 0) from its G chunks.  Up to 64 of them are combined by the first
// wave, a chunk a lane; with more each wave takes its share (two barriers more, a quarter of the exponentials).
template <typename T, uint32_t NT>
__device__ __forceinline__ LineStats combine_chunks(const ChunkStat *cs, uint32_t G, float *wave_m, double *wave_s) {
    static_assert(NT / kWave == 4, "the two combinations below");
    const uint32_t tid = threadIdx.x;
    const uint32_t takers = G <= static_cast<uint32_t>(kWave) ? static_cast<uint32_t>(kWave) : NT;
    float M = -INFINITY;
    double part = 0.0;
    if (tid < takers) {
        for (uint32_t g = tid; g < G; g += takers) M = fmaxf(M, cs[g].m);
        M = group_max<kWave>(M);
    }
    if (takers == NT) {
        if ((tid & (kWave - 1)) == 0) wave_m[tid / kWave] = M;
        __syncthreads();
        M = fmaxf(fmaxf(wave_m[0], wave_m[1]), fmaxf(wave_m[2], wave_m[3]));
    }
    if (tid < takers) {
        for (uint32_t g = tid; g < G; g += takers) {
            const ChunkStat st = cs[g];
            if (st.s != 0.0) part += st.s * sum_rescale(st.s, st.ref, M);
            if (st.nmin != 0u) part += static_cast<double>(st.nmin) * static_cast<double>(softmax_term_as<T>(st.vmin, M));
        }
        part = group_sum<kWave>(part);
    }
    if (takers == NT) {
        if ((tid & (kWave - 1)) == 0) wave_s[tid / kWave] = part;
        __syncthreads();
        part = (wave_s[0] + wave_s[1]) + (wave_s[2] + wave_s[3]);
    }
    return LineStats{M, 0.f, 1.0 / part};
}

// ---- chunked rows: exp(x - M) / S -----------------------------------------------------
// Launch: rows * GS workgroups of 256, V vectors a thread, GS = ceil(n / (256 * V * VEC)); G: the
// chunks a row of the statistics kernel.  In-place calls are fine: see the moved vector.
// [64,128256] f32, both kernels: 24.9 -> 22.3 us (2 reads and 1 write of 33 MB: 4.4 TB/s);
// [63,132402] (rows off 16 bytes) f32 35.9 -> 24.3, f16 34.8 -> 17.3; [32,50257] f16 10.1 -> 8.0.
constexpr int kSoftmaxScaleThreads = 256;
template <typename T, int V>
__global__ __launch_bounds__(kSoftmaxScaleThreads) void softmax_scale_kernel(const T *in, T *out, const ChunkStat *__restrict__ stats,
                                                                            uint32_t n, uint32_t G, uint32_t GS, int nan_where,
                                                                            float nan_value) {
    constexpr uint32_t VEC = Vec128<T>::N, NT = kSoftmaxScaleThreads;
    __shared__ LineStats row_stats;
    __shared__ float wave_m[NT / kWave];
    __shared__ double wave_s[NT / kWave];
    const uint32_t tid = threadIdx.x;
    const uint32_t row = blockIdx.x / GS, chunk = blockIdx.x - row * GS;
    const uint32_t e_first = chunk * (NT * V * VEC) + tid * VEC;
    const size_t row0 = static_cast<size_t>(row) * n;
    const T *rowp = in + row0;
    Vec128<T> q[V];
#pragma unroll
    for (int i = 0; i < V; i++) q[i].v = load16_stream(rowp + min(e_first + static_cast<uint32_t>(i) * NT * VEC, n - VEC));
    // (under everyone's loads)
    const LineStats combined = combine_chunks<T, NT>(stats + static_cast<size_t>(row) * G, G, wave_m, wave_s);
    if (tid == 0) row_stats = combined;
    __syncthreads();
    const Quotient<T> over_sum(row_stats.rinv);
    const float m = row_stats.m;
    T *orow = out + row0;
#pragma unroll
    for (int i = 0; i < V; i++) {
        const uint32_t e0 = e_first + static_cast<uint32_t>(i) * NT * VEC;
        float e[VEC];
#pragma unroll
        for (int c = 0; c < static_cast<int>(VEC); c++) e[c] = term_of_row(q[i], c, m);
        const Vec128<T> r = probabilities<T>(e, [&](int) { return over_sum; }, nan_where, nan_value);
        if (e0 <= n - VEC) {
            store16_stream(orow + e0, r.v);
        } else if (e0 < n) {
            // (the moved vector: its own elements alone -- those it repeats may be another workgroup's,
            // which in an in-place call has replaced them by now)
            const uint32_t dup = e0 - (n - VEC);
#pragma unroll
            for (int c = 1; c < static_cast<int>(VEC); c++)
                if (static_cast<uint32_t>(c) >= dup) store_elem(orow, n - VEC + static_cast<uint32_t>(c), r.get(c));
        }
    }
}

// The largest probability of each row, out[row], in place of the above.  Launch: a workgroup a row.
template <typename T>
__global__ __launch_bounds__(kSoftmaxScaleThreads) void softmax_fold_max_kernel(T *__restrict__ out, const ChunkStat *__restrict__ stats, uint32_t G) {
    constexpr uint32_t NT = kSoftmaxScaleThreads;
    __shared__ float wave_m[NT / kWave];
    __shared__ double wave_s[NT / kWave];
    const LineStats st = combine_chunks<T, NT>(stats + static_cast<size_t>(blockIdx.x) * G, G, wave_m, wave_s);
    if (threadIdx.x == 0) store_elem(out, blockIdx.x, round_to_storage<T>(softmax_prob_as<T>(st.m, st)));
}

// ---- long strided lines: a tile of neighbouring lines per workgroup -----------------------------
// Lines along a non-last axis that the register kernel below does not hold (n above
// kStridedMaxN).  A workgroup takes TI neighbouring lines (TI = the power of two at or
// above min(inner, 64)); lane l of a wave looks at line l % TI of the tile and, with 64 / TI
// rows per instruction, at row l / TI of the instruction's rows, so every load and store
// covers contiguous pieces of TI elements; the workgroup's waves take the rows in turn.
// Three passes over the tile (maximum, sum of terms, output; the second and third come
// from the cache for tiles of a few hundred kilobytes), each reduced across a wave's row
// groups by shuffles and across the waves through LDS.  One thread per line -- what this
// replaces -- had 2048 threads on a [32,1000,64] tensor: 741 us for 16 MB.
constexpr int kStridedTileThreads = 1024;
// What a launch of the tile kernel does: the whole softmax of its tiles, or -- when the tensor
// has too few tiles to fill the chip -- one of the two halves of a split over G row chunks a
// tile: every chunk's maximum and sum (hardware-exp terms against the chunk's own maximum, as
// in the chunked row kernels) into stats[(tile * G + chunk) * TI + line], then the
// probabilities from the line's G results.  G * TI <= 1024.
// The ...Max modes write, instead of the tensor, each line's largest probability to out[line]
// (softmax followed by a max over the same axis): from the same statistics, so bit-equal to
// the maximum of what the other modes write.
enum { kTileWhole = 0, kTileStats = 1, kTileScale = 2, kTileWholeMax = 3, kTileFoldMax = 4 };
template <typename T, int MODE>
__global__ __launch_bounds__(kStridedTileThreads) void softmax_strided_tile_kernel(const T *__restrict__ in, T *__restrict__ out,
                                                                                    ChunkStat *__restrict__ stats, LineGeom g,
                                                                                    uint32_t ti_shift, uint32_t G, uint32_t per,
                                                                                    int nan_where, float nan_value) {
    constexpr int NT = kStridedTileThreads, NW = NT / kWave;
    constexpr int U = 16;  // rows a lane has in flight (a pass is a chain of n / (16 waves * U) round trips)
    __shared__ float fmax_lds[NW * kWave];
    __shared__ double dsum_lds[NW * kWave];
    __shared__ uint32_t ucnt_lds[MODE == kTileStats ? NW * kWave : 1];
    const uint32_t tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    const uint32_t TI = 1u << ti_shift, RPW = kWave >> ti_shift;  // lines a tile, rows per wave instruction
    const uint32_t tiles = (g.inner + TI - 1) >> ti_shift;
    const uint32_t tileid = blockIdx.x / G, chunk = blockIdx.x - tileid * G;
    const uint32_t o = tileid / tiles, tile = tileid - o * tiles;
    const uint32_t c0 = min(chunk * per, g.n), c1 = min(c0 + per, g.n);  // this workgroup's rows
    const uint32_t mine = lane & (TI - 1);                               // this lane's line of the tile
    const uint32_t col = (tile << ti_shift) + mine, r = lane >> ti_shift;
    const bool col_ok = col < g.inner;
    const size_t base = static_cast<size_t>(o) * g.n * g.inner + (col_ok ? col : 0u);
    const uint32_t step = NW * RPW;  // rows the workgroup covers per turn
    // element of row j of this lane's line
    auto at = [&](uint32_t j) { return base + static_cast<size_t>(j) * g.inner; };
    // combine v over the lanes of a wave that look at the same line, then over the waves; all threads call
    auto reduce_max = [&](float v) -> float {
        for (uint32_t off = TI; off < static_cast<uint32_t>(kWave); off <<= 1) v = fmaxf(v, __shfl_xor(v, static_cast<int>(off), kWave));
        fmax_lds[tid] = v;
        __syncthreads();
        float m = fmax_lds[mine];
#pragma unroll
        for (int w = 1; w < NW; w++) m = fmaxf(m, fmax_lds[w * kWave + mine]);
        return m;
    };
    auto reduce_sum = [&](double v) -> double {
        for (uint32_t off = TI; off < static_cast<uint32_t>(kWave); off <<= 1) v += __shfl_xor(v, static_cast<int>(off), kWave);
        dsum_lds[tid] = v;
        __syncthreads();
        double sum = dsum_lds[mine];
#pragma unroll
        for (int w = 1; w < NW; w++) sum += dsum_lds[w * kWave + mine];  // fixed order: run-to-run stable
        return sum;
    };
    // one pass over the workgroup's rows: use(x, j) for every element of this lane's line
    auto pass = [&](auto use) {
        for (uint32_t j0 = c0 + wave * RPW + r; j0 < c1; j0 += step * U) {
            float x[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const uint32_t j = j0 + static_cast<uint32_t>(u) * step;
                x[u] = load_elem(in, at(j < c1 ? j : c0));
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const uint32_t j = j0 + static_cast<uint32_t>(u) * step;
                if (j < c1) use(x[u], j);
            }
        }
    };
    constexpr bool kFold = MODE == kTileScale || MODE == kTileFoldMax;
    constexpr bool kMaxOnly = MODE == kTileWholeMax || MODE == kTileFoldMax;
    if (MODE == kTileFoldMax && chunk != 0) return;  // (the whole workgroup: one writer a tile)
    LineStats st{0.f, 0.f, 0.0};
    if constexpr (!kFold) {
        // ---- 1. the lines' maxima
        float m = -INFINITY;
        pass([&](float x, uint32_t) { m = fmaxf(m, x); });  // (drops NaN)
        m = reduce_max(m);
        // ---- 2. the sums of the terms
        double acc = 0.0;
        if constexpr (MODE != kTileStats) {
            pass([&](float x, uint32_t) { acc += static_cast<double>(softmax_term_as<T>(x, m)); });
            st = LineStats{m, 0.f, 1.0 / reduce_sum(acc)};
        } else {
            // reference of the chunk's sum: its maximum, or 0 when that is not finite (then
            // every term is 0, inf or NaN, and NaN / inf must reach the sum)
            const float ref = (m > -INFINITY && m < INFINITY) ? m : 0.f;
            // The copies of ONE value are counted apart (as in softmax_stats_kernel: the kernel that knows
            // the line's maximum adds the accurate term for each): the line's first element in this chunk,
            // where the second equals it -- a value that fills a line turns up at once, every lane of the
            // line reads the same two elements (from the cache) and decides alike, and a line of spread-out
            // values pays a comparison per element and nothing else.
            const float x0 = load_elem(in, at(c0 < c1 ? c0 : 0u)), x1 = load_elem(in, at(c0 + 1u < c1 ? c0 + 1u : 0u));
            const bool apart = c0 + 1u < c1 && x0 == x1 && x0 > -INFINITY && x0 < INFINITY;
            uint32_t copies = 0;
            pass([&](float x, uint32_t) {
                if (apart && x == x0) copies += 1u;
                else acc += static_cast<double>(fast_term_unbiased(x, ref));
            });
            // (both sums in one round: over the lanes of a wave that look at the same line, then over the waves)
            for (uint32_t off = TI; off < static_cast<uint32_t>(kWave); off <<= 1) {
                acc += __shfl_xor(acc, static_cast<int>(off), kWave);
                copies += __shfl_xor(copies, static_cast<int>(off), kWave);
            }
            dsum_lds[tid] = acc;
            ucnt_lds[tid] = copies;
            __syncthreads();
            if (tid < TI) {
                double sum = dsum_lds[tid];
                uint32_t nx0 = ucnt_lds[tid];
#pragma unroll
                for (int w = 1; w < NW; w++) {  // fixed order: run-to-run stable
                    sum += dsum_lds[w * kWave + tid];
                    nx0 += ucnt_lds[w * kWave + tid];
                }
                stats[(static_cast<size_t>(tileid) * G + chunk) * TI + tid] = ChunkStat{sum, m, ref, x0, nx0};
            }
            return;
        }
    } else {
        // thread c * TI + l fetches chunk c's result for line l; every lane then folds its line's G
        const bool holds = tid < G * TI;
        ChunkStat cs{0.0, -INFINITY, 0.f, 0.f, 0u};
        if (holds) cs = stats[(static_cast<size_t>(tileid) * G + (tid >> ti_shift)) * TI + mine];
        fmax_lds[tid] = cs.m;
        __syncthreads();
        float M = fmax_lds[mine];
        for (uint32_t c = 1; c < G; c++) M = fmaxf(M, fmax_lds[c * TI + mine]);
        dsum_lds[tid] = ((holds && cs.s != 0.0) ? cs.s * sum_rescale(cs.s, cs.ref, M) : 0.0) +
                        ((holds && cs.nmin != 0u) ? static_cast<double>(cs.nmin) * static_cast<double>(softmax_term_as<T>(cs.vmin, M)) : 0.0);
        __syncthreads();
        double sum = dsum_lds[mine];
        for (uint32_t c = 1; c < G; c++) sum += dsum_lds[c * TI + mine];
        st = LineStats{M, 0.f, 1.0 / sum};
    }
    if constexpr (kMaxOnly) {
        // the line's maximum has the term exp_accurate(0) = 1 (NaN statistics give NaN, as the tensor would)
        if (tid < TI && col_ok) store_elem(out, static_cast<size_t>(o) * g.inner + col, softmax_prob_as<T>(st.m, st));
        return;
    }
    // ---- 3. the probabilities
    pass([&](float x, uint32_t j) {
        float p = round_to_storage<T>(softmax_prob_as<T>(x, st));
        if (nan_where && p != p) p = nan_value;
        if (col_ok) store_elem(out, at(j), p);
    });
}

// ---- short strided lines held in registers -------------------------------------------------
// Lines along a non-last axis with n <= kStridedMaxN elements (scores laid out
// [batch, classes, anchors]: softmax over the classes).  Lanes run along the
// contiguous inner axis, so every load is a coalesced piece of a row of the slab.
// P lanes of a wave share a line (lane l and l + 64/P, ...: element j belongs to
// part j mod P), each keeps its part in registers: one read of the input, no LDS,
// and enough waves to hide the loads and the exponentials even when the lines
// are few (one thread per line left two waves per SIMD on [16,80,8400]; staging
// the lines in LDS, the first version, no more).  NMAX: compile-time bound of n,
// a multiple of 16 and of P (the loops are unrolled over NMAX / P and masked).
constexpr int kStridedThreads = 128;
constexpr int kStridedMaxN = 128;

// MAX_ONLY: instead of the softmax tensor write, per line, its largest entry --
// the probability of the line's maximum, (float)(exp_accurate(0) / S) -- to
// out[line]: softmax followed by a max over the same axis, in one read.
template <typename T, int NMAX, int P, bool MAX_ONLY>
__global__ __launch_bounds__(kStridedThreads) void softmax_strided_reg_kernel(const T *in, T *out, LineGeom g,
                                                                              int nan_where, float nan_value) {
    constexpr int LPW = kWave / P;  // lines per wave
    constexpr int NPER = NMAX / P;  // elements per lane
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t part = lane / LPW;
    // (neighbouring groups of lines share cache lines where rows of the slab start off a line boundary)
    const uint32_t wave_id = (xcd_grouped_block() * kStridedThreads + threadIdx.x) / kWave;
    const uint32_t lines = g.outer * g.inner;
    const uint32_t line_raw = wave_id * LPW + (lane % LPW);
    const bool live = line_raw < lines;
    const uint32_t line = live ? line_raw : 0u;  // (idle lanes shadow line 0 and store nothing)
    const size_t base = g.base(line);
    const uint32_t n = g.n;
    float x[NPER];
    // every load in flight before the first use (slots past the line re-read element 0)
#pragma unroll
    for (int i = 0; i < NPER; i++) {
        const uint32_t j = static_cast<uint32_t>(i) * P + part;
        x[i] = load_elem(in, base + static_cast<size_t>(j < n ? j : 0u) * g.inner);
    }
    float m = -INFINITY;
#pragma unroll
    for (int i = 0; i < NPER; i++)
        if (static_cast<uint32_t>(i) * P + part < n) m = fmaxf(m, x[i]);
#pragma unroll
    for (int o = LPW; o < kWave; o <<= 1) m = fmaxf(m, __shfl_xor(m, o, kWave));
    // terms replace the elements; the parts' sums are added in a fixed order
    TermSum<T> s_own = 0;
#pragma unroll
    for (int i = 0; i < NPER; i++) {
        if (static_cast<uint32_t>(i) * P + part < n) {
            x[i] = softmax_term_as<T>(x[i], m);
            s_own += static_cast<TermSum<T>>(x[i]);
        }
    }
    double s = static_cast<double>(s_own);
#pragma unroll
    for (int o = LPW; o < kWave; o <<= 1) s += __shfl_xor(s, o, kWave);
    const double rinv = 1.0 / s;
    if constexpr (MAX_ONLY) {
        // the largest term is exp_accurate(0) = 1 unless the line holds no finite maximum
        float top = 0.f;
#pragma unroll
        for (int i = 0; i < NPER; i++) {
            if (static_cast<uint32_t>(i) * P + part < n) {
                const float e = x[i];
                top = (e != e) ? e : ((top != top) ? top : fmaxf(top, e));  // NaN propagates
            }
        }
#pragma unroll
        for (int o = LPW; o < kWave; o <<= 1) {
            const float other = __shfl_xor(top, o, kWave);
            top = (other != other) ? other : ((top != top) ? top : fmaxf(top, other));
        }
        float p = round_to_storage<T>(scale_term<T>(top, rinv));
        if (nan_where && p != p) p = nan_value;
        if (live && part == 0) store_elem(out, line, p);
        return;
    }
    const Quotient<T> over_sum(rinv);
#pragma unroll
    for (int i = 0; i < NPER; i++) {
        const uint32_t j = static_cast<uint32_t>(i) * P + part;
        if (live && j < n) {
            float p = round_to_storage<T>(over_sum(x[i]));
            if (nan_where && p != p) p = nan_value;
            store_elem(out, base + static_cast<size_t>(j) * g.inner, p);
        }
    }
}

}  // namespace vkop
