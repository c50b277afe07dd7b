// Device-side building blocks shared by the softmax / top-k kernels (gfx950,
// wave64).  Header only; every function is __device__ __forceinline__.
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace vkop {

constexpr int kWave = 64;

// ---------------------------------------------------------------- loads ----

// Element of a float or half (uint16_t bits) tensor, widened to float.
template <typename T> __device__ __forceinline__ float load_elem(const T *p, size_t i);
template <> __device__ __forceinline__ float load_elem<float>(const float *p, size_t i) { return p[i]; }
template <> __device__ __forceinline__ float load_elem<uint16_t>(const uint16_t *p, size_t i) {
    return __half2float(__ushort_as_half(p[i]));
}

// Element of a float or half tensor whose order is turned round: it reads as its negative, and what is
// stored is turned back, so a kernel written for the k largest gives the k smallest, ties by lower index
// as before.  NaN still ranks as the largest value, which is last now: a loaded vector gives -inf for it
// (Vec128, kernels_rows.hpp), which never becomes a candidate; where -inf itself is placed -- fewer than
// k+1 other elements -- and in the exact selects, NaN comes behind it (plain_key).
template <typename B> struct Reversed {
    B bits;
};
template <typename T> constexpr bool kReversed = false;
template <typename B> constexpr bool kReversed<Reversed<B>> = true;
template <> __device__ __forceinline__ float load_elem<Reversed<float>>(const Reversed<float> *p, size_t i) { return -p[i].bits; }
template <> __device__ __forceinline__ float load_elem<Reversed<uint16_t>>(const Reversed<uint16_t> *p, size_t i) {
    return -__half2float(__ushort_as_half(p[i].bits));
}

// Round-to-nearest-even store of a float into a float or half tensor.
template <typename T> __device__ __forceinline__ void store_elem(T *p, size_t i, float v);
template <> __device__ __forceinline__ void store_elem<float>(float *p, size_t i, float v) { p[i] = v; }
template <> __device__ __forceinline__ void store_elem<uint16_t>(uint16_t *p, size_t i, float v) {
    p[i] = __half_as_ushort(__float2half_rn(v));
}

template <> __device__ __forceinline__ void store_elem<Reversed<float>>(Reversed<float> *p, size_t i, float v) { p[i].bits = -v; }
template <> __device__ __forceinline__ void store_elem<Reversed<uint16_t>>(Reversed<uint16_t> *p, size_t i, float v) {
    p[i].bits = __half_as_ushort(__float2half_rn(-v));
}

// Value as the tensor type would hold it (float stays, half is rounded to
// binary16 and widened again).
template <typename T> __device__ __forceinline__ float round_to_storage(float v);
template <> __device__ __forceinline__ float round_to_storage<float>(float v) { return v; }
template <> __device__ __forceinline__ float round_to_storage<uint16_t>(float v) {
    return __half2float(__float2half_rn(v));
}

// 16 bytes of a tensor that start on any element: a 128-bit load or store needs no more than the
// element's own alignment on this chip (rows of odd length start anywhere).  Measured on a stream
// of 128 MB: starts on 4 or 8 bytes cost nothing (6.3 TB/s read), starts on 2 bytes a fifth (5.1).
// The _stream ones are non-temporal: what a softmax tensor holds is not
// used again by the call, and keeping it out of the caches' way takes a copy of 1 GB from 5.7 to 6.2 TB/s
// (four vectors a thread).  Where ordinary ones are better: softmax_caching.
typedef uint32_t vec16_any __attribute__((ext_vector_type(4), aligned(2)));
template <typename T> __device__ __forceinline__ uint4 load16_stream(const T *p) {
    const auto v = __builtin_nontemporal_load(reinterpret_cast<const vec16_any *>(p));
    return make_uint4(v.x, v.y, v.z, v.w);
}
template <typename T> __device__ __forceinline__ uint4 load16_any(const T *p) {
    const auto v = *reinterpret_cast<const vec16_any *>(p);
    return make_uint4(v.x, v.y, v.z, v.w);
}
template <typename T> __device__ __forceinline__ void store16_stream(T *p, const uint4 &u) {
    vec16_any v;
    v.x = u.x, v.y = u.y, v.z = u.z, v.w = u.w;
    __builtin_nontemporal_store(v, reinterpret_cast<vec16_any *>(p));
}

template <typename T> __device__ __forceinline__ void store16_any(T *p, const uint4 &u) {
    vec16_any v;
    v.x = u.x, v.y = u.y, v.z = u.z, v.w = u.w;
    *reinterpret_cast<vec16_any *>(p) = v;
}

// Which accesses of a softmax kernel to its tensors are ordinary ones (a template parameter: of two branches on a flag the
// compiler makes one).
enum Caching : int { kCacheNone = 0, kCacheLoads = 1, kCacheStores = 2, kCacheBoth = kCacheLoads | kCacheStores };
template <int CACHE, typename T> __device__ __forceinline__ uint4 load16(const T *p) {
    if constexpr ((CACHE & kCacheLoads) != 0) return load16_any(p);
    else return load16_stream(p);
}
template <int CACHE, typename T> __device__ __forceinline__ void store16(T *p, const uint4 &u) {
    if constexpr ((CACHE & kCacheStores) != 0) store16_any(p, u);
    else store16_stream(p, u);
}

// Larger of three floats, quiet NaN dropped (fmaxf on loaded values costs one more instruction an operand:
// the compiler first turns every value that may be a signalling NaN into a quiet one).  A signalling NaN
// may come out as a quiet one: for callers whose result is NaN wherever an operand was -- a softmax's
// maximum, the smallest value of a chunk whose sum is NaN either way.
__device__ __forceinline__ float max3(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
__device__ __forceinline__ float min3(float a, float b, float c) {
    float r;
    asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
// Larger and smaller halves of two pairs, quiet NaN dropped (signalling: as above).
__device__ __forceinline__ uint32_t max_half2(uint32_t a, uint32_t b) {
    uint32_t r;
    asm("v_pk_max_f16 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// The larger halves of three pairs, the larger and the smaller of three floats, NaN wherever one of them is NaN.
__device__ __forceinline__ uint32_t maximum_half2(uint32_t a, uint32_t b, uint32_t c) {
    uint32_t r;
    asm("v_pk_maximum3_f16 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
__device__ __forceinline__ float maximum(float a, float b, float c) {
    float r;
    asm("v_maximum3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

__device__ __forceinline__ float minimum(float a, float b, float c) {
    float r;
    asm("v_minimum3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

__device__ __forceinline__ uint32_t min_half2(uint32_t a, uint32_t b) {
    uint32_t r;
    asm("v_pk_min_f16 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// A half of a word, widened, minus m: one instruction and one rounding, as the conversion and the difference have.
__device__ __forceinline__ float half_minus(uint32_t w, bool high, float m) {
    float d;
    if (high) asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(d) : "v"(w), "v"(m));
    else asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel_hi:[1,0,0]" : "=v"(d) : "v"(w), "v"(m));
    return d;
}
// (a s, b t), each rounded to float and then to a half.
__device__ __forceinline__ uint32_t half2_of_products(float a, float s, float b, float t) {
    uint32_t w;
    asm("v_fma_mixlo_f16 %0, %1, %2, 0\n\tv_fma_mixhi_f16 %0, %3, %4, 0" : "=&v"(w) : "v"(a), "v"(s), "v"(b), "v"(t));
    return w;
}

// x * scale rounded to float on its own: never contracted into a fused multiply-add
// with what follows, so that a kernel given a scale computes on exactly the values
// a tensor scaled beforehand would hold.
// (the empty asm hides the product from the optimizer; `__fmul_rn` alone is a plain
// multiplication to this compiler and does get contracted)
__device__ __forceinline__ float scaled(float x, float scale) {
#pragma clang fp contract(off)
    float p = x * scale;
    asm volatile("" : "+v"(p));
    return p;
}

// ------------------------------------------------------------ ordering ----

// Maps a float to a uint32 whose unsigned order is the ranking top-k uses:
// NaN (either sign) above +inf, -0 == +0, otherwise the numeric order.
__device__ __forceinline__ uint32_t order_key(float v) {
    if (v != v) return 0xFFFFFFFFu;
    uint32_t u = __float_as_uint(v + 0.0f);  // -0 + +0 = +0
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// The key plain top-k ranks an element by: order_key, and for a reversed element NaN below everything
// (above 0, "no element").
template <typename T> __device__ __forceinline__ uint32_t plain_key(float v) {
    if constexpr (kReversed<T>) return v != v ? 1u : order_key(v);
    else return order_key(v);
}

// Composite of key and position: larger composite = ranks earlier; among equal
// keys the lower index is the larger composite.  Never 0 for idx < 2^32-1.
__device__ __forceinline__ uint64_t composite(uint32_t key, uint32_t idx) {
    return (static_cast<uint64_t>(key) << 32) | static_cast<uint64_t>(0xFFFFFFFFu - idx);
}
__device__ __forceinline__ uint32_t composite_index(uint64_t c) {
    return 0xFFFFFFFFu - static_cast<uint32_t>(c);
}

// Number of lanes below the caller among those set in `mask`.
__device__ __forceinline__ uint32_t lanes_below(uint64_t mask) {
    return __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(mask >> 32),
                                     __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(mask), 0u));
}

// hist[d] += 1 for every lane that calls (lanes may call under divergence).  The lanes that
// share the first such lane's digit add once between them: keys repeat (tied data, a dominant
// value, the leading bits of a sorted row), and same-address LDS atomics of one instruction
// are carried out one after the other.
__device__ __forceinline__ void hist_add_grouped(uint32_t *hist, uint32_t d) {
    const uint32_t lead = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(d)));
    const uint64_t same = __ballot(d == lead);
    if (d == lead) {
        if (lanes_below(same) == 0) atomicAdd(&hist[lead], static_cast<uint32_t>(__popcll(same)));
    } else {
        atomicAdd(&hist[d], 1u);
    }
}

// ------------------------------------------------------- block order ----
// Workgroups are handed to the chip's 8 XCDs in turn (workgroup b runs on XCD b mod 8),
// and each XCD has an L2 of its own: two workgroups with neighbouring blockIdx never
// share one.  For kernels whose neighbouring pieces of work touch the same cache lines
// (rows of a slab that do not start on a line boundary), this gives the position in
// the work's own order that workgroup blockIdx.x should take so that neighbouring
// pieces run on one XCD: XCD x takes the x-th eighth of the pieces.  A bijection on
// [0, gridDim.x).
constexpr uint32_t kXcds = 8;
__device__ __forceinline__ uint32_t xcd_grouped_block() {
    const uint32_t nb = gridDim.x, b = blockIdx.x;
    const uint32_t xcd = b % kXcds, local = b / kXcds;
    const uint32_t each = nb / kXcds, rem = nb % kXcds;  // the first `rem` XCDs get one piece more
    return xcd * each + min(xcd, rem) + local;
}

// ---------------------------------------------------------- reductions ----

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, kWave));
    return v;
}
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
    return v;
}
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
    return v;
}
__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
    return v;
}

// Block-wide max / sum through a small LDS array (one slot per wave).  Every
// thread of the block must call; the result is returned to all of them.
// `scratch` needs NT / 64 slots and is reusable after the call returns.
template <int NT> __device__ __forceinline__ float block_max(float v, float *scratch) {
    constexpr int NW = NT / kWave;
    v = wave_max(v);
    if constexpr (NW == 1) return v;
    __syncthreads();  // scratch may still be read from a previous call
    if ((threadIdx.x & (kWave - 1)) == 0) scratch[threadIdx.x / kWave] = v;
    __syncthreads();
    float r = scratch[0];
#pragma unroll
    for (int w = 1; w < NW; w++) r = fmaxf(r, scratch[w]);
    return r;
}
template <int NT> __device__ __forceinline__ double block_sum(double v, double *scratch) {
    constexpr int NW = NT / kWave;
    v = wave_sum(v);
    if constexpr (NW == 1) return v;
    __syncthreads();
    if ((threadIdx.x & (kWave - 1)) == 0) scratch[threadIdx.x / kWave] = v;
    __syncthreads();
    double r = scratch[0];
#pragma unroll
    for (int w = 1; w < NW; w++) r += scratch[w];  // fixed order: run-to-run stable
    return r;
}

// --------------------------------------------------------------- softmax ----

// The larger of d and -104, below which a term is 0.  NAN_TOO: NaN stays NaN (else it is -104; half the cycles).
template <bool NAN_TOO> __device__ __forceinline__ float at_least_minus_104(float d) {
    float r;
    if constexpr (NAN_TOO) asm("v_maximum3_f32 %0, %1, %2, %2" : "=v"(r) : "v"(d), "s"(-104.0f));
    else asm("v_max_f32 %0, %2, %1" : "=v"(r) : "v"(d), "s"(-104.0f));
    return r;
}

// exp(d) rounded to float, evaluated in double, for d up to 88 (a term's exponent is at most a
// little above 0) or NaN: the relative error before the final rounding is below 2^-39, so the
// result is the correctly rounded float except within that distance of a rounding midpoint,
// where it is the other neighbour.  d below -104 (including -inf) gives 0; NaN gives NaN.
// It is the one thing a float softmax tensor computes per element.  Single-precision sums and products issue in 2.4
// cycles a wave here, double ones, conversions and everything else in 4.4: the multiple of ln 2 is found in single precision
// by adding and subtracting 1.5 2^23 (any integer near d log2 e serves: |r| <= 0.34662
// covers the rounding of d * log2 e), the low bits of that sum go into the double's exponent as they are --
// before the one rounding to float, which a subnormal result needs -- and the polynomial is
// the one of degree 8 that interpolates e^r at the nine Chebyshev points of that interval, its
// coefficients rounded to double (2^-39.7; the Taylor polynomial of degree 9 it replaces: 2^-37).
template <bool NAN_TOO = true> __device__ __forceinline__ float exp_accurate(float d) {
    d = at_least_minus_104<NAN_TOO>(d);
    constexpr float kMagic = 12582912.f;
    const float nb = fmaf(d, 1.44269504088896341f, kMagic);
    const float n = nb - kMagic;
    const double r = fma(-static_cast<double>(n), 0.69314718055994530942, static_cast<double>(d));
    double p = 0x1.a15a6596eb202p-16;
    p = fma(p, r, 0x1.a1aa9a9593b29p-13);
    p = fma(p, r, 0x1.6c164de469f83p-10);
    p = fma(p, r, 0x1.1110809a3308dp-7);
    p = fma(p, r, 0x1.555555742f31dp-5);
    p = fma(p, r, 0x1.555555a27dcddp-3);
    p = fma(p, r, 0x1.fffffffff71a8p-2);
    p = fma(p, r, 0x1.ffffffffd37fep-1);
    p = fma(p, r, 1.0);
    const uint32_t hi = static_cast<uint32_t>(__double2hiint(p)) + (__float_as_uint(nb) << 20);  // (0.7 <= p <= 1.5, -150 <= n: still a normal double)
    const float e = static_cast<float>(__hiloint2double(static_cast<int>(hi), __double2loint(p)));
    // (a NaN's low bits have gone into that exponent: e may be any number, and is NaN again with d * 0; else e + 0)
    return NAN_TOO ? fmaf(d, 0.f, e) : e;
}

// One softmax term: exp of the single-precision difference x - m.
__device__ __forceinline__ float softmax_term(float x, float m) { return exp_accurate(x - m); }

// exp(d) in single precision throughout, good to about two units in the last place of a float: the
// hardware exponential of a = fl(d log2 e), and what d is more than a ln 2 as a first-order factor
// (exp(d) = 2^a e^r, r = d - a ln 2, |r| < 2^-18: the first product-and-sum is exact but for its last rounding).  For results that are
// stored in half precision: 2^-22.8 relative (every 29th float from 0 to -87; 2^-25.3 in the mean square) before a rounding to 11 bits moves one result in two
// thousand by one unit of a half, and costs a third of exp_accurate.  Results below 2^-126 are 0.
template <bool NAN_TOO = true> __device__ __forceinline__ float exp_half_grade(float d) {
    constexpr float kLog2E = 1.44269502162933349609375f;
    constexpr float kLn2Hi = 0.693147182464599609375f, kLn2Lo = -1.904654323148236017e-9f;  // ln 2 in two floats
    d = at_least_minus_104<NAN_TOO>(d);  // (there the hardware exponential is 0, and what follows is finite)
    const float a = d * kLog2E;
    const float r = fmaf(-a, kLn2Lo, fmaf(-a, kLn2Hi, d));
    const float e = __builtin_amdgcn_exp2f(a);
    return fmaf(e, r, e);
}

// The term as the element type asks for it: float tensors get the correctly rounded exponential,
// half tensors (uint16_t) the single-precision one.  Every kernel that writes a softmax TENSOR
// takes its terms from here, so the results of one element type agree between them.
template <typename T> __device__ __forceinline__ float softmax_term_as(float x, float m) {
    if constexpr (sizeof(T) == 2) return exp_half_grade(x - m);
    else return exp_accurate(x - m);
}

// What a thread adds its own few terms up in, and how a term becomes a probability, in the same
// kernels: double for float tensors (the sum and the quotient as the definition rounds them), float
// for half tensors (a few dozen terms a thread: 2^-19 relative at worst, against 2^-11 of a half;
// the threads' sums are then added in double like everyone's).  Conversions to and from double are
// a quarter-rate instruction each, four of them an element: half tensors ran at the speed of float
// tensors of the same shape, for half the bytes.
template <typename T> using TermSum = std::conditional_t<sizeof(T) == 2, float, double>;
template <typename T> __device__ __forceinline__ float scale_term(float e, double rinv) {
    if constexpr (sizeof(T) == 2) return e * static_cast<float>(rinv);
    else return static_cast<float>(static_cast<double>(e) * rinv);
}

// scale_term for many terms of one row, bit for bit: what is the same for all of them is worked out once.
template <typename T> struct Quotient;
template <> struct Quotient<float> {
    double rinv;
    Quotient() = default;
    __device__ __forceinline__ explicit Quotient(double r) : rinv(r) {}
    __device__ __forceinline__ float operator()(float e) const { return scale_term<float>(e, rinv); }
};
template <> struct Quotient<uint16_t> {
    float high;
    Quotient() = default;
    __device__ __forceinline__ explicit Quotient(double rinv) : high(static_cast<float>(rinv)) {}
    __device__ __forceinline__ float operator()(float e) const { return e * high; }
};

// The nucleus cut of a sorted result, by all 64 lanes of one wave: the number of leading values whose
// running sum -- added in order, in float, sum = fl(sum + v) -- first reaches p, or k if it never does
// (a NaN reaches nothing).  value(r) gives rank r < k.  The running sums move through the lanes: every lane
// keeps adding its own value to what its left neighbour holds (one instruction across the wave; lane 0
// holds fl(carry + v0) and adds 0 to itself), and after t steps lanes 0..t hold their final sums -- the
// additions of the walk one value at a time, in the same order, each a wave-wide instruction instead of
// a read of one lane, an addition, a comparison and a branch.
template <typename F> __device__ __forceinline__ uint32_t nucleus_count_wave(uint32_t k, float p, F &&value) {
    const uint32_t lane = threadIdx.x & (kWave - 1);
    float carry = 0.f;
    for (uint32_t base = 0; base < k; base += kWave) {
        const uint32_t m = min(static_cast<uint32_t>(kWave), k - base);
        const float v = base + lane < k ? value(base + lane) : 0.f;
        float s = lane == 0 ? __fadd_rn(carry, v) : v;
        const float own = lane == 0 ? 0.f : v;
        for (uint32_t t = 1; t < m; t += 4) {  // (steps past m - 1 change nothing below lane m)
#pragma unroll
            for (int u = 0; u < 4; u++) {
                // wave_shr:1 -- lane l reads lane l - 1, lane 0 (no source) keeps its own
                const float left = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(s), __float_as_int(s), 0x138, 0xF, 0xF, false));
                s = __fadd_rn(own, left);
            }
        }
        const unsigned long long reached = __ballot(lane < m && s >= p);
        if (reached != 0ull) return base + static_cast<uint32_t>(__builtin_ctzll(reached)) + 1u;
        carry = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s), static_cast<int>(m - 1u)));
    }
    return k;
}

}  // namespace vkop
