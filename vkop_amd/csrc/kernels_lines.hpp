// Softmax along a non-last axis, lines of up to kLinesMaxN elements: one read, one write.
//
// A tensor is [outer][n][inner]; a line is the n elements that lie inner apart.  A lane holds L
// neighbouring lines (a 16-byte vector of the inner axis, at any alignment), of every line the
// elements part, part + parts, ..., K of them at most.  The parts of a line are P groups of lanes of
// a wave times W waves of a workgroup: maxima and sums cross the lanes by register exchanges and,
// with W > 1, the waves through LDS (three barriers).
// What bounds it: with wide rows the memory system ([8,21,262144] f32 81.5 -> 66.3 us, 5.3 TB/s; the
// largest probability alone, one read, 65.6 -> 42.2), with long lines the workgroups that hold them --
// 1024 elements are 8 waves of 100 registers, two a CU, and loads, exponentials and stores of two
// overlap little ([8,1000,8000] f32 192 -> 113 us, 4.5 TB/s, where three passes of 4-byte accesses
// ran before).  The rule that picks P, W and K, with what it was measured on: plan_lines.
#pragma once

#include "kernels_softmax.hpp"

namespace vkop {

constexpr int kLinesWavesMax = 16;

// The value of the lane whose number differs in bit STRIDE.
template <int STRIDE> __device__ __forceinline__ uint32_t lane_xor(uint32_t v) {
    if constexpr (STRIDE == 32) {
        const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
        return (threadIdx.x & 32u) ? r[0] : r[1];
    } else if constexpr (STRIDE == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
        return (threadIdx.x & 16u) ? r[0] : r[1];
    } else if constexpr (STRIDE == 8) {
        return dpp_u32<0x128>(v);  // (a rotation of sixteen by eight)
    } else {
        return static_cast<uint32_t>(__shfl_xor(static_cast<int>(v), STRIDE, kWave));
    }
}
// Maxima and sums over the P lanes of a wave that look at the same lines (lanes 64 / P apart), L values a lane.  The lanes share
// the lines out: a step exchanges one half of the values for the other lane's other half (one swap and one operation for two
// values), so that after the steps of 32 and 16 lanes a lane holds kOwned = L / min(P, 4) of the lines, from owned_line() on;
// the steps of 8 and 4 leave both lanes of a pair with them.  (With every value to every lane each step costs four times as much:
// exchanges, not terms, were 40 % of the instructions of a line's largest probability: [16,80,8400] f32 13.5 -> 12.2 us; the tensor's time is the memory's and did not change.)  The sum adds
// both lanes of a pair in the same order, so every lane ends with the same bits.
template <int STRIDE> __device__ __forceinline__ void swap_lanes(uint32_t &a, uint32_t &b) {
    if constexpr (STRIDE == 32) {
        const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
        a = r[0], b = r[1];
    } else {
        const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
        a = r[0], b = r[1];
    }
}
template <int STRIDE> __device__ __forceinline__ void swap_lanes(double &a, double &b) {
    uint64_t x = static_cast<uint64_t>(__double_as_longlong(a)), y = static_cast<uint64_t>(__double_as_longlong(b));
    uint32_t xl = static_cast<uint32_t>(x), xh = static_cast<uint32_t>(x >> 32), yl = static_cast<uint32_t>(y), yh = static_cast<uint32_t>(y >> 32);
    swap_lanes<STRIDE>(xl, yl);
    swap_lanes<STRIDE>(xh, yh);
    a = __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(xh) << 32) | xl));
    b = __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(yh) << 32) | yl));
}
template <int STRIDE> __device__ __forceinline__ double lane_xor(double v) {
    const uint64_t u = static_cast<uint64_t>(__double_as_longlong(v));
    const uint64_t o = (static_cast<uint64_t>(lane_xor<STRIDE>(static_cast<uint32_t>(u >> 32))) << 32) | lane_xor<STRIDE>(static_cast<uint32_t>(u));
    return __longlong_as_double(static_cast<long long>(o));
}
template <int STRIDE> __device__ __forceinline__ float lane_xor(float v) { return __uint_as_float(lane_xor<STRIDE>(__float_as_uint(v))); }
template <int P> constexpr int kLineSharers = P < 4 ? P : 4;
// The steps of 8 and 4 lanes.
template <int P, typename V, typename F> __device__ __forceinline__ V join_rest(V v, F op) {
    if constexpr (P >= 8) v = op(v, lane_xor<8>(v));
    if constexpr (P >= 16) v = op(v, lane_xor<4>(v));
    return v;
}
// Afterwards v[0 .. L / kLineSharers<P>) are the lane's own.
template <int P, int L, typename V, typename F> __device__ __forceinline__ void share_out(V (&v)[L], F op) {
    if constexpr (P >= 2) {
#pragma unroll
        for (int i = 0; i < L / 2; i++) {
            swap_lanes<32>(v[i], v[i + L / 2]);
            v[i] = op(v[i], v[i + L / 2]);
        }
    }
    if constexpr (P >= 4) {
#pragma unroll
        for (int i = 0; i < L / 4; i++) {
            swap_lanes<16>(v[i], v[i + L / 4]);
            v[i] = op(v[i], v[i + L / 4]);
        }
    }
#pragma unroll
    for (int i = 0; i < L / kLineSharers<P>; i++) v[i] = join_rest<P>(v[i], op);
}
// The way back: every lane's own values to all lanes of the same lines.
template <int P, int L> __device__ __forceinline__ void hand_out(float (&f)[L]) {
    uint32_t v[L];
#pragma unroll
    for (int i = 0; i < L / kLineSharers<P>; i++) v[i] = __float_as_uint(f[i]);
    if constexpr (P >= 4) {
#pragma unroll
        for (int i = 0; i < L / 4; i++) {
            v[i + L / 4] = v[i];
            swap_lanes<16>(v[i], v[i + L / 4]);
        }
    }
    if constexpr (P >= 2) {
#pragma unroll
        for (int i = 0; i < L / 2; i++) {
            v[i + L / 2] = v[i];
            swap_lanes<32>(v[i], v[i + L / 2]);
        }
    }
#pragma unroll
    for (int i = 0; i < L; i++) f[i] = __uint_as_float(v[i]);
}
template <int P, int L> __device__ __forceinline__ uint32_t owned_line(uint32_t lane) {
    return (P >= 2 ? (lane >> 5) * (L / 2) : 0u) + (P >= 4 ? ((lane >> 4) & 1u) * (L / 4) : 0u);
}

// MAX_ONLY: instead of the softmax tensor write each line's largest probability to out[line]: from
// the same sums, so bit-equal to the maximum of what the other form writes.
// K = ceil(n / (P * W)): every element but a lane's last exists.
// Launch: blockDim = teams * W waves, a team of W waves per 64 / P vectors; LDS for W > 1:
// 64 / P * L * (W * teams) doubles.
// CACHE: softmax_caching (stored past the caches, the parts of a cache line go to memory one by one: [8,100,83886] f32 235 us,
// with ordinary stores 120; [8,128,65537] f16 169 / 85).
// WIDE: a lane adds its terms in double.  Halves in one wave a line add up to eight of them in float (TermSum), which
// [8,21,262144] is worth 2 %; longer lines, more of them in all, do not.
// (the largest probability of halves is held to 64 registers, which K = 8 exceeds by one: two workgroups of 16 waves a CU
// instead of one, [8,1000,8000] 47 against 61 us)
template <typename T, int K, int P, bool MAX_ONLY, bool WIDE, int CACHE>
__global__ __launch_bounds__(kLinesWavesMax *kWave) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 2 && MAX_ONLY ? 8 : 4))) void softmax_lines_reg_kernel(const T *in, T *out, LineGeom g, uint32_t W,
                                                                                int nan_where, float nan_value) {
    constexpr int L = Vec128<T>::N;
    constexpr uint32_t LPW = kWave / P;  // vectors (of L lines) a wave
    extern __shared__ double lines_lds[];
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t wave = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / kWave)));
    const uint32_t teams = blockDim.x / kWave / W, team = wave / W, tw = wave - team * W;
    const uint32_t vpo = (g.inner + L - 1u) / L, total = g.outer * vpo;  // vectors an outer index, and in all
    const uint32_t slot = lane & (LPW - 1u), part = tw * P + lane / LPW, parts = W * P;
    // (neighbouring vectors share cache lines where rows of the slab start off a line boundary)
    const uint32_t vec = (xcd_grouped_block() * teams + team) * LPW + slot;
    const bool live = vec < total;
    const uint32_t o = (live ? vec : 0u) / vpo, iv = (live ? vec : 0u) - o * vpo;  // (idle lanes shadow the first vector and store nothing)
    const uint32_t col = min(iv * L, g.inner - L);  // the last vector of a row is moved back to end with it ...
    const uint32_t skip = iv * L - col;             // ... and this many of its lines are the one's before
    const size_t base = static_cast<size_t>(o) * g.n * g.inner + col;
    const uint32_t n = g.n;
    const bool last_ok = (K - 1) * parts + part < n;
    Vec128<T> q[K];
#pragma unroll
    for (int i = 0; i < K; i++) {
        const uint32_t j = static_cast<uint32_t>(i) * parts + part;
        q[i].v = load16<CACHE>(in + base + static_cast<size_t>(i < K - 1 || last_ok ? j : n - 1u) * g.inner);
    }
    constexpr int C = L / kLineSharers<P>, EXTRA = P / kLineSharers<P>;  // lines a lane owns, lanes that own the same
    const uint32_t own0 = owned_line<P, L>(lane), extra = (lane / LPW) % EXTRA;
    float m[L];
    if constexpr (sizeof(T) == 2) {
        uint32_t pk[4] = {q[0].v.x, q[0].v.y, q[0].v.z, q[0].v.w};
#pragma unroll
        for (int i = 1; i < K; i += 2) {
            const Vec128<T> &a = q[i], &b = q[i + 1 < K ? i + 1 : i];
            pk[0] = maximum_half2(pk[0], a.v.x, b.v.x), pk[1] = maximum_half2(pk[1], a.v.y, b.v.y);
            pk[2] = maximum_half2(pk[2], a.v.z, b.v.z), pk[3] = maximum_half2(pk[3], a.v.w, b.v.w);
        }
        share_out<P>(pk, [](uint32_t a, uint32_t b) { return maximum_half2(a, b, b); });
#pragma unroll
        for (int w = 0; w < C / 2; w++) {
            m[2 * w] = __half2float(__ushort_as_half(static_cast<uint16_t>(pk[w] & 0xFFFFu)));
            m[2 * w + 1] = __half2float(__ushort_as_half(static_cast<uint16_t>(pk[w] >> 16)));
        }
    } else {
        uint32_t mu[L];
#pragma unroll
        for (int c = 0; c < L; c++) {
            m[c] = K == 1 ? maximum(q[0].get(c), q[0].get(c), q[0].get(c)) : q[0].get(c);
#pragma unroll
            for (int i = 1; i < K; i += 2) m[c] = maximum(m[c], q[i].get(c), q[i + 1 < K ? i + 1 : i].get(c));
            mu[c] = __float_as_uint(m[c]);
        }
        share_out<P>(mu, [](uint32_t a, uint32_t b) { return __float_as_uint(maximum(__uint_as_float(a), __uint_as_float(b), __uint_as_float(b))); });
#pragma unroll
        for (int c = 0; c < C; c++) m[c] = __uint_as_float(mu[c]);
    }
    auto larger = [](float a, float b) { return maximum(a, b, b); };  // (NaN where a line holds one)
    if (W > 1) {
        // a wave's maxima go to LDS, and the lanes that own the same lines read their share of the waves
        float *fl = reinterpret_cast<float *>(lines_lds) + team * (W * LPW * L);
        if (extra == 0) {
#pragma unroll
            for (int c = 0; c < C; c++) fl[(tw * L + own0 + c) * LPW + slot] = m[c];
        }
        __syncthreads();
        for (uint32_t w = extra; w < W; w += EXTRA) {
#pragma unroll
            for (int c = 0; c < C; c++) m[c] = larger(m[c], fl[(w * L + own0 + c) * LPW + slot]);
        }
#pragma unroll
        for (int c = 0; c < C; c++) m[c] = join_rest<P>(m[c], larger);
        __syncthreads();  // (the sums take the same place)
    }
    float own_m[C];
#pragma unroll
    for (int c = 0; c < C; c++) own_m[c] = m[c];
    hand_out<P>(m);
    float e[K][L];
    std::conditional_t<WIDE, double, TermSum<T>> acc[L];
#pragma unroll
    for (int c = 0; c < L; c++) acc[c] = 0;
#pragma unroll
    for (int i = 0; i < K; i++) {
        // (a vector after the other: scheduled together, the terms of sixteen do not fit the registers)
        asm volatile("" : "+v"(q[i].v.x), "+v"(q[i].v.y), "+v"(q[i].v.z), "+v"(q[i].v.w));
#pragma unroll
        for (int c = 0; c < L; c++) {
            e[i][c] = term_of_row(q[i], c, m[c]);
            acc[c] += i < K - 1 || last_ok ? e[i][c] : 0.f;
        }
    }
    double s[L];  // (the lane's own C lines)
#pragma unroll
    for (int c = 0; c < L; c++) s[c] = static_cast<double>(acc[c]);
    auto sum = [](double a, double b) { return a + b; };
    share_out<P>(s, sum);
    if (W > 1) {
        double *dl = lines_lds + team * (W * LPW * L);
        if (extra == 0) {
#pragma unroll
            for (int c = 0; c < C; c++) dl[(tw * L + own0 + c) * LPW + slot] = s[c];
        }
        __syncthreads();
#pragma unroll
        for (int c = 0; c < C; c++) s[c] = 0.0;
        for (uint32_t w = extra; w < W; w += EXTRA) {  // fixed order: run-to-run stable
#pragma unroll
            for (int c = 0; c < C; c++) s[c] += dl[(w * L + own0 + c) * LPW + slot];
        }
#pragma unroll
        for (int c = 0; c < C; c++) s[c] = join_rest<P>(s[c], sum);
    }
    if constexpr (MAX_ONLY) {
        if (live && extra == 0 && tw == 0) {
            // the line's maximum has the term exp(0) = 1 (NaN where there is none, as the tensor would hold)
            const size_t at = static_cast<size_t>(o) * g.inner + col;
            Vec128<T> r;
            r.v = make_uint4(0, 0, 0, 0);
            float p[C];
#pragma unroll
            for (int c = 0; c < C; c++) {
                p[c] = scale_term<T>(softmax_term_as<T>(own_m[c], own_m[c]), row_reciprocal(s[c], own_m[c]));
                if constexpr (C == L) r.set(c, p[c]);
            }
            if (C == L && skip == 0) store16_stream(out + at, r.v);
            else {
#pragma unroll
                for (int c = 0; c < C; c++)
                    if (own0 + static_cast<uint32_t>(c) >= skip) store_elem(out, at + own0 + c, p[c]);
            }
        }
        return;
    }
    Quotient<T> over_sum[L];
    if constexpr (sizeof(T) == 2) {
        float high[L];
#pragma unroll
        for (int c = 0; c < C; c++) high[c] = Quotient<T>(row_reciprocal(s[c], own_m[c])).high;
        hand_out<P>(high);
#pragma unroll
        for (int c = 0; c < L; c++) over_sum[c].high = high[c];
    } else {
        // (a double's two words as two floats)
        float low[L], high[L];
#pragma unroll
        for (int c = 0; c < C; c++) {
            const double r = row_reciprocal(s[c], own_m[c]);
            low[c] = __int_as_float(__double2loint(r)), high[c] = __int_as_float(__double2hiint(r));
        }
        hand_out<P>(low);
        hand_out<P>(high);
#pragma unroll
        for (int c = 0; c < L; c++) over_sum[c].rinv = __hiloint2double(__float_as_int(high[c]), __float_as_int(low[c]));
    }
    size_t at = base + static_cast<size_t>(part) * g.inner;
    asm volatile("" : "+v"(at));  // (places again: sixteen of them kept from the loads are 32 registers)
#pragma unroll
    for (int i = 0; i < K; i++, at += static_cast<size_t>(parts) * g.inner) {
#pragma unroll
        for (int c = 0; c < L; c++) asm volatile("" : "+v"(e[i][c]));
        const Vec128<T> r = probabilities<T>(e[i], [&](int c) { return over_sum[c]; }, nan_where, nan_value);
        if (live && (i < K - 1 || last_ok)) {
            if (skip == 0) store16<CACHE>(out + at, r.v);
            else {
                // (its own lines alone: the others are another wave's, which may have stored them, in place, already)
#pragma unroll
                for (int c = 1; c < L; c++)
                    if (static_cast<uint32_t>(c) >= skip) store_elem(out, at + c, r.get(c));
            }
        }
    }
}

}  // namespace vkop
