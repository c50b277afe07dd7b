// Softmax of long last-axis rows in one launch, one read and one write.
//
// A row is split into G chunks (plan_joined: at most 20; the reader of the records holds 64), a workgroup each, as in the pair of
// kernels in kernels_softmax.hpp (statistics, scale), which reads the tensor twice.  Here a workgroup keeps its chunk in registers,
// publishes the chunk's statistics, waits until those of the row's other chunks are there and writes its probabilities.
// The wait needs no particular number of workgroups on the chip: workgroups start in order, so those of the rows before end
// without this one's help, and after `polls` looks a workgroup that still misses a chunk (its workgroup has not started:
// other streams' kernels hold the chip) reads that chunk itself.  Every wait ends, whatever else runs.
// in == out is fine: a chunk is read by its own workgroup before that writes, and one that is read for another workgroup while its
// own writes over it has its record in memory by then, which is looked for again after the read.  (Its last vector must not
// reach back into the chunk before, which may have been written: the pair takes such rows in place.)
// What bounds it: the arithmetic and the loads of the few workgroups a CU holds, half each -- [64,128256] f32 with neither
// exponential takes 11.5 us, without the wait as long as with it -- and, with few rows, the wait.  us, the pair / this:
// [64,128256] f32 21.9 / 16.3, f16 14.9 / 13.2; [500,50257] f32 55.3 / 43.5, f16 37.8 / 28.3; [32,33001] f32 8.7 / 8.0, f16 7.8 / 7.3.
// The pair stays for few rows of many chunks, where the wait is all there is.
#pragma once

#include "kernels_softmax.hpp"

namespace vkop {

constexpr uint32_t kJoinedMaxChunks = kWave;
constexpr int kJoinedWords = 4;  // 64-bit words of a chunk's record

// A record is four words of 40 bits each under a tag of 24 that differs from launch to launch and from word to word: a word
// with its tag has arrived, whatever lay there before, and no word needs to arrive before another.  22 bits are the launch's,
// which are not all 0 (a cleared word has not arrived) and come again after 2^22 - 1 launches; two are the word's.
constexpr uint32_t launch_tag(uint32_t launch) { return ((launch % 0x3FFFFFu + 1u) * 0x9E3779u) & 0x3FFFFFu; }  // (an odd factor)
__host__ __device__ constexpr uint32_t word_tag(uint32_t tag, int i) { return (tag << 2) | static_cast<uint32_t>(i); }
__device__ __forceinline__ void publish_chunk(uint64_t *rec, const ChunkStat &c, uint32_t tag) {
    const uint64_t low40 = (1ull << 40) - 1u, s = static_cast<uint64_t>(__double_as_longlong(c.s));
    auto put = [&](int i, uint64_t bits) { publish(rec + i, (static_cast<uint64_t>(word_tag(tag, i)) << 40) | bits); };
    put(0, s & low40);
    put(1, (s >> 40) | (static_cast<uint64_t>(c.nmin) << 24));
    put(2, __float_as_uint(c.m));
    put(3, __float_as_uint(c.vmin));
}
struct ChunkWords {
    uint64_t w[kJoinedWords];
    __device__ __forceinline__ void read(const uint64_t *rec) {
#pragma unroll
        for (int i = 0; i < kJoinedWords; i++) w[i] = fetch(rec + i);
    }
    __device__ __forceinline__ bool arrived(uint32_t tag) const {
        bool ok = true;
#pragma unroll
        for (int i = 0; i < kJoinedWords; i++) ok = ok && static_cast<uint32_t>(w[i] >> 40) == word_tag(tag, i);
        return ok;
    }
    __device__ __forceinline__ ChunkStat stat() const {
        const uint64_t low40 = (1ull << 40) - 1u;
        const float m = __uint_as_float(static_cast<uint32_t>(w[2]));
        const double s = __longlong_as_double(static_cast<long long>((w[0] & low40) | (w[1] << 40)));
        return ChunkStat{s, m, (m > -INFINITY && m < INFINITY) ? m : 0.f, __uint_as_float(static_cast<uint32_t>(w[3])),
                         static_cast<uint32_t>(w[1] >> 24) & 0xFFFFu};
    }
};
// The row's maximum and the reciprocal of its sum from a chunk a lane, in every lane of the wave: combine_chunks's, bit for bit.
template <typename T> __device__ __forceinline__ LineStats combine_wave(const ChunkStat &c, bool holds) {
    const float M = group_max<kWave>(holds ? c.m : -INFINITY);
    double part = 0.0;
    if (holds) {
        if (c.s != 0.0) part += c.s * sum_rescale(c.s, c.ref, M);
        if (c.nmin != 0u) part += static_cast<double>(c.nmin) * static_cast<double>(softmax_term_as<T>(c.vmin, M));
    }
    return LineStats{M, 0.f, 1.0 / group_sum<kWave>(part)};
}

// Launch: rows * G workgroups, G = ceil(n / (NT * V * VEC)); recs: [rows][G] records, done: [rows], at zero before and after.
template <typename T, int NT, int V>
__global__ __launch_bounds__(NT) void softmax_joined_kernel(const T *in, T *out, uint64_t *recs, uint32_t *done, uint32_t n, uint32_t G,
                                                            uint32_t tag, uint32_t polls, int nan_where, float nan_value) {
    constexpr uint32_t VEC = Vec128<T>::N;
    static_assert(NT * V * VEC < (1 << 16), "a record's count");
    __shared__ ChunkScratch<NT> sh;
    __shared__ ChunkStat stats[kJoinedMaxChunks];  // where this workgroup has to read chunks itself
    __shared__ LineStats row_stats;
    __shared__ uint64_t sh_missing;
    const uint32_t tid = threadIdx.x;
    const uint32_t row = blockIdx.x / G, own = blockIdx.x - row * G;
    const size_t row0 = static_cast<size_t>(row) * n;
    const T *rowp = in + row0;
    uint64_t *rrecs = recs + static_cast<size_t>(row) * G * kJoinedWords;
    Chunk<T, NT, V> ch;
    ch.template load<kCacheNone>(rowp, own, n);
    const ChunkStat mine = chunk_stats(ch, own, n, sh);
    if (tid < static_cast<uint32_t>(kWave)) {
        if (tid == 0) publish_chunk(rrecs + own * kJoinedWords, mine, tag);
        ChunkWords w;
        uint64_t missing;
        for (uint32_t poll = 0;; poll++) {
            bool absent = false;
            if (tid < G) {
                w.read(rrecs + tid * kJoinedWords);
                absent = !w.arrived(tag);
            }
            missing = __ballot(absent);
            // (its own may be missing too: a call that breaks the rules for a workspace can take it away)
            if (missing == 0ull || poll >= polls) break;
            __builtin_amdgcn_s_sleep(1);
        }
        const ChunkStat c = w.stat();
        if (missing == 0ull) {
            const LineStats st = combine_wave<T>(c, tid < G);
            if (tid == 0) row_stats = st;
        } else if (tid < G) {
            stats[tid] = c;  // (those of the missing chunks are written below)
        }
        if (tid == 0) sh_missing = missing;
        // Its own record is in memory before the counter is raised -- whoever clears the records clears that too -- and before
        // any of its probabilities is written.
        asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
    }
    __syncthreads();
    if (sh_missing != 0ull) {
        for (uint64_t left = sh_missing; left != 0ull; left &= left - 1ull) {
            const uint32_t c = static_cast<uint32_t>(__builtin_ctzll(left));
            ch.template load<kCacheNone>(rowp, c, n);
            ChunkStat st = chunk_stats(ch, c, n, sh);
            if (tid < static_cast<uint32_t>(kWave)) {
                // (in place the chunk's workgroup may have started and written over it by now: then its record came first)
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
                ChunkWords w;
                w.read(rrecs + c * kJoinedWords);
                if (w.arrived(tag)) st = w.stat();
                if (tid == 0) stats[c] = st;
            }
        }
        __syncthreads();
        if (tid < static_cast<uint32_t>(kWave)) {
            const LineStats st = combine_wave<T>(stats[tid < G ? tid : 0u], tid < G);
            if (tid == 0) row_stats = st;
        }
        uint32_t again = own;
        asm volatile("" : "+s"(again));  // (places again: the first load's, kept till here, are 16 registers)
        ch.template load<kCacheNone>(rowp, again, n);
        __syncthreads();
    }
    // This workgroup has read what it needs of the row's records.  (Whose answer is not waited for here: at an address the
    // compiler takes for the same in every lane it would be, before the lanes that ask share it out.)
    uint32_t before = 0, same = 0;
    asm volatile("" : "+v"(same));
    if (tid == 0) before = __hip_atomic_fetch_add(done + row + same, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const Quotient<T> over_sum(row_stats.rinv);
    const float m = row_stats.m;
    T *orow = out + row0;
    const uint32_t e_first = ch.first(own);
#pragma unroll
    for (int i = 0; i < V; i++) {
        const uint32_t e0 = e_first + static_cast<uint32_t>(i) * (NT * VEC);
        float e[VEC];
#pragma unroll
        for (int c = 0; c < static_cast<int>(VEC); c++) e[c] = term_of_row(ch.q[i], c, m);
        const Vec128<T> r = probabilities<T>(e, [&](int) { return over_sum; }, nan_where, nan_value);
        if (e0 <= n - VEC) {
            store16_stream(orow + e0, r.v);
        } else if (e0 < n) {
            const uint32_t dup = e0 - (n - VEC);
#pragma unroll
            for (int c = 1; c < static_cast<int>(VEC); c++)
                if (static_cast<uint32_t>(c) >= dup) store_elem(orow, n - VEC + static_cast<uint32_t>(c), r.get(c));
        }
    }
    // the last workgroup to have read what it needs of the row's records clears them
    if (tid < static_cast<uint32_t>(kWave)) {
        before = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(before)));
        if (before == G - 1u) {
            if (tid < G) {
#pragma unroll
                for (int i = 0; i < kJoinedWords; i++) publish(rrecs + tid * kJoinedWords + i, 0ull);
            }
            if (tid == 0) __hip_atomic_store(done + row, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

}  // namespace vkop
