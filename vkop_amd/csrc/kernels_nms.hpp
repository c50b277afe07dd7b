// Non-maximum suppression: the operator behind the detection chain's top-k.
//
// boxes [B][N][4], scores [B][C][N].  One workgroup per (batch, class), as in the
// reference (ops/Nms.hpp:115, shaders/nms.comp:74-82), but every phase is done by
// the whole workgroup instead of its first thread:
//   1. the boxes whose score is greater than the threshold are collected, in any
//      order (in box order where they are more than kNmsMaxCandidates, of which the first stay);
//   2. they are sorted by (score, then lower box index) as 64-bit composites in LDS
//      (counting sort for few, their boxes loaded under it; bitonic network for many,
//      and every thread loads the corner coordinates of its own sorted positions into registers);
//   3. the sorted list is walked in blocks of 64: all waves compute, for every
//      candidate of the block, which other ones of the block overlap it
//      (IoU as in shaders/nms.comp:61-72, every operation rounded on its own so
//      that the comparison with the threshold is the same bit for bit on the
//      host); the first wave finds the kept set with a few ballots (a fixed-point
//      iteration instead of one step per kept box).  Up to 512 candidates, the
//      usual case, have their boxes in LDS: the waves share a block's tests
//      against the boxes kept so far as they share those within it, and the kept
//      boxes gather at the front.  Of more, every thread tests its own later
//      candidates, held in registers, against the block's survivors and clears
//      their bits in the active mask.  Two barriers per block of 64 instead of
//      one per selection;
//   4. the (batch, class, box) records of all pairs are written one after the other, in order of
//      batch and class: the result does not depend on scheduling (the reference appends through a
//      global atomic counter).  Of pairs that the chip holds at once every workgroup publishes its
//      number of records, waits for those of the pairs before it and writes its own (place_records);
//      of more, and in a recording, the selected box indices go to the pair's segment of the
//      workspace and nms_pack_kernel writes them all.
#pragma once

#include "device_utils.hpp"
#include "kernels_rows.hpp"
#include "select.hpp"

namespace vkop {

constexpr int kNmsThreadsWide = 1024;   // few (batch, class) pairs
constexpr int kNmsThreadsNarrow = 256;  // twice as many as the chip holds wide workgroups at a time, two a CU
// (us a call at f32, wide / narrow: [4,80,8400] 11.9 / 11.8, [8,80,8400] 15.2 / 13.0, [8,91,1917] 11.5 / 10.7,
// [12,80,8400] 18.7 / 15.3, [16,80,8400] 22.9 / 18.2; with 400 candidates a pair [16,20,8400] 24.3 / 29.7,
// [32,20,8400] 33.3 / 34.7.  From 513 pairs on narrow ones gain where candidates are
// few, but where all of 2048 are they lose more: [8,80,2048] 285 / 424)
constexpr int kNmsNarrowMinPairs = 1024;
// One launch where the chip holds all workgroups at once (six narrow ones a CU, two wide: waves_per_eu of nms_kernel).  Of more, those
// that wait for the pairs before them keep the rest from starting: us, two launches / one, [8,91,1917] f32 11.7 / 13.4, [20,90,3000]
// 14.1 / 16.5; held at once [16,80,8400] 18.7 / 17.4, [1,80,8400] 9.8 / 8.3, [2,80,1000] 9.8 / 7.3.
constexpr uint32_t kNmsHeldNarrow = 1536, kNmsHeldWide = 512;
constexpr int kNmsMaxCandidates = 2048;  // per (batch, class); the reference's shader holds 1024
constexpr int kNmsRankSortMax = 512;     // up to here a counting sort beats the bitonic network's barriers

__device__ __forceinline__ uint32_t uniform_u32(uint32_t x) {
    return static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(x)));
}

// Four consecutive scores from p on: 16 (half: 8) bytes that start on any element.
__device__ __forceinline__ float4 nms_load4(const float *p) {
    const uint4 w = load16_any(p);
    return make_float4(__uint_as_float(w.x), __uint_as_float(w.y), __uint_as_float(w.z), __uint_as_float(w.w));
}
__device__ __forceinline__ float4 nms_load4(const uint16_t *p) {
    typedef uint32_t vec8_any __attribute__((ext_vector_type(2), aligned(2)));
    const auto w = *reinterpret_cast<const vec8_any *>(p);
    return make_float4(__half2float(__ushort_as_half(static_cast<unsigned short>(w.x & 0xFFFFu))),
                       __half2float(__ushort_as_half(static_cast<unsigned short>(w.x >> 16))),
                       __half2float(__ushort_as_half(static_cast<unsigned short>(w.y & 0xFFFFu))),
                       __half2float(__ushort_as_half(static_cast<unsigned short>(w.y >> 16))));
}

// Areas of the intersection and of the union of two boxes that overlap (false: they do not), every operation rounded on
// its own.  (Plain operators without contraction: __fmul_rn is an ordinary product to this compiler, which fused that of one
// area into the sum of both -- IoU(a, b) was not IoU(b, a).  It costs an instruction a pair: [16,80,8400] 26.0 us either way.)
__device__ __forceinline__ bool nms_areas(const float4 &a, const float4 &b, float &inter, float &uni) {
#pragma clang fp contract(off)
    const float x1 = fmaxf(a.x, b.x), y1 = fmaxf(a.y, b.y), x2 = fminf(a.z, b.z), y2 = fminf(a.w, b.w);
    if (x2 <= x1 || y2 <= y1) return false;
    inter = (x2 - x1) * (y2 - y1);
    const float area_a = (a.z - a.x) * (a.w - a.y);
    const float area_b = (b.z - b.x) * (b.w - b.y);
    uni = (area_a + area_b) - inter;
    return true;
}

__device__ __forceinline__ float nms_iou(const float4 &a, const float4 &b) {
    float inter, uni;
    if (!nms_areas(a, b, inter, uni)) return 0.f;
    return uni > 0.f ? __fdiv_rn(inter, uni) : 0.f;
}

// IoU(a, b) > threshold, the division left out where the comparison does not need it: with t = threshold
// and f = fl(t * uni), away from underflow and overflow inter > f (1 + 2^-21) means a quotient above t (1 + 2^-22)
// (f is within 2^-24 of t * uni), whose rounding lies above t, and inter < f (1 - 2^-21) one below t, whose
// rounding does not.  It is a third of the instructions of the whole, paid for every pair of a block.  (The walk of
// more than kNmsRankSortMax candidates divides: its loop ends at the first overlap, and the branches around the
// division cost it more than that -- [8,80,2048] all candidates 288 us, by products 325; [1,1,2048] 698 / 747.)
__device__ __forceinline__ bool nms_overlap(const float4 &a, const float4 &b, float threshold) {
    float inter, uni;
    if (!nms_areas(a, b, inter, uni)) return 0.f > threshold;
    const float f = __fmul_rn(threshold, uni);
    const bool plain = threshold > 0x1p-20f && threshold < 0x1p20f && f > 0x1p-80f && f < 0x1p80f;
    const bool above = inter > __fmul_rn(f, 1.f + 0x1p-21f), below = inter < __fmul_rn(f, 1.f - 0x1p-21f);
    if (plain && (above || below)) return above;
    return (uni > 0.f ? __fdiv_rn(inter, uni) : 0.f) > threshold;
}

// ---- a pair's records, by the workgroup that selected them ---------------------------------------
// What a workgroup publishes: under the call's tag of 40 bits, its number of records (at most 2048), whether boxes were left out, and
// whether it has given up waiting.  No other call has the tag, so nothing has to be cleared, whatever operator the workspace served
// before.  (It is an argument of the launch.  In a recording, whose every replay has the same arguments, the words of the replay
// before would pass for this one's: a recorded call takes the two launches.  A word of the workspace that every replay moves
// on does not tell them apart: it is scratch to the other operators.)
struct NmsJoined {
    uint64_t *words;  // a word a pair, kNmsCopies times, then the tag of the call that a workgroup last gave up in
    int32_t *out, *out_count;
    uint32_t capacity, polls;
    uint64_t tag;  // 1 .. 2^40 - 1
};
// Copies of the words, each read by every eighth workgroup: a thousand that read the same few lines again and again wait for each
// other ([16,80,8400] f32 18.5 us with one copy, 17.0 with 8, 17.1 with 32).
constexpr uint32_t kNmsCopies = 8;
__host__ __device__ constexpr uint32_t nms_copy_stride(uint32_t pairs) { return (pairs + 31u) / 32u * 32u; }
constexpr size_t nms_words(uint32_t pairs) { return static_cast<size_t>(kNmsCopies) * nms_copy_stride(pairs) + 1; }
constexpr uint32_t kNmsCount = 0xFFFFu, kNmsOver = 1u << 16, kNmsGaveUp = 1u << 17;
__device__ __forceinline__ void nms_put_record(int32_t *out, uint32_t capacity, uint32_t at, int32_t batch, int32_t cls, int32_t box) {
    if (at >= capacity) return;
    out[static_cast<size_t>(at) * 3 + 0] = batch;
    out[static_cast<size_t>(at) * 3 + 1] = cls;
    out[static_cast<size_t>(at) * 3 + 2] = box;
}
// The end of a call, one thread: the number of all records, the overflow flag, and the (-1, -1, -1) behind the last record.
__device__ __forceinline__ void nms_put_total(const NmsJoined &j, uint32_t total, bool over) {
    j.out_count[0] = static_cast<int32_t>(total);
    j.out_count[1] = over ? 1 : 0;
    nms_put_record(j.out, j.capacity, total, -1, -1, -1);
}
// The records of workgroups that gave up, as far as all the pairs before them have arrived: a wave.  (Two that find the same ones
// write the same.)
__device__ __forceinline__ void nms_place_late(const NmsJoined &j, const int32_t *selected, uint32_t pairs, uint32_t C, uint32_t max_sel) {
    const uint32_t lane = threadIdx.x & (kWave - 1);
    uint32_t total = 0, over = 0;
    for (uint32_t base = 0; base < pairs; base += kWave) {
        const uint32_t q = base + lane;
        const uint64_t word = q < pairs ? fetch(j.words + q) : j.tag << 24;
        const uint64_t absent = __ballot((word >> 24) != j.tag);
        const uint32_t w = static_cast<uint32_t>(word), have = absent != 0ull ? static_cast<uint32_t>(__builtin_ctzll(absent)) : static_cast<uint32_t>(kWave);
        const uint32_t incl = wave_inclusive_sum_u32(w & kNmsCount);
        over |= w & kNmsOver;
        for (uint64_t left = __ballot(lane < have && (w & kNmsGaveUp) != 0u); left != 0ull; left &= left - 1ull) {
            const int l = static_cast<int>(__builtin_ctzll(left));
            const uint32_t m = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(w), l)) & kNmsCount;
            const uint32_t first = total + static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(incl), l)) - m;
            const uint32_t of = base + static_cast<uint32_t>(l);
            for (uint32_t r = lane; r < m; r += kWave) {
                const int32_t box = __hip_atomic_load(selected + static_cast<size_t>(of) * max_sel + r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                nms_put_record(j.out, j.capacity, first + r, static_cast<int32_t>(of / C), static_cast<int32_t>(of % C), box);
            }
        }
        if (have != static_cast<uint32_t>(kWave)) return;
        total += static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(incl), kWave - 1));
    }
    const bool any_over = __ballot(over != 0u) != 0ull;
    if (lane == 0) nms_put_total(j, total, any_over);
}
// All threads call, behind a barrier after the last write to picks (LDS: the n selected boxes in order).  The wait needs no
// particular number of workgroups on the chip to end: after `polls` looks a workgroup leaves its boxes in its segment, says so, and
// looks once more; one that has published then looks whether any has.  Each does so after its own word is in memory, so that
// at least one of the two finds the other, and the records are placed.  (A counter of the workgroups that are done, on whose
// last one the rest could be left, costs their turns at one address: 1280 of them 10 us.)
template <int NT>
__device__ __forceinline__ void place_records(const NmsJoined &j, const uint32_t *picks, uint32_t n, bool over, int32_t *selected,
                                              uint32_t pair, uint32_t pairs, uint32_t C, uint32_t max_sel, uint32_t *scratch) {
    constexpr int NW = NT / kWave, U = NT >= 1024 ? 2 : 6;
    const uint32_t tid = threadIdx.x, lane = tid & (kWave - 1), wave = uniform_u32(tid) / kWave;
    const uint64_t tag = j.tag, own = (tag << 24) | (over ? kNmsOver : 0u) | n;
    const uint32_t stride = nms_copy_stride(pairs);
    uint64_t *late_word = j.words + kNmsCopies * stride;
    if (tid < kNmsCopies) publish(j.words + tid * stride + pair, own);
    const uint64_t *words = j.words + pair % kNmsCopies * stride;
    uint32_t before = 0, flags = over ? kNmsOver : 0u;
    for (uint32_t base = 0; base < pair; base += U * NT) {
        uint64_t w[U];
        auto at = [&](int u) { return base + static_cast<uint32_t>(u) * NT + tid; };
#pragma unroll
        for (int u = 0; u < U; u++) w[u] = at(u) < pair ? fetch(words + at(u)) : tag << 24;
        for (uint32_t poll = 0;; poll++) {
            bool absent = false;
#pragma unroll
            for (int u = 0; u < U; u++) absent = absent || (w[u] >> 24) != tag;
            if (!absent) break;
            if (poll >= j.polls) {
                flags |= kNmsGaveUp;
                break;
            }
            __builtin_amdgcn_s_sleep(1);
#pragma unroll
            for (int u = 0; u < U; u++)
                if ((w[u] >> 24) != tag) w[u] = fetch(words + at(u));
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            before += static_cast<uint32_t>(w[u]) & kNmsCount;
            flags |= static_cast<uint32_t>(w[u]) & kNmsOver;
        }
    }
    before = wave_sum(before);
    flags = (__ballot((flags & kNmsOver) != 0u) != 0ull ? kNmsOver : 0u) | (__ballot((flags & kNmsGaveUp) != 0u) != 0ull ? kNmsGaveUp : 0u);
    drain_stores();  // (this workgroup's word: its loads have come back behind it)
    if (lane == 0) {
        scratch[wave] = before;
        scratch[NW + wave] = flags;
    }
    __syncthreads();
    before = flags = 0;
#pragma unroll
    for (int w = 0; w < NW; w++) {
        before += scratch[w];
        flags |= scratch[NW + w];
    }
    if ((flags & kNmsGaveUp) != 0u) {  // (the same in every thread)
        for (uint32_t r = tid; r < n; r += NT)
            __hip_atomic_store(selected + static_cast<size_t>(pair) * max_sel + r, static_cast<int32_t>(picks[r]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        drain_stores();
        __syncthreads();
        if (wave != 0) return;
        if (lane == 0) {
            publish(j.words + pair, own | kNmsGaveUp);
            publish(late_word, tag);
        }
        drain_stores();
        nms_place_late(j, selected, pairs, C, max_sel);
        return;
    }
    const uint64_t late = wave == 0 ? fetch(late_word) : 0ull;
    const int32_t batch = static_cast<int32_t>(pair / C), cls = static_cast<int32_t>(pair % C);
    for (uint32_t r = tid; r < n; r += NT) nms_put_record(j.out, j.capacity, before + r, batch, cls, static_cast<int32_t>(picks[r]));
    if (pair == pairs - 1 && tid == 0) nms_put_total(j, before + n, (flags & kNmsOver) != 0u);
    if (wave == 0 && late == tag) nms_place_late(j, selected, pairs, C, max_sel);
}

// Without JOINED: counts[pair] = boxes selected; counts[pairs + pair] = 1 if more than
// kNmsMaxCandidates boxes passed the score threshold (the later ones were left out).
// selected: [pairs][max_sel] box indices.  Launch: B * C workgroups of NT threads:
// 1024 when there are few pairs (one pair's work spread wide), 256 when there are
// enough pairs to put many workgroups on a CU, so that one's score loads overlap
// another's sort and walk.  With more than kNmsRankSortMax candidates each thread keeps the
// boxes of its own kNmsMaxCandidates / NT sorted ones in registers.
// What bounds it: the scores from HBM, the last of them there 6.3 us after the first workgroup's
// start of [16,80,8400] f32 (7 TB/s), and then each workgroup's own chain, 6 us: the list of candidates 2.7, sort and
// boxes 1.3, the block's overlaps 1.5, its kept set 0.4 (a second block, one pair in twenty, 1.6).  A chain this
// short is bound by instruction fetch as much as by anything: a launch finds none of its code in the CUs' caches,
// and forms of these steps that run fewer instructions out of more code were slower, step by step.  us a call with the
// records, 0.25 / 0.45, 51 kept a pair: [16,80,8400] f32 26.1 -> 18.5 -> 17.2 (by place_records), f16 24.1 -> 16.5 -> 15.7; [16,91,8399]
// f32 27.0 -> 18.7 -> 17.1; [1,80,8400] f32 11.6 -> 9.9 -> 8.3; [8,91,1917] f32 15.2 -> 11.6; [16,20,8400], 400 candidates, 26.1 -> 24.7 -> 23.2;
// [8,80,400] all candidates 33.4 -> 29.3; more than 2048 of 8400 ([4,4,8400], the list made twice) 64.2 -> 64.6.
// JOINED: the records too (joined); else nms_pack_kernel follows.
// WHOLE: N is a multiple of four, and no load needs the step for a row's end (it costs a row that has one 0.4 us).
template <typename T, int NT, bool WHOLE, bool JOINED>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(NT >= 1024 ? 8 : 6))) void nms_kernel(
    const T *__restrict__ boxes, const T *__restrict__ scores, int32_t *__restrict__ selected, uint32_t *__restrict__ counts,
    uint32_t pairs, uint32_t C, uint32_t N, int center_point_box, uint32_t max_out, float iou_threshold, float score_threshold,
    uint32_t max_sel, NmsJoined joined) {
    static_assert(NT % kWave == 0 && kNmsMaxCandidates % NT == 0 && (kNmsRankSortMax % NT == 0 || NT % kNmsRankSortMax == 0), "workgroup size");
    constexpr int NW = NT / kWave;
    constexpr int PER = kNmsMaxCandidates / NT;      // sorted candidates per thread
    constexpr int JP = kWave / NW;                   // candidates of a block each wave tests the block against
    constexpr int TILES = NT >= 1024 ? 12 : 36;      // scores per thread and round
    __shared__ __align__(16) uint64_t comp[kNmsMaxCandidates];
    __shared__ float4 block_box[2][kWave];
    __shared__ unsigned long long active[kNmsMaxCandidates / 64];
    __shared__ unsigned long long block_cols[kWave];
    __shared__ unsigned long long block_keep, block_gone;
    __shared__ uint32_t wave_n[2][NW], listed;
    // the selected boxes, where nothing else of a step lies any more: the list before its sort, or sorted candidates at or below the block's
    typedef uint32_t __attribute__((may_alias)) Pick;
    Pick *const picks = reinterpret_cast<Pick *>(comp);
    const uint32_t tid = threadIdx.x, lane = tid & (kWave - 1), wave = uniform_u32(tid) / kWave;  // (scalar)
    const uint32_t pair = blockIdx.x, batch = pair / C;
    const T *srow = scores + static_cast<size_t>(pair) * N;
    const T *brow = boxes + static_cast<size_t>(batch) * N * 4;
    if (tid < static_cast<uint32_t>(kNmsMaxCandidates / 64)) active[tid] = ~0ull;  // positions at or after K are masked where read
    if (tid >= NT - kWave) block_cols[lane] = 0;
    if (tid == 0) block_gone = 0, listed = 0;
    for (uint32_t t = tid; t < static_cast<uint32_t>(kNmsRankSortMax); t += NT) comp[t] = 0;  // (below every real composite)
    __syncthreads();

    // ---- 1. candidates, in any order (2. sorts them) -----------------------------------
    // A round covers NT * TILES boxes, each wave a contiguous run of them (tiles of 64), so that all of a thread's
    // scores are in flight together.  A lane marks its vectors that hold a candidate in a word, and the wave takes
    // them out a vector a lane at a time: few lanes of a detection head have any.  What counts is how much code a wave
    // comes by: with places by ballots, tile by tile in box order, these were 14 KB, and 4.2 us of [16,80,8400] from the
    // scores' arrival to the list where they are 2.7 now.
    uint32_t found = 0;  // the same in every thread
    if (!WHOLE && N < 4) {  // (rows shorter than a load)
        for (uint32_t i = 0; i < N; i++) {
            const float v = load_elem(srow, i);
            if (v > score_threshold) {  // (the same in every thread)
                if (tid == 0) comp[found] = composite(order_key(v), i);
                found++;
            }
        }
        __syncthreads();
    } else {
        // A lane takes four consecutive scores with one load, at any alignment.
        constexpr int VT = TILES / 4;
        for (uint32_t base = 0; base < N; base += NT * TILES) {  // (to the end: the count tells whether boxes were left out)
            const uint32_t tiles = min(static_cast<uint32_t>(VT), (N - base + NT * 4 - 1) / (NT * 4));  // per wave, this round
            const uint32_t wave_first = base + wave * tiles * (kWave * 4);
            float4 s[VT];
#pragma unroll
            for (int u = 0; u < VT; u++)  // (past the end of the row: its last four again, masked out below)
                s[u] = nms_load4(srow + min(wave_first + static_cast<uint32_t>(u) * (kWave * 4) + lane * 4, N - 4));
            if constexpr (!WHOLE) {
                // the four that the row's end cuts short, moved into place (-inf is above no threshold)
#pragma unroll
                for (int u = 0; u < VT; u++) {
                    const uint32_t t0 = wave_first + static_cast<uint32_t>(u) * (kWave * 4);
                    if (t0 < N && N - t0 < kWave * 4) {  // (the same in every lane)
                        const uint32_t e0 = t0 + lane * 4, by = e0 - (N - 4);
                        const float4 v = s[u];
                        if (e0 > N - 4 && e0 < N)
                            s[u] = make_float4(by == 1 ? v.y : by == 2 ? v.z : v.w, by == 1 ? v.z : by == 2 ? v.w : -INFINITY, by == 1 ? v.w : -INFINITY, -INFINITY);
                    }
                }
            }
            // bit u of the lane's word: some score of vector u is above the threshold
            uint32_t word = 0;
#pragma unroll
            for (int u = 0; u < VT; u++)
                word |= fmaxf(fmaxf(s[u].x, s[u].y), fmaxf(s[u].z, s[u].w)) > score_threshold ? 1u << u : 0u;
            // vectors of the lane within the row and the round: the first of them, as the row ends after them
            const int32_t reach = static_cast<int32_t>(min(N - min(N, wave_first), tiles * (kWave * 4))) - static_cast<int32_t>(lane * 4);
            word &= (1u << (reach > 0 ? (static_cast<uint32_t>(reach) + kWave * 4 - 1) / (kWave * 4) : 0u)) - 1u;
            uint32_t own_listed = 0;  // (0, but for all that the compiler knows another one in every lane: it would add up over the lanes)
            asm("" : "+v"(own_listed));
            for (;;) {
                const bool any = word != 0u;
                const uint64_t some = __builtin_amdgcn_ballot_w64(any);
                if (some == 0ull) break;
                const uint32_t first = any ? static_cast<uint32_t>(__builtin_ctz(word)) : ~0u;  // (none: zeros below)
                word &= word - 1u;
                // (bitwise selects: by conditions the scores go to scratch memory, to be indexed there)
                uint32_t x[4] = {};
#pragma unroll
                for (int u = 0; u < VT; u++) {
                    const uint32_t on = first == static_cast<uint32_t>(u) ? ~0u : 0u;
                    x[0] |= on & __float_as_uint(s[u].x);
                    x[1] |= on & __float_as_uint(s[u].y);
                    x[2] |= on & __float_as_uint(s[u].z);
                    x[3] |= on & __float_as_uint(s[u].w);
                }
                uint32_t above = 0;
#pragma unroll
                for (int c = 0; c < 4; c++) above |= __uint_as_float(x[c]) > score_threshold ? 1u << c : 0u;
                above = any ? above : 0u;
                const uint32_t box0 = wave_first + first * (kWave * 4) + lane * 4;
                // room for n more, and this lane's place behind the lanes below it
                auto reserve = [&](uint32_t n) -> uint32_t {
                    uint32_t at = 0;
                    if (lane == 0) at = atomicAdd(&listed + own_listed, n);
                    return uniform_u32(at);
                };
                if (__builtin_amdgcn_ballot_w64((above & (above - 1u)) != 0u) == 0ull) {
                    // one a lane, the rule (a quarter of the instructions behind the selects)
                    const uint32_t at = reserve(static_cast<uint32_t>(__popcll(some))) + lanes_below(some);
                    const uint32_t c = static_cast<uint32_t>(__builtin_ctz(above | 8u));
                    const uint32_t v = c == 0u ? x[0] : c == 1u ? x[1] : c == 2u ? x[2] : x[3];
                    if (any && at < static_cast<uint32_t>(kNmsMaxCandidates)) comp[at] = composite(order_key(__uint_as_float(v)), box0 + c);
                } else {
                    uint64_t mask[4];
                    uint32_t n = 0;
#pragma unroll
                    for (int c = 0; c < 4; c++) {
                        mask[c] = __builtin_amdgcn_ballot_w64((above & (1u << c)) != 0u);
                        n += static_cast<uint32_t>(__popcll(mask[c]));
                    }
                    uint32_t at = reserve(n);
#pragma unroll
                    for (int c = 0; c < 4; c++) {
                        const uint32_t place = at + lanes_below(mask[c]);
                        if ((above & (1u << c)) != 0u && place < static_cast<uint32_t>(kNmsMaxCandidates))
                            comp[place] = composite(order_key(__uint_as_float(x[c])), box0 + static_cast<uint32_t>(c));
                        at += static_cast<uint32_t>(__popcll(mask[c]));
                    }
                }
            }
        }
        __syncthreads();
        found = listed;
        if (found > static_cast<uint32_t>(kNmsMaxCandidates)) {  // (the same in every thread)
            // more than the list holds: the first ones in box order, of the whole row again
            uint32_t have = 0;
            for (uint32_t base = 0, round = 0; base < N && have < static_cast<uint32_t>(kNmsMaxCandidates); base += NT, round++) {
                const uint32_t i = base + tid;
                const float v = load_elem(srow, min(i, N - 1u));
                const uint64_t mask = __ballot(i < N && v > score_threshold);
                if (lane == 0) wave_n[round & 1u][wave] = static_cast<uint32_t>(__popcll(mask));
                __syncthreads();
                uint32_t at = have + lanes_below(mask);
                for (int w = 0; w < NW; w++) {
                    const uint32_t c = wave_n[round & 1u][w];
                    at += (static_cast<uint32_t>(w) < wave) ? c : 0u;
                    have += c;
                }
                if (((mask >> lane) & 1ull) && at < static_cast<uint32_t>(kNmsMaxCandidates)) comp[at] = composite(order_key(v), i);
            }
            __syncthreads();
        }
    }
    const uint32_t K = min(found, static_cast<uint32_t>(kNmsMaxCandidates));

    // ---- 2. by score, largest first; equal scores: lower box index first --------------
    if (K > static_cast<uint32_t>(kNmsRankSortMax)) {
        uint32_t p2 = 1;
        while (p2 < K) p2 <<= 1;
        for (uint32_t t = K + tid; t < p2; t += NT) comp[t] = 0;  // below every real composite
        __syncthreads();
        bitonic_sort_desc<NT>(comp, p2);
    }
    // a candidate's box, and its corners
    auto box_of = [&](uint64_t c) {
        const T *r = brow + static_cast<size_t>(composite_index(c)) * 4;
        return make_float4(load_elem(r, 0), load_elem(r, 1), load_elem(r, 2), load_elem(r, 3));
    };
    auto corners = [&](float4 b) {
#pragma clang fp contract(off)
        if (center_point_box) {  // (x_center, y_center, width, height), shaders/nms.comp:55-58
            const float hw = b.z * 0.5f, hh = b.w * 0.5f;
            b = make_float4(b.x - hw, b.y - hh, b.x + hw, b.y + hh);
        }
        return b;
    };
    const uint32_t limit = max_out > 0 ? min(max_out, K) : K;
    uint32_t chosen = 0;
    // b. (both walks) the first wave resolves a block.  Kept = alive and suppressed by nobody kept before it: that set
    //    is the only fixed point of  S -> { i alive : no member of S suppresses i },  and iterating from any S
    //    reaches it, one more leading position settled per step at worst, a handful of steps as a rule.
    auto resolve = [&](const uint64_t *sorted, uint32_t base, bool alive, unsigned long long col) -> uint64_t {
        uint64_t keep = __ballot(alive);
        for (int step = 0; step < kWave; step++) {
            const uint64_t next = __ballot(alive && (col & keep) == 0);
            if (next == keep) break;
            keep = next;
        }
        const uint32_t room = limit - chosen;  // > 0 here
        if (static_cast<uint32_t>(__popcll(keep)) > room) keep = __ballot(((keep >> lane) & 1ull) && lanes_below(keep) < room);
        if (lane == 0) block_keep = keep;
        if ((keep >> lane) & 1u) {
            const uint32_t slot = chosen + lanes_below(keep);
            const uint32_t box = composite_index(sorted[base + lane]);
            if (JOINED) picks[slot] = box;
            else if (slot < max_sel) selected[static_cast<size_t>(pair) * max_sel + slot] = static_cast<int32_t>(box);
        }
        return keep;
    };
    auto finish = [&](bool over) __attribute__((always_inline)) {
        if constexpr (JOINED) {
            place_records<NT>(joined, picks, min(chosen, max_sel), over, selected, pair, pairs, C, max_sel, &wave_n[0][0]);
        } else if (tid == 0) {
            counts[pair] = min(chosen, max_sel);
            counts[pairs + pair] = over ? 1u : 0u;
        }
    };
    auto uniform_keep = [&]() -> uint64_t {
        const unsigned long long kept = block_keep;
        return (static_cast<uint64_t>(uniform_u32(static_cast<uint32_t>(kept >> 32))) << 32) | uniform_u32(static_cast<uint32_t>(kept));
    };

    // ---- 3a. up to 512 candidates: sorted list and boxes in the LDS behind the unsorted list -----------------
    if (K <= static_cast<uint32_t>(kNmsRankSortMax)) {
        static_assert(kNmsMaxCandidates * sizeof(uint64_t) >= kNmsRankSortMax * (2 * sizeof(uint64_t) + sizeof(float4)), "two lists and the boxes");
        float4 *box = reinterpret_cast<float4 *>(comp + kNmsRankSortMax);
        uint64_t *sorted = comp + kNmsMaxCandidates - kNmsRankSortMax;
        // Each candidate counts the composites above its own (all distinct) and moves there, its box, loaded under the
        // counting, with it: nothing is written where others still read, one barrier for all of it.
        constexpr int PART = NT >= kNmsRankSortMax ? 1 : kNmsRankSortMax / NT;  // candidates a thread
        uint64_t c[PART];
        uint32_t rank[PART];
        float4 own[PART];
#pragma unroll
        for (int e = 0; e < PART; e++) {
            const uint32_t p = static_cast<uint32_t>(e) * NT + tid;
            c[e] = p < K ? comp[p] : 0;
            rank[e] = 0;
            own[e] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (p < K) own[e] = box_of(c[e]);
        }
#pragma unroll
        for (int e = 0; e < PART; e++) {
            if (wave * kWave + static_cast<uint32_t>(e) * NT < K) {  // (the same for the whole wave)
#pragma unroll 1
                for (uint32_t q = 0; q < K; q += 16u) {  // (the list ends in zeros)
                    const uint4 *src = reinterpret_cast<const uint4 *>(comp + q);
                    uint4 o[8];
#pragma unroll
                    for (int u = 0; u < 8; u++) o[u] = src[u];
                    __builtin_amdgcn_sched_barrier(0);  // (all in flight: one at a time 400 candidates took 9.4 us, 6.3 so)
#pragma unroll
                    for (int u = 0; u < 8; u++) {
                        rank[e] += ((static_cast<uint64_t>(o[u].y) << 32) | o[u].x) > c[e] ? 1u : 0u;
                        rank[e] += ((static_cast<uint64_t>(o[u].w) << 32) | o[u].z) > c[e] ? 1u : 0u;
                    }
                }
            }
        }
#pragma unroll
        for (int e = 0; e < PART; e++) {
            if (static_cast<uint32_t>(e) * NT + tid < K) {
                sorted[rank[e]] = c[e];
                box[rank[e]] = corners(own[e]);
            }
        }
        __syncthreads();
        for (uint32_t base = 0; base < K && chosen < limit; base += kWave) {
            const uint32_t in_block = min(static_cast<uint32_t>(kWave), K - base);
            // (a block of at most 32, 16 ... candidates: two, four ... lanes each, that share its tests)
            const uint32_t spread = in_block > 1u ? static_cast<uint32_t>(__clz(in_block - 1u)) - 26u : 6u;  // its logarithm
            const uint32_t i = min(lane & ((kWave >> spread) - 1u), in_block - 1u);
            const uint32_t part = (wave << spread) + (lane >> (6u - spread)), parts = static_cast<uint32_t>(NW) << spread;
            const float4 bi = box[base + i];
            // a. for candidate i of the block (one per lane, in every wave), a share of the boxes kept so far and of
            //    the other candidates of the block.  An overlap is the same from either side: candidate i is tested against
            //    the in_block / 2 that follow it, cyclically, and every pair of the block is met once (the farthest of
            //    an even number twice).  Two rolled loops, the next box in flight: unrolled by four, every pair from
            //    both sides, 2.6 us of [16,80,8400], 1.5 so; with the areas left to a second pass over the few pairs that
            //    overlap at all 1.6, and 4.9 against 3.6 for 400 candidates.
            bool dead = false;
            float4 next = box[part < chosen ? part : 0u];
#pragma unroll 1
            for (uint32_t r = part; r < chosen;) {
                const float4 other = next;
                r += parts;
                next = box[r < chosen ? r : 0u];
                dead = nms_overlap(bi, other, iou_threshold) || dead;
            }
            const uint32_t around = in_block / 2u;
            uint32_t j = i + 1u + part;
            j = j >= in_block ? j - in_block : j;
            next = box[base + min(j, in_block - 1u)];
#pragma unroll 1
            for (uint32_t d = part; d < around; d += parts) {
                const float4 other = next;
                const uint32_t at = j;
                j += parts;
                j = j >= in_block ? j - in_block : j;
                next = box[base + min(j, in_block - 1u)];
                if (nms_overlap(bi, other, iou_threshold)) atomicOr(&block_cols[max(i, at)], 1ull << min(i, at));
            }
            unsigned long long gone = __ballot(dead);
            for (uint32_t by = kWave >> spread; by < kWave; by *= 2u) gone |= gone >> by;  // (the sums of parts: the lowest bits count)
            if (lane == 0 && gone != 0) atomicOr(&block_gone, gone);
            __syncthreads();
            if (wave == 0) {
                const unsigned long long col = block_cols[lane], out_of = block_gone;
                block_cols[lane] = 0;  // for the next block (its additions come after the next barrier)
                if (lane == 0) block_gone = 0;
                const uint64_t keep = resolve(sorted, base, lane < in_block && !((out_of >> lane) & 1ull), col);
                // (places at or below the block's own, which no one reads any more)
                if ((keep >> lane) & 1ull) box[chosen + lanes_below(keep)] = bi;
            }
            __syncthreads();
            chosen += static_cast<uint32_t>(__popcll(uniform_keep()));
        }
        finish(false);
        return;
    }

    float4 mine[PER];  // corners of this thread's candidates: sorted positions e * NT + tid
#pragma unroll
    for (int e = 0; e < PER; e++) {
        const uint32_t p = static_cast<uint32_t>(e) * NT + tid;
        mine[e] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (p < K) mine[e] = corners(box_of(comp[p]));
    }

    // ---- 3b. more: 64 candidates at a time, each thread with its own --------------------------------
    for (uint32_t base = 0; base < K && chosen < limit; base += kWave) {
        // the block's boxes go to LDS: its 64 positions belong to the lanes of one wave (two buffers in turn:
        // the block before may still be read by slower waves in step c)
        float4(&box)[kWave] = block_box[(base / kWave) & 1u];
        if (wave == (base % NT) / kWave) {
            float4 b = mine[0];
#pragma unroll
            for (int e = 1; e < PER; e++)
                if (static_cast<uint32_t>(e) == base / NT) b = mine[e];
            box[lane] = b;
        }
        __syncthreads();
        // a. for candidate i of the block (one per lane, in every wave) the earlier candidates of the block that
        //    would suppress it: each wave tests JP of them and adds its bits to the lane's word
        //    (positions at or after K hold zeros: they are never active below)
        const float4 bi = box[lane];
        uint32_t bits = 0;
#pragma unroll
        for (int r = 0; r < JP; r++) {
            const uint32_t j = wave * JP + static_cast<uint32_t>(r);
            if (lane > j && nms_iou(bi, box[j]) > iou_threshold) bits |= 1u << r;
        }
        if (bits != 0) atomicOr(&block_cols[lane], static_cast<unsigned long long>(bits) << (wave * JP));
        __syncthreads();  // (also: the bits cleared by the block before are in place)
        if (wave == 0) {
            const unsigned long long col = block_cols[lane];
            block_cols[lane] = 0;  // for the next block (its additions come after the next barrier)
            resolve(comp, base, base + lane < K && ((active[base / kWave] >> lane) & 1ull), col);
        }
        __syncthreads();
        const uint64_t keep = uniform_keep();
        chosen += static_cast<uint32_t>(__popcll(keep));
        if (chosen >= limit) break;
        // c. every later candidate still active against the block's survivors
#pragma unroll
        for (int e = 0; e < PER; e++) {
            const uint32_t p = static_cast<uint32_t>(e) * NT + tid;
            if (p >= base + kWave && p < K && ((active[p / 64] >> (p % 64)) & 1ull)) {
                bool dead = false;
                for (uint64_t kk = keep; kk != 0 && !dead; kk &= kk - 1)
                    dead = nms_iou(mine[e], box[static_cast<uint32_t>(__builtin_ctzll(kk))]) > iou_threshold;
                if (dead) atomicAnd(&active[p / 64], ~(1ull << (p % 64)));
            }
        }
        // (no barrier here: the next block writes the other box buffer, and its barriers order the rest)
    }
    finish(found > static_cast<uint32_t>(kNmsMaxCandidates));
}

// The records of all pairs one after the other.  out: [capacity][3]; out_count[0] =
// records in all (also when capacity holds fewer), out_count[1] = 1 if some pair
// had more candidates than kNmsMaxCandidates; a (-1,-1,-1) record follows the last
// one when capacity allows.  Launch: a workgroup of 256 for every kNmsPackPairs pairs, a wave a pair.
// What bounds it: its round trips to memory, so a thread's counts are loaded eight at a time, under them the
// first selected boxes, and only the last workgroup asks for overflows ([16,80,8400], the shortest and the mean: a workgroup a pair, a count at a time 4.2 and 4.4 us, so 2.6 and 4.0).
constexpr uint32_t kNmsPackPairs = 256 / kWave;
__global__ __launch_bounds__(256) void nms_pack_kernel(const int32_t *__restrict__ selected,
                                                              const uint32_t *__restrict__ counts, int32_t *__restrict__ out,
                                                              int32_t *__restrict__ out_count, uint32_t pairs, uint32_t C,
                                                              uint32_t max_sel, uint32_t capacity) {
    __shared__ uint32_t scratch[kNmsPackPairs];
    const uint32_t tid = threadIdx.x, lane = tid & (kWave - 1), wave = uniform_u32(tid) / kWave;  // (scalar)
    const uint32_t first = blockIdx.x * kNmsPackPairs, pair = first + wave;
    const bool here = pair < pairs;
    const int32_t *mine = selected + static_cast<size_t>(here ? pair : first) * max_sel;
    int32_t head = mine[min(lane, max_sel - 1u)];  // (read whether or not the pair has as many: the segment has)
    // the pairs of the workgroup up to the wave's own, in the lanes of every wave
    const uint32_t beside = lane <= wave && first + lane < pairs ? counts[first + lane] : 0u;
    uint32_t before = 0;
    for (uint32_t base = 0; base < first; base += 8u * 256u) {
        uint32_t c[8];
#pragma unroll
        for (uint32_t u = 0; u < 8; u++) {
            const uint32_t q = base + u * 256u + tid;
            c[u] = counts[min(q, first - 1u)];
        }
#pragma unroll
        for (uint32_t u = 0; u < 8; u++) before += base + u * 256u + tid < first ? c[u] : 0u;
    }
    before = wave_sum(before);
    if (lane == 0) scratch[wave] = before;
    __syncthreads();
    uint32_t offset = 0;
#pragma unroll
    for (uint32_t w = 0; w < kNmsPackPairs; w++) offset += scratch[w];
    const uint32_t n = here ? static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(beside), static_cast<int>(wave))) : 0u;
    offset += wave_sum(beside) - n;
    const int32_t batch = static_cast<int32_t>(pair / C), cls = static_cast<int32_t>(pair % C);
    for (uint32_t r = lane; r < n; r += kWave) {
        const uint32_t o = offset + r;
        if (r >= kWave) head = mine[r];
        if (o < capacity) {
            out[static_cast<size_t>(o) * 3 + 0] = batch;
            out[static_cast<size_t>(o) * 3 + 1] = cls;
            out[static_cast<size_t>(o) * 3 + 2] = head;
        }
    }
    if (pair == pairs - 1) {  // (the same for the whole wave)
        uint32_t over = 0;
#pragma unroll 8
        for (uint32_t q = lane; q < pairs; q += kWave) over |= counts[pairs + q];
        const bool any = __ballot(over != 0u) != 0ull;
        if (lane == 0) {
            const uint32_t total = offset + n;
            out_count[0] = static_cast<int32_t>(total);
            out_count[1] = any ? 1 : 0;
            if (total < capacity) {  // end of the list for a reader of the tensor alone (the reference writes such a record too)
                out[static_cast<size_t>(total) * 3 + 0] = -1;
                out[static_cast<size_t>(total) * 3 + 1] = -1;
                out[static_cast<size_t>(total) * 3 + 2] = -1;
            }
        }
    }
}

}  // namespace vkop
