// One element type's slice of the register kernel for lines along a non-last axis:
//   hipcc -DVKOP_ROWS_T=float|uint16_t -c lines_inst.hip
#include "kernels_lines.hpp"
#include "rows_launch.hpp"

namespace vkop {

template <typename T> bool launch_softmax_lines(const LinesLaunch &a) {
    constexpr uint32_t L = 16 / sizeof(T);
    const uint32_t per_team = static_cast<uint32_t>(kWave) / a.p, teams = a.w >= 4 ? 1u : 4u / a.w;
    const uint32_t vectors = a.g.outer * ((a.g.inner + L - 1) / L);
    const uint32_t blocks = (vectors + per_team * teams - 1) / (per_team * teams);
    const uint32_t threads = teams * a.w * kWave;
    const size_t lds = a.w > 1 ? static_cast<size_t>(teams) * a.w * per_team * L * sizeof(double) : 0;
    const T *in = static_cast<const T *>(a.in);
    T *out = static_cast<T *>(a.out);
#define VKOP_LINES_CACHED(K, P, WIDE, CACHE) \
    softmax_lines_reg_kernel<T, K, P, false, WIDE, CACHE><<<blocks, threads, lds, a.stream>>>(in, out, a.g, a.w, a.nan_where, a.nan_value)
#define VKOP_LINES_LAUNCH(K, P, WIDE)                                                                                                      \
    if (a.max_only && a.caching == kCacheNone)                                                                                             \
        softmax_lines_reg_kernel<T, K, P, true, WIDE, kCacheNone><<<blocks, threads, lds, a.stream>>>(in, out, a.g, a.w, 0, 0.f);           \
    else if (a.max_only)                                                                                                                   \
        softmax_lines_reg_kernel<T, K, P, true, WIDE, kCacheLoads><<<blocks, threads, lds, a.stream>>>(in, out, a.g, a.w, 0, 0.f);          \
    else if (a.caching == kCacheLoads) VKOP_LINES_CACHED(K, P, WIDE, kCacheLoads);                                                          \
    else if (a.caching == kCacheStores) VKOP_LINES_CACHED(K, P, WIDE, kCacheStores);                                                        \
    else if (a.caching == kCacheBoth) VKOP_LINES_CACHED(K, P, WIDE, kCacheBoth);                                                            \
    else VKOP_LINES_CACHED(K, P, WIDE, kCacheNone)
#define VKOP_LINES(K, P)                                                                                                                   \
    if (a.k == K && a.p == P) {                                                                                                            \
        if (sizeof(T) == 4 || a.w > 1) VKOP_LINES_LAUNCH(K, P, true);                                                                      \
        else VKOP_LINES_LAUNCH(K, P, (sizeof(T) == 4));                                                                                    \
        return true;                                                                                                                       \
    }
#define VKOP_LINES_5_8(P) VKOP_LINES(5, P) VKOP_LINES(6, P) VKOP_LINES(7, P) VKOP_LINES(8, P)
#define VKOP_LINES_9_16(P)                                                                                     \
    VKOP_LINES(9, P) VKOP_LINES(10, P) VKOP_LINES(11, P) VKOP_LINES(12, P) VKOP_LINES(13, P) VKOP_LINES(14, P) \
        VKOP_LINES(15, P) VKOP_LINES(16, P)
    if constexpr (sizeof(T) == 4) {
        VKOP_LINES(1, 1) VKOP_LINES(2, 1) VKOP_LINES(3, 1) VKOP_LINES(4, 1) VKOP_LINES_5_8(1) VKOP_LINES_9_16(1)
        VKOP_LINES(3, 2) VKOP_LINES(4, 2) VKOP_LINES_5_8(2) VKOP_LINES_9_16(2)
        VKOP_LINES(3, 4) VKOP_LINES(4, 4) VKOP_LINES_9_16(4)
        VKOP_LINES(3, 8) VKOP_LINES(4, 8) VKOP_LINES_9_16(8)
        VKOP_LINES(11, 16) VKOP_LINES(12, 16) VKOP_LINES(13, 16) VKOP_LINES(14, 16) VKOP_LINES(15, 16) VKOP_LINES(16, 16)
    }
    VKOP_LINES_5_8(4) VKOP_LINES_5_8(8) VKOP_LINES(3, 16) VKOP_LINES(4, 16) VKOP_LINES_5_8(16)
#undef VKOP_LINES_9_16
#undef VKOP_LINES_5_8
#undef VKOP_LINES
#undef VKOP_LINES_LAUNCH
#undef VKOP_LINES_CACHED
    return false;
}

template bool launch_softmax_lines<VKOP_ROWS_T>(const LinesLaunch &);

}  // namespace vkop
