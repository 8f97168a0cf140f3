// Instantiates the per-row update kernel for one Gram precision (ALS_PREC is
// set by the build: 0 FP32, 1 BF16, 2 FP16) and one form of the system
// (ALS_AUG: 1 augmented, T = 1..9; 0 f = 16T, T = 1..8), every solver.
// Compiled once per pair so that they build in parallel.
#include "als_device.hpp"

#ifndef ALS_PREC
#error "ALS_PREC must be defined"
#endif
#ifndef ALS_AUG
#error "ALS_AUG must be defined"
#endif

namespace als {

constexpr bool AUG = ALS_AUG != 0;
constexpr int LAST_T = AUG ? MAX_T : MAX_T - 1;
template <int T> using Sys = Geo<T, ALS_PREC, AUG>;

// FN<T>(args) for a tile count known at run time, T in FIRST .. LAST_T; BAD
// outside.
template <int FIRST, class FN, class R>
static R by_tiles(int T, FN fn, R bad) {
    if constexpr (FIRST > LAST_T) return bad;
    else return T == FIRST ? fn(std::integral_constant<int, FIRST>{}) : by_tiles<FIRST + 1>(T, fn, bad);
}

// S at T tiles. Variant 1: one wave per SIMD (no waves-per-EU bound: the
// whole register file for one wave, spill-free at the widest tile counts),
// built for the warm-started solver at f >= 96; selectable per side.
static const void *update_kernel_for(int T, int solve, int variant) {
    return by_tiles<1>(
        T,
        [&](auto t) -> const void * {
            constexpr int N = decltype(t)::value;
            if (variant == 1) {
                if constexpr (Sys<N>::TA >= 7)
                    return solve == SOLVE_CHOL_WARM ? (const void *)&update_kernel<N, ALS_PREC, SOLVE_CHOL_WARM, AUG>
                                                    : nullptr;
                return nullptr;
            }
            if (variant != 0) return nullptr;
            return solve == SOLVE_CHOL  ? (const void *)&update_kernel<N, ALS_PREC, SOLVE_CHOL, AUG>
                   : solve == SOLVE_CG  ? (const void *)&update_kernel<N, ALS_PREC, SOLVE_CG, AUG>
                   : solve == SOLVE_CHOL_WARM
                       ? (const void *)&update_kernel_w2<N, ALS_PREC, SOLVE_CHOL_WARM, AUG>
                       : (const void *)&update_kernel_w2<N, ALS_PREC, SOLVE_CHOL_REFINE, AUG>;
        },
        (const void *)nullptr);
}

// The dual system exists for f >= 64 (Geo::DUAL_TD > 0), after the plain
// Cholesky solve or the warm-started one.
static const void *dual_kernel_for(int T, int solve) {
    return by_tiles<1>(
        T,
        [&](auto t) -> const void * {
            constexpr int N = decltype(t)::value;
            if constexpr (Sys<N>::DUAL_TD > 0)
                return solve == SOLVE_CHOL        ? (const void *)&dual_kernel<N, ALS_PREC, SOLVE_CHOL, AUG>
                       : solve == SOLVE_CHOL_WARM ? (const void *)&dual_kernel<N, ALS_PREC, SOLVE_CHOL_WARM, AUG>
                                                  : nullptr;
            return nullptr;
        },
        (const void *)nullptr);
}

#define ALS_CAT2(a, b, c) a##b##c
#define ALS_CAT(a, b, c) ALS_CAT2(a, b, c)
#if ALS_AUG
#define ALS_NAME(x) ALS_CAT(x##_p, ALS_PREC, a)
#else
#define ALS_NAME(x) ALS_CAT(x##_p, ALS_PREC, b)
#endif

const void *ALS_NAME(update_kernel_ptr)(int T, int solve, int variant) { return update_kernel_for(T, solve, variant); }

int ALS_NAME(update_lds_bytes)(int T, int solve) {
    return by_tiles<1>(
        T,
        [&](auto t) {
            using G = Sys<decltype(t)::value>;
            return solve == SOLVE_CHOL_REFINE ? G::refine_lds_bytes() : G::lds_bytes();
        },
        -1);
}

const void *ALS_NAME(dual_kernel_ptr)(int T, int solve) { return dual_kernel_for(T, solve); }

int ALS_NAME(dual_lds_bytes)(int T) {
    return by_tiles<1>(
        T, [](auto t) { return Sys<decltype(t)::value>::DUAL_TD > 0 ? Sys<decltype(t)::value>::dual_lds_bytes() : 0; }, 0);
}

int ALS_NAME(dual_max_ratings)(int T) {
    return by_tiles<1>(T, [](auto t) { return 16 * Sys<decltype(t)::value>::DUAL_TD; }, 0);
}

}  // namespace als
