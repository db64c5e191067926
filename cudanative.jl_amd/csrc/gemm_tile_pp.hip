// Instances of the ping-pong GEMM kernel (see gemm_pingpong.hpp).
#include "gemm_pingpong.hpp"

namespace miw {

template <int BI, int BJ, int WI, int WJ, bool XK, bool YK>
static const void *pp_types(int c_type, int d_type, bool fold)
{
    if constexpr (!pp_fits(BI, BJ, XK, YK)) {
        return nullptr;
    } else {
        if (fold && d_type == 0) return (const void *)k_gemm_pp_fold<BI, BJ, WI, WJ, XK, YK, half_t>;
        if (fold) return (const void *)k_gemm_pp_fold<BI, BJ, WI, WJ, XK, YK, float>;
        if (c_type == 0 && d_type == 0) return (const void *)k_gemm_pp<BI, BJ, WI, WJ, XK, YK, half_t, half_t>;
        if (c_type == 0 && d_type == 1) return (const void *)k_gemm_pp<BI, BJ, WI, WJ, XK, YK, half_t, float>;
        if (c_type == 1 && d_type == 0) return (const void *)k_gemm_pp<BI, BJ, WI, WJ, XK, YK, float, half_t>;
        return (const void *)k_gemm_pp<BI, BJ, WI, WJ, XK, YK, float, float>;
    }
}

template <int BI, int BJ, int WI, int WJ>
static const void *pp_layout(bool xk, bool yk, int c_type, int d_type, bool fold)
{
    if (xk && yk) return pp_types<BI, BJ, WI, WJ, true, true>(c_type, d_type, fold);
    if (xk && !yk) return pp_types<BI, BJ, WI, WJ, true, false>(c_type, d_type, fold);
    if (!xk && yk) return pp_types<BI, BJ, WI, WJ, false, true>(c_type, d_type, fold);
    return pp_types<BI, BJ, WI, WJ, false, false>(c_type, d_type, fold);
}

// Kernel for a bm x bn tile, or null when there is none (tile not instantiated, or its ring does not fit in LDS);
// fold: the one that adds a Float32 C in the K loop.
const void *pp_kernel(int bm, int bn, bool xk, bool yk, int c_type, int d_type, bool fold)
{
    if (bm == 256 && bn == 256) return pp_layout<256, 256, 2, 4>(xk, yk, c_type, d_type, fold);
    return nullptr;
}
// Does k_gemm_pp_fold run the problem?  C Float32, laid out as D, lane offsets into its tile within 32 bits; more k-steps
// than tiles of C, one of which each of the last ones adds; and alpha of 1.  Every MFMA behind C's addition rounds at C's
// magnitude: with |C| of a hundred times |A B| that is three to five times the error of adding it once, behind the loop.
// So alpha = -1 and sixteen slots of K do not take it, although they would gain: 8192x8192x1024, alpha = -1, takes 180 us, 159 with C folded.
bool pp_folds(const tiled_params &p, int c_type)
{
    return p.use_c && c_type == 1 && !p.c_trans && p.alpha == 1.0f && p.ldc < (1l << 22) &&
           (p.K + KGRAN - 1) / KGRAN * 2 > PP_FOLD_STEPS;
}
int pp_lds(int bm, int bn, bool xk, bool yk) { return pp_lds_bytes(bm, bn, xk, yk); }

}  // namespace miw
