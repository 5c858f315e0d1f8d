// vbs_kern_mfma_blk.hip — the batch-1 matrix-core matvec (k_mvf, vbs_mfma.h)
// for the 32-element block types Q4_0, Q4_1 and Q8_0 (plain and accumulating
// launches), in a translation unit of its own so it compiles in parallel.
#include "vbs_mfma.h"

namespace vbs {

hipError_t launch_blk_linear(int type, const uint8_t *w, const float *x, float *y, uint32_t cols,
                             uint32_t rows, int accumulate, hipStream_t s) {
    if (rows == 0 || !mv_fits_blk(type, w, x, cols, rows)) return hipErrorNotSupported;
    // Up to 2048 rows the general kernel (k_rows, vbs_kern_linear.hip) is
    // through sooner: here / there, Q8_0 256 x 4096 4.9 / 2.5 us, 1024 x 4096
    // 5.8 / 3.9, 2048 x 4096 6.0 / 5.0, 2048 x 11008 11.6 / 10.0; Q4_0 2048 x 4096
    // 4.9 / 4.5, 2048 x 11008 9.0 / 8.6; but Q8_0 4096 x 4096 6.9 / 7.1, 4096 x 11008
    // 13.3 / 15.0, Q4_0 4096 x 4096 5.2 / 6.1.
    if (rows <= 2048u) return hipErrorNotSupported;
    MvArgs a{};
    a.w[0] = w;
    a.y[0] = y;
    a.rows[0] = rows;
    a.nmat = 1;
    a.cols = cols;
    a.x = x;
    set_tiles(a);
    if (type == kQ4_0)
        return accumulate ? launch_plan<Q40, false, E_ACC>(a, s) : launch_plan<Q40, false, E_STORE>(a, s);
    if (type == kQ4_1)
        return accumulate ? launch_plan<Q41, false, E_ACC>(a, s) : launch_plan<Q41, false, E_STORE>(a, s);
    return accumulate ? launch_plan<Q80, false, E_ACC>(a, s) : launch_plan<Q80, false, E_STORE>(a, s);
}

}  // namespace vbs
