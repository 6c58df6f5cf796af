// p8x_gemv_rgm.hip -- single-GEMV row-group kernel instantiations: two columns of class-3 tensors, and one column over
// several linears that share their input (p8x_mul_mat_vec_multi / _glu).
#include "p8x_gemv.h"

namespace p8x {

// several linears on one activation vector (one column): the MULTI instantiations
int launch_gemv_rg_multi(int cm, const RgJobs &jobs, int ng, const uint32_t *a2, hipStream_t st) {
    if (cm == kCmC3) return launch_gemv_rg_t<kCmC3, 1, true>(jobs, ng, a2, st);
    if (cm == kCmC234) return launch_gemv_rg_t<kCmC234, 1, true>(jobs, ng, a2, st);
    if (cm == kCmC6) return launch_gemv_rg_t<kCmC6, 1, true>(jobs, ng, a2, st);
    if (cm == kCmC2346) return launch_gemv_rg_t<kCmC2346, 1, true>(jobs, ng, a2, st);
    return launch_gemv_rg_t<kCmAll, 1, true>(jobs, ng, a2, st);
}

int launch_gemv_rg_mc(int ncols, int cm, const RgJobs &job, int ng, const uint32_t *a2, hipStream_t st) {
    if (ncols == 2 && cm == kCmC3) return launch_gemv_rg_t<kCmC3, 2, false>(job, ng, a2, st);
    return set_error(P8X_ERR_UNSUPPORTED, "k_gemv_rg: %d columns, class set %d", ncols, cm);
}

}  // namespace p8x
