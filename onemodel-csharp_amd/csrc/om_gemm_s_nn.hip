// Instances of the dense product's kernel (om_gemm_s.hpp), C = A B: B contiguous along n (input gradients).
#include "om_gemm_s.hpp"

namespace omg {
void launch_s_nn(int cfg, bool exact, const Params &p, unsigned grid, hipStream_t st) {
#define X(ID, TN, MG, KG)                                                                                              \
    if (cfg == ID && exact)                                                                                            \
        hipLaunchKernelGGL((gs::k_gemm_s<TN, MG, KG, false, false, true>), dim3(grid), dim3(64 * MG * KG), 0, st, p);    \
    if (cfg == ID && !exact)                                                                                           \
        hipLaunchKernelGGL((gs::k_gemm_s<TN, MG, KG, false, false, false>), dim3(grid), dim3(64 * MG * KG), 0, st, p);
    OMG_S_CONFIGS(X)
#undef X
}
}  // namespace omg
