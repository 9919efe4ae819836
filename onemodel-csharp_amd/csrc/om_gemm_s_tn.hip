// Instances of the dense product's kernel (om_gemm_s.hpp), C = A^T B: both operands contiguous along their rows (weight gradients, alone and grouped).
#include "om_gemm_s.hpp"

namespace omg {
void launch_s_tn(int cfg, bool exact, const Params &p, unsigned grid, hipStream_t st) {
#define X(ID, TN, MG, KG)                                                                                              \
    if (cfg == ID && exact)                                                                                            \
        hipLaunchKernelGGL((gs::k_gemm_s<TN, MG, KG, true, false, true>), dim3(grid), dim3(64 * MG * KG), 0, st, p);    \
    if (cfg == ID && !exact)                                                                                           \
        hipLaunchKernelGGL((gs::k_gemm_s<TN, MG, KG, true, false, false>), dim3(grid), dim3(64 * MG * KG), 0, st, p);
    OMG_S_CONFIGS(X)
#undef X
}

void launch_s_tn_group(int cfg, bool exact, const GroupParams &g, unsigned grid, hipStream_t st) {
#define X(ID, TN, MG, KG)                                                                                              \
    if (cfg == ID && exact)                                                                                            \
        hipLaunchKernelGGL((gs::k_gemm_s_tn_group<TN, MG, KG, true>), dim3(grid), dim3(64 * MG * KG), 0, st, g);       \
    if (cfg == ID && !exact)                                                                                           \
        hipLaunchKernelGGL((gs::k_gemm_s_tn_group<TN, MG, KG, false>), dim3(grid), dim3(64 * MG * KG), 0, st, g);
    OMG_S_CONFIGS(X)
#undef X
}
}  // namespace omg
