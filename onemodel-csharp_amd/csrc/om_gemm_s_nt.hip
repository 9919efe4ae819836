// Instances of the dense product's kernel (om_gemm_s.hpp), C = A B^T: both operands contiguous along k (Linear forward, attention scores).
#include "om_gemm_s.hpp"

namespace omg {
void launch_s_nt(int cfg, bool exact, const Params &p, unsigned grid, hipStream_t st) {
#define X(ID, TN, MG, KG)                                                                                              \
    if (cfg == ID && exact)                                                                                            \
        hipLaunchKernelGGL((gs::k_gemm_s<TN, MG, KG, false, true, true>), dim3(grid), dim3(64 * MG * KG), 0, st, p);    \
    if (cfg == ID && !exact)                                                                                           \
        hipLaunchKernelGGL((gs::k_gemm_s<TN, MG, KG, false, true, false>), dim3(grid), dim3(64 * MG * KG), 0, st, p);
    OMG_S_CONFIGS(X)
#undef X
}
}  // namespace omg
