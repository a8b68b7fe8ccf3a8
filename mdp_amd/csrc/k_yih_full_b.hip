// compute_bi on the upstream U layout from LDS-staged half rows, one element (see k_yih.hpp).
#include "k_yih.hpp"

namespace mdp {

// `groups` so that blocks x groups reaches the 256 CUs from 2,048 atoms on, and no more: each group stages the block's U
// again.  15,972 atoms at twojmax 8: 123 us, against 501 for a triple per wave from global memory.
void launch_b_full(const SnapDev& s, const double* Ur, const double* Ui, double* blist, int N, int bnorm,
                   hipStream_t st) {
    if (N <= 0) return;
    const int blocks = (N + 63) / 64;
    const int groups = blocks >= 128 ? 1 : (blocks >= 64 ? 2 : (blocks >= 32 ? 4 : 8));
    const dim3 grid(blocks * groups);
    switch (s.J) {
#define BF_CASE(JV, WV)                                                                                              \
    case JV:                                                                                                         \
        hipLaunchKernelGGL((k_b_half<JV, WV, true, true>), grid, dim3(64 * WV), 0, st, s.cg, Ur, Ui, blist, N, bnorm, \
                           groups);                                                                                  \
        break;
        BF_CASE(2, 4)
        BF_CASE(4, 4)
        BF_CASE(6, 8)
        BF_CASE(8, 12)
#undef BF_CASE
        default: break;
    }
}

}  // namespace mdp
