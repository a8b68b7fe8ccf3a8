// compute_yi by classes of output rows, twojmax 2, 4 and 6 (see k_yic.hpp).
#include "k_yic.hpp"

namespace mdp {

void launch_yi_class_small(const SnapDev& s, const double* Ur, const double* Ui, const double* beta_t, double* Yr,
                           double* Yi, double* epart, int N, hipStream_t st) {
    const dim3 grid((N + 63) / 64);
    switch (s.J) {
#define YC_CASE(JV, WV)                                                                                                \
    case JV:                                                                                                           \
        hipLaunchKernelGGL((k_yi_class<JV, WV>), grid, dim3(64 * WV), 0, st, s.cg, Ur, Ui, beta_t, Yr, Yi, epart, N);  \
        break;
        YC_CASE(2, 3)
        YC_CASE(4, 5)
        YC_CASE(6, 4)
#undef YC_CASE
        default: break;
    }
}

// the learned surrogate at twojmax 2 and 4: Y with per-atom weights (65,536 atoms, twojmax 4: 40 us a row at a time, 29 so)
bool launch_yi_half_pa(const SnapDev& s, const double* Ur, const double* Ui, const double* beta_pa, double* Yr,
                       double* Yi, int N, hipStream_t st) {
    if (N <= 0) return true;
    const dim3 grid((N + 63) / 64);
    switch (s.J) {
        case 2: hipLaunchKernelGGL((k_yi_class<2, 3, true>), grid, dim3(64 * 3), 0, st, s.cg, Ur, Ui, beta_pa, Yr, Yi, nullptr, N); return true;
        case 4: hipLaunchKernelGGL((k_yi_class<4, 5, true>), grid, dim3(64 * 5), 0, st, s.cg, Ur, Ui, beta_pa, Yr, Yi, nullptr, N); return true;
        default: return false;
    }
}

}  // namespace mdp
