// compute_yi and compute_bi on the upstream U and Y layouts, twojmax 8 (see k_yih.hpp).
#include "k_yic.hpp"

namespace mdp {

void launch_yi_full_8(const SnapDev& s, const double* Ur, const double* Ui, const double* beta_t, double* Yr, double* Yi,
                      const int* order, int N, bool rows, hipStream_t st) {
    if (rows)
        launch_yi_rows<8, 12, true>(s, Ur, Ui, beta_t, Yr, Yi, nullptr, order, N, st);
    else
        hipLaunchKernelGGL((k_yi_class<8, 8, false, true>), dim3((N + 63) / 64), dim3(64 * 8), 0, st, s.cg, Ur, Ui, beta_t,
                           Yr, Yi, nullptr, N);
}

}  // namespace mdp
