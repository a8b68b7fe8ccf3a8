// compute_yi by classes of output rows, twojmax 8 (see k_yic.hpp).
#include "k_yic.hpp"

namespace mdp {

void launch_yi_class_8(const SnapDev& s, const double* Ur, const double* Ui, const double* beta_t, double* Yr, double* Yi,
                       double* epart, int N, hipStream_t st) {
    hipLaunchKernelGGL((k_yi_class<8, 8>), dim3((N + 63) / 64), dim3(64 * 8), 0, st, s.cg, Ur, Ui, beta_t, Yr, Yi, epart, N);
}

}  // namespace mdp
