// compute_yi of the MD path, twojmax 8, one workgroup of 12 waves per (64-atom block, output row).
#include "k_yih.hpp"

namespace mdp {

void launch_yi_rows_8(const SnapDev& s, const double* Ur, const double* Ui, const double* beta_t, double* Yr, double* Yi,
                      double* epart, const int* order, int N, hipStream_t st) {
    launch_yi_rows<8, 12>(s, Ur, Ui, beta_t, Yr, Yi, epart, order, N, st);
}

}  // namespace mdp
