// compute_yi of the MD path, twojmax 2, 4 and 6, one workgroup of 8 waves per (64-atom block, output row).
#include "k_yih.hpp"

namespace mdp {

void launch_yi_rows_small(const SnapDev& s, const double* Ur, const double* Ui, const double* beta_t, double* Yr,
                          double* Yi, double* epart, const int* order, int N, hipStream_t st) {
    switch (s.J) {
        case 2: launch_yi_rows<2, 8>(s, Ur, Ui, beta_t, Yr, Yi, epart, order, N, st); break;
        case 4: launch_yi_rows<4, 8>(s, Ur, Ui, beta_t, Yr, Yi, epart, order, N, st); break;
        case 6: launch_yi_rows<6, 8>(s, Ur, Ui, beta_t, Yr, Yi, epart, order, N, st); break;
        default: break;
    }
}

}  // namespace mdp
