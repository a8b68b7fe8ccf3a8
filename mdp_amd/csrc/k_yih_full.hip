// compute_yi on the upstream U and Y layouts, one element (see k_yih.hpp): twojmax 2, 4 and 6, and the dispatch.
#include "k_yic.hpp"

namespace mdp {

void launch_yi_full_8(const SnapDev& s, const double* Ur, const double* Ui, const double* beta_t, double* Yr, double* Yi,
                      const int* order, int N, bool rows, hipStream_t st);

// A workgroup per output row where yi_default_variant says so (a workgroup per 64 atoms would leave most CUs idle), else the
// classes.  15,972 atoms at twojmax 8: 167 us, against 203 with the rows of 64 atoms in one workgroup and 699 for the row
// per wave from global memory that any U and any coupling table still take.
void launch_yi_full(const SnapDev& s, const double* Ur, const double* Ui, const double* beta_t, double* Yr, double* Yi,
                    const int* order, int N, hipStream_t st) {
    if (N <= 0) return;
    const bool rows = yi_default_variant(s.J, N) == YI_ROWS;
    switch (s.J) {
#define YF_CASE(JV, WV)                                                                                              \
    case JV:                                                                                                         \
        if (rows)                                                                                                    \
            launch_yi_rows<JV, 8, true>(s, Ur, Ui, beta_t, Yr, Yi, nullptr, order, N, st);                            \
        else                                                                                                         \
            hipLaunchKernelGGL((k_yi_class<JV, WV, false, true>), dim3((N + 63) / 64), dim3(64 * WV), 0, st, s.cg, Ur, \
                               Ui, beta_t, Yr, Yi, nullptr, N);                                                      \
        break;
        YF_CASE(2, 3)
        YF_CASE(4, 5)
        YF_CASE(6, 4)
#undef YF_CASE
        case 8: launch_yi_full_8(s, Ur, Ui, beta_t, Yr, Yi, order, N, rows, st); break;
        default: break;
    }
}

}  // namespace mdp
