// compute_yi on the upstream U and Y layouts, one element (see k_yih.hpp): twojmax 2, 4 and 6, and the dispatch.
#include "k_yih.hpp"

namespace mdp {

void launch_yi_full_8(const SnapDev& s, const double* Ur, const double* Ui, const double* beta_t, double* Yr, double* Yi,
                      const int* order, int N, bool rows, hipStream_t st);

// A workgroup per output row where a workgroup per 64 atoms would leave most CUs idle (the lines of the MD engine).
// 15,972 atoms at twojmax 8: 203 us, against 699 for the row per wave from global memory that any U and any coupling
// table still take; bound by the FP64 pipe, like the MD engine's own.
void launch_yi_full(const SnapDev& s, const double* Ur, const double* Ui, const double* beta_t, double* Yr, double* Yi,
                    const int* order, int N, hipStream_t st) {
    if (N <= 0) return;
    const bool rows = N <= 64 * (s.J == 8 ? 80 : 128);
    switch (s.J) {
#define YF_CASE(JV)                                                                                              \
    case JV:                                                                                                     \
        if (rows)                                                                                                \
            launch_yi_rows<JV, 8, true>(s, Ur, Ui, beta_t, Yr, Yi, nullptr, order, N, st);                        \
        else                                                                                                     \
            hipLaunchKernelGGL((k_yi_half<JV, 8, false, true, true, true, 1, true>), dim3((N + 63) / 64),         \
                               dim3(64 * 8), 0, st, s.cg, Ur, Ui, beta_t, Yr, Yi, nullptr, order, N);             \
        break;
        YF_CASE(2)
        YF_CASE(4)
        YF_CASE(6)
#undef YF_CASE
        case 8: launch_yi_full_8(s, Ur, Ui, beta_t, Yr, Yi, order, N, rows, st); break;
        default: break;
    }
}

}  // namespace mdp
