// compute_yi of the MD path: row order and launch dispatch over the (twojmax, waves) instantiations.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "snap_device.hpp"
#include "snap_launch.hpp"

namespace mdp {

#define YH_DECL(JV, WV)                                                                                   \
    void launch_yi_half_##JV##_##WV(const SnapDev&, const double*, const double*, const double*, double*, \
                                    double*, double*, const int*, int, hipStream_t);
YH_DECL(2, 8)
YH_DECL(4, 8)
YH_DECL(6, 8)
YH_DECL(8, 8)
YH_DECL(8, 12)
YH_DECL(8, 4)
YH_DECL(8, 12s)
YH_DECL(8, 12c)
YH_DECL(8, 12y)
YH_DECL(8, 12u1)
#undef YH_DECL
void launch_yi_rows_8(const SnapDev&, const double*, const double*, const double*, double*, double*, double*, const int*,
                      int, hipStream_t);
void launch_yi_rows_small(const SnapDev&, const double*, const double*, const double*, double*, double*, double*,
                          const int*, int, hipStream_t);

void launch_yi_class_8(const SnapDev&, const double*, const double*, const double*, double*, double*, double*, int,
                       hipStream_t);
void launch_yi_class_small(const SnapDev&, const double*, const double*, const double*, double*, double*, double*, int,
                           hipStream_t);

void yi_row_order(int J, int* out) {
    auto cgn = [](int m, int j1, int j2, int j) {
        const int lo = std::max(0, (2 * m - j - j2 + j1) / 2);
        return std::min(j1, (2 * m - j + j2 + j1) / 2) - lo + 1;
    };
    std::vector<std::pair<long, int>> cost;
    int r = 0;
    for (int j = 0; j <= J; ++j)
        for (int mb = 0; 2 * mb <= j; ++mb, ++r) {
            long t = 0;
            for (int j1 = 0; j1 <= J; ++j1)
                for (int j2 = 0; j2 <= j1; ++j2)
                    if (j >= j1 - j2 && j <= j1 + j2 && (j1 + j2 + j) % 2 == 0) {
                        const int nb = cgn(mb, j1, j2, j);
                        for (int ma = 0; ma <= j; ++ma)
                            if (2 * mb < j || ma <= mb) t += static_cast<long>(cgn(ma, j1, j2, j)) * nb;
                        t += 4L * nb * (j1 + j2 + 2);   // row loads
                    }
            cost.emplace_back(-t, r);
        }
    std::stable_sort(cost.begin(), cost.end());
    for (size_t k = 0; k < cost.size(); ++k) out[k] = cost[k].second;
}

// A workgroup per output row where a workgroup per 64 atoms would leave most CUs idle, then the classes; at twojmax 6, where
// the classes' longest wave is as long as a block of rows, these in between.  us, per row (208) / rows of a block (8; 116 at
// twojmax 8) / classes (308): twojmax 4, 1,024 atoms 5.4 / 9.9 / 8.3, 4,394 atoms 9.7 / 10.2 / 8.4, 16,000 atoms
// 23 / 12.7 / 10.5; twojmax 6, 4,394 atoms 26 / 38 / 40, 8,192 atoms 44 / 41 / 44, 16,000 atoms 87 / 53 / 53, 31,250 atoms
// - / 92 / 77; twojmax 8, 1,024 atoms 30 / 127 / 92, 4,394 atoms 108 / 144 / 98, 128,000 atoms - / 1,277 / 941.
int yi_default_variant(int J, int N) {
    if (N <= 64 * (J == 8 ? 60 : (J == 6 ? 112 : 50))) return YI_ROWS;
    return J == 6 && N <= 64 * 250 ? 8 : YI_CLASS;
}

int yi_half_variants(int J, int* ids) {
    if (J == 8) {   // waves per workgroup; 112: 12 waves, the larger layer's U rows shared across couplings;
                    // 113: the same with (re, im) adjacent in LDS; 115: 113 with the swap symmetry of the
                    // (j1, j1) couplings; 116: 115 with the row index made wave-uniform explicitly;
                    // 208: a workgroup per output row (k_yi_rows); 308: a wave per class of rows (k_yi_class)
        ids[0] = 8; ids[1] = 12; ids[2] = 4; ids[3] = 112; ids[4] = 113; ids[5] = 115; ids[6] = 116; ids[7] = YI_ROWS;
        ids[8] = YI_CLASS;
        return 9;
    }
    ids[0] = 8; ids[1] = YI_ROWS; ids[2] = YI_CLASS;
    return 3;
}

void launch_yi_half(const SnapDev& s, const double* Ur, const double* Ui, const double* beta_t, double* Yr, double* Yi,
                    double* epart, const int* order, int N, hipStream_t st, int waves) {
    if (N <= 0) return;
    if (waves == YI_ROWS) {
        if (s.J == 8)
            launch_yi_rows_8(s, Ur, Ui, beta_t, Yr, Yi, epart, order, N, st);
        else
            launch_yi_rows_small(s, Ur, Ui, beta_t, Yr, Yi, epart, order, N, st);
        return;
    }
    if (waves == YI_CLASS) {
        if (s.J == 8)
            launch_yi_class_8(s, Ur, Ui, beta_t, Yr, Yi, epart, N, st);
        else
            launch_yi_class_small(s, Ur, Ui, beta_t, Yr, Yi, epart, N, st);
        return;
    }
    switch (s.J) {
        case 2: launch_yi_half_2_8(s, Ur, Ui, beta_t, Yr, Yi, epart, order, N, st); break;
        case 4: launch_yi_half_4_8(s, Ur, Ui, beta_t, Yr, Yi, epart, order, N, st); break;
        case 6: launch_yi_half_6_8(s, Ur, Ui, beta_t, Yr, Yi, epart, order, N, st); break;
        case 8:
            if (waves == 12)
                launch_yi_half_8_12(s, Ur, Ui, beta_t, Yr, Yi, epart, order, N, st);
            else if (waves == 112)
                launch_yi_half_8_12s(s, Ur, Ui, beta_t, Yr, Yi, epart, order, N, st);
            else if (waves == 113)
                launch_yi_half_8_12c(s, Ur, Ui, beta_t, Yr, Yi, epart, order, N, st);
            else if (waves == 115)
                launch_yi_half_8_12y(s, Ur, Ui, beta_t, Yr, Yi, epart, order, N, st);
            else if (waves == 116)
                launch_yi_half_8_12u1(s, Ur, Ui, beta_t, Yr, Yi, epart, order, N, st);
            else if (waves == 4)
                launch_yi_half_8_4(s, Ur, Ui, beta_t, Yr, Yi, epart, order, N, st);
            else
                launch_yi_half_8_8(s, Ur, Ui, beta_t, Yr, Yi, epart, order, N, st);
            break;
        default: break;
    }
}

}  // namespace mdp
