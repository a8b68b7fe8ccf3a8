// compute_yi with the products of two U elements shared by the layers they couple to.
//
// Z of layer j at (mb, ma) takes the products u1(mb1, m1) u2(mb2, m2) with mb1 + mb2 - (j1 + j2)/2 = mb - j/2 and the same
// for m1 + m2: the products depend on mb - j/2, not on j.  All output rows with one k = j - 2 mb >= 0 (a class: rows
// j = k, k + 2, ..., J) therefore need the same products, each weighted with its own layer's coefficients.  A row at a time
// (k_yi_half) takes 6 FP64 operations per product and layer; here a wave has the whole class, 4 per product and 2 per layer:
// 137,000 against 206,000 operations per atom at twojmax 8, 30,200 against 41,500 at 6, and the U rows are read from LDS
// once per class instead of once per row (6,000 against 10,500 reads of 16 bytes).
//
// The sums of all rows of a class stay in registers (24 complex at twojmax 8, with two U rows some 200 VGPRs): two waves
// per SIMD.  128,000 atoms: twojmax 8 1,277 -> 941 us, 6 293 -> 268, 4 74 -> 69.  Bound by FP64 issue (about half of it at
// twojmax 8) and, at 6 and 4, by the longest class.  Each class is code of its own: with k a run-time value the tests per
// column and layer and the products kept for them spilled (1,465 registers).
//
// Index functions with loops (cg_block, triple_id, h_block) are taken as constexpr values throughout: called with template
// arguments in ordinary expressions they were executed, 4 scalar instructions to a vector one (twojmax 6 and 4 of the rows'
// kernel 424 -> 293 and 109 -> 74 us without them).
#pragma once
#include "k_yih.hpp"

namespace mdp {

// first accumulator of layer j in class k
__host__ __device__ constexpr int class_acc(int k, int j) {
    int a = 0;
    for (int l = k; l < j; l += 2) a += l + 1;
    return a;
}
// largest layer that j1 and j2 couple to
__host__ __device__ constexpr int class_top(int J, int j1, int j2) {
    return j1 + j2 <= J ? j1 + j2 : J - (J + j1 + j2) % 2;
}
__host__ __device__ constexpr int half_row_id(int j, int mb) {
    int r = 0;
    for (int l = 0; l < j; ++l) r += l / 2 + 1;
    return r + mb;
}

// The terms of one pair of U rows a (layer J1, row mb1) and b (layer J2, row mb2) for every layer JO of class K: cb[JO / 2]
// holds its mb-direction coefficient times the weight of (J1, J2, JO).  SAME: a = b, each unordered pair of columns once
// (as z_terms_same_row).  HALF: columns behind the middle (m1 + m2 > (J1 + J2)/2) are not needed.
template <int J, int K, int J1, int J2, bool SAME, bool HALF, int NACC>
__device__ __forceinline__ void class_terms(const double (&ar)[J1 + 1], const double (&ai)[J1 + 1],
                                            const double (&br)[J2 + 1], const double (&bi)[J2 + 1],
                                            const double (&cb)[J / 2 + 1], double (&zr)[NACC], double (&zi)[NACC]) {
    constexpr int JHI = class_top(J, J1, J2);
    static_for<0, J1 + J2 + 1>([&](auto Tc) {
        constexpr int T = decltype(Tc)::value;
        constexpr int MA2 = 2 * T - J1 - J2;   // 2 ma - j of the column this T goes to
        constexpr int ABS = MA2 < 0 ? -MA2 : MA2;
        if constexpr (ABS <= JHI && !(HALF && MA2 > 0)) {
            // smallest layer of the class that couples and has the column
            constexpr int JLO = cx_max(cx_max(ABS, J1 - J2), K), NJ = (JHI - JLO) / 2 + 1;
            constexpr int LO = T > J2 ? T - J2 : 0;
            constexpr int HI0 = J1 < T ? J1 : T;
            constexpr int NP = (SAME ? T / 2 : HI0) - LO + 1;
            double sr[NJ], si[NJ];
            static_for<0, NP>([&](auto Ic) {
                constexpr int I = decltype(Ic)::value, M1 = LO + I, M2 = T - M1;
                const double pr = ar[M1] * br[M2] - ai[M1] * bi[M2];
                const double pi = ar[M1] * bi[M2] + ai[M1] * br[M2];
                static_for<0, NJ>([&](auto Qc) {
                    constexpr int Q = decltype(Qc)::value;
                    constexpr double c = (SAME && M1 < M2 ? 2.0 : 1.0) * cg_const(J1, J2, JLO + 2 * Q, M1, M2);
                    sr[Q] = I == 0 ? c * pr : sr[Q] + c * pr;
                    si[Q] = I == 0 ? c * pi : si[Q] + c * pi;
                });
            });
            static_for<0, NJ>([&](auto Qc) {
                constexpr int Q = decltype(Qc)::value, JO = JLO + 2 * Q;
                constexpr int A = class_acc(K, JO) + (JO + MA2) / 2;
                zr[A] += cb[JO / 2] * sr[Q];
                zi[A] += cb[JO / 2] * si[Q];
            });
            __builtin_amdgcn_sched_barrier(0);   // a column's temporaries end here, or the accumulators spill
        }
    });
}

// All output rows of class K for this lane's atom.  PA: weights beta_t[triple * N + atom] per atom, no energy partials;
// FULL: the upstream layout of Y, every column (see full_element).
template <int J, int K, bool PA, bool FULL>
__device__ __forceinline__ void y_class(const double* __restrict__ cg, const double* __restrict__ beta_t,
                                        const double* __restrict__ lbuf, int lane, int atom, bool live, int N,
                                        double* __restrict__ Yr, double* __restrict__ Yi, double* __restrict__ epart) {
    constexpr bool HALF = !FULL && K == 0;
    constexpr int NACC = class_acc(K, J + 2 - (J + K) % 2);
    const size_t n = static_cast<size_t>(N);
    double zr[NACC], zi[NACC];
#pragma unroll
    for (int a = 0; a < NACC; ++a) { zr[a] = 0.0; zi[a] = 0.0; }
    static_for<0, J + 1>([&](auto J1c) {
        constexpr int J1 = decltype(J1c)::value;
        static_for<0, J1 + 1>([&](auto J2c) {
            constexpr int J2 = decltype(J2c)::value;
            constexpr int JHI = class_top(J, J1, J2), JLO = cx_max(J1 - J2, K);
            if constexpr ((J1 + J2 + K) % 2 == 0 && JLO <= JHI) {
                constexpr int S = (J1 + J2 - K) / 2;   // mb1 + mb2
                constexpr int NJ = (JHI - JLO) / 2 + 1;
                [[maybe_unused]] double w[NJ];
                if constexpr (PA)
                    static_for<0, NJ>([&](auto Qc) {
                        constexpr int Q = decltype(Qc)::value, T = triple_id(J, J1, J2, JLO + 2 * Q);
                        w[Q] = live ? beta_t[static_cast<size_t>(T) * n + atom] : 0.0;
                    });
                constexpr int FIRST = cx_max(0, S - J2), LAST = J1 == J2 ? S / 2 : cx_min(J1, S);
#pragma unroll 1
                for (int m = FIRST; m <= LAST; ++m) {
                    int mb1 = __builtin_amdgcn_readfirstlane(m);
                    asm volatile("" : "+s"(mb1));   // unknown to the compiler: rows and weights are read here, not kept from earlier
                    int zero = 0;
                    asm volatile("" : "+s"(zero));
                    const int mb2 = S - mb1;
                    double ar[J1 + 1], ai[J1 + 1];
                    lds_row<J1, true>(mb1, lbuf, nullptr, lane, ar, ai);
                    double cb[J / 2 + 1];
                    static_for<0, NJ>([&](auto Qc) {
                        constexpr int Q = decltype(Qc)::value, JO = JLO + 2 * Q;
                        constexpr int CGB = cg_block(J, J1, J2, JO), T = triple_id(J, J1, J2, JO);
                        cb[JO / 2] = cg[CGB + mb1 * (J2 + 1) + mb2] * (PA ? w[Q] : beta_t[T + zero]);
                        if (J1 == J2 && mb1 != mb2) cb[JO / 2] *= 2.0;   // for (mb2, mb1) too
                    });
                    if constexpr (J1 == J2) {
                        if (mb1 == mb2) {
                            class_terms<J, K, J1, J2, true, HALF>(ar, ai, ar, ai, cb, zr, zi);
                            continue;
                        }
                    }
                    double br[J2 + 1], bi[J2 + 1];
                    lds_row<J2, true>(mb2, lbuf, nullptr, lane, br, bi);
                    class_terms<J, K, J1, J2, false, HALF>(ar, ai, br, bi, cb, zr, zi);
                }
            }
        });
    });
    if (!live) return;
    const double2* __restrict__ lc = reinterpret_cast<const double2*>(lbuf);
    static_for<0, J + 1>([&](auto JOc) {
        constexpr int JO = decltype(JOc)::value;
        if constexpr (JO >= K && (JO + K) % 2 == 0) {
            constexpr int MB = (JO - K) / 2, HROW = h_block(JO) + (JO + 1) * MB, MALIM = HALF ? MB : JO;
            constexpr int OROW = FULL ? u_block(JO) + (JO + 1) * MB : HROW, ROW = half_row_id(JO, MB);
            constexpr int ACC = class_acc(K, JO);
            const size_t o = static_cast<size_t>(OROW) * n + atom;
            double e = 0.0;
#pragma unroll
            for (int ma = 0; ma <= MALIM; ++ma) {
                const double yr = zr[ACC + ma], yi = zi[ACC + ma];
                Yr[o + ma * n] = yr;
                Yi[o + ma * n] = yi;
                if constexpr (!PA && !FULL) {
                    const double wt = (K > 0 || ma < MB) ? 1.0 : 0.5;
                    const double2 u = lc[(HROW + ma) * 64 + lane];
                    e += wt * (u.x * yr + u.y * yi);
                }
            }
            if constexpr (!PA && !FULL) epart[static_cast<size_t>(ROW) * n + atom] = e;
        }
    });
}

// Classes of wave `wave`, in turn: the sums of their operations are about equal (twojmax 8: k = 0 .. 8 take 15, 21, 24,
// 18, 19, 13, 13, 7 and 7 thousand), and the two waves of a SIMD (wave and wave + 4) add up to the same.  -1: done.
template <int J, int W>
__device__ __forceinline__ int class_of(int wave, int turn) {
    if constexpr (J == 8 && W == 8) {
        constexpr int C[2][8] = {{2, 1, 4, 3, 6, 5, 0, 7}, {-1, -1, -1, -1, -1, -1, -1, 8}};
        return turn < 2 ? C[turn][wave] : -1;
    } else if constexpr (J == 6 && W == 4) {
        constexpr int C[2][4] = {{2, 1, 4, 0}, {-1, 6, 5, 3}};
        return turn < 2 ? C[turn][wave] : -1;
    } else {
        const int k = wave + W * turn;
        return k <= J ? k : -1;
    }
}

// A workgroup per 64 atoms, the half rows of their U in LDS as (re, im) pairs.
template <int J, int W, bool PA = false, bool FULL = false>
__global__ __launch_bounds__(64 * W, 2) void k_yi_class(const double* __restrict__ cg, const double* __restrict__ Ur,
                                                        const double* __restrict__ Ui, const double* __restrict__ beta_t,
                                                        double* __restrict__ Yr, double* __restrict__ Yi,
                                                        double* __restrict__ epart, int N) {
    constexpr int HE = n_half_elems(J);
    __shared__ double lbuf[2 * HE * 64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int atom = blockIdx.x * 64 + lane;
    const bool live = atom < N;
    const size_t n = static_cast<size_t>(N);
    for (int e = wave; e < HE; e += W) {
        const size_t g = static_cast<size_t>(FULL ? full_element<J>(e) : e) * n + atom;
        reinterpret_cast<double2*>(lbuf)[e * 64 + lane] = live ? make_double2(Ur[g], Ui[g]) : make_double2(0.0, 0.0);
    }
    __syncthreads();
    for (int turn = 0;; ++turn) {
        const int k = __builtin_amdgcn_readfirstlane(class_of<J, W>(wave, turn));
        if (k < 0) break;
        static_for<0, J + 1>([&](auto Kc) {
            constexpr int K = decltype(Kc)::value;
            if (k == K) {
                // values the classes have in common are made anew in each: kept for all of them they would fill the registers
                int ln = lane, zero = 0, nn = N;
                asm volatile("" : "+v"(ln));
                asm volatile("" : "+s"(zero));
                asm volatile("" : "+s"(nn));
                const int at = blockIdx.x * 64 + ln;
                y_class<J, K, PA, FULL>(cg + zero, beta_t + zero, lbuf, ln, at, at < nn, nn, Yr, Yi, epart);
            }
        });
    }
}

}  // namespace mdp
