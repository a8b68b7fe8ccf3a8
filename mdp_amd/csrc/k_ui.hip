// compute_ui for gfx950 (cpuSnap.cpp:312-542 semantics).
//
// Lane = atom: a wavefront covers 64 consecutive atoms and each lane walks its own pairs.  The U
// rows of one "row group" (rows RLO..RHI of the half domain) are accumulated in registers over all
// pairs, so there are no atomics and the result is independent of scheduling.  Rows below RLO are
// advanced only up to the seed of the next row.  At twojmax = 8 the 155 half-U elements are split
// into four groups ({0}, {1}, {2}, {3,4}: 45/42/35/33 elements) run by separate workgroups of one
// launch.  U is stored atom-fastest, so every store of a wave is one contiguous 512-byte segment.
#include <hip/hip_runtime.h>

#include "snap_device.hpp"
#include "snap_launch.hpp"

namespace mdp {

bool templated_j(int J) { return J == 2 || J == 4 || J == 6 || J == 8; }

// Sum over the SUB adjacent lanes that share an atom, by DPP within a row of 16 lanes; every lane gets the same sum
// (quad permutes swap neighbours 1 and 2 apart; the half-row and row mirrors then pair quads and octets).
template <int CTRL>
__device__ __forceinline__ double dpp_add(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xF, 0xF, true);
    return v + __hiloint2double(hi, lo);
}
template <int SUB>
__device__ __forceinline__ double sub_sum(double v) {
    static_assert(SUB == 1 || SUB == 4 || SUB == 16, "lanes per atom");
    if constexpr (SUB >= 4) {
        v = dpp_add<0xB1>(v);    // quad_perm [1, 0, 3, 2]
        v = dpp_add<0x4E>(v);    // quad_perm [2, 3, 0, 1]
    }
    if constexpr (SUB >= 16) {
        v = dpp_add<0x141>(v);   // row_half_mirror
        v = dpp_add<0x140>(v);   // row_mirror
    }
    return v;
}

// GEO: the pair's Cayley-Klein parameters and weighted switching factor come precomputed from
// pgeo[5q..5q+4] = (a_r, a_i, b_r, b_i, sfac * w_j) (the MD pair list writes them once per step with the
// same pair_geometry), instead of being derived here from r_ij in every row group.
// SUB > 1 (with GEO): SUB adjacent lanes share an atom and take every SUB-th of its pairs, so that a
// small system puts SUB times as many waves on the chip and each walks a SUB-th of the serial chain of pairs; the
// partial sums are added across the lanes at the end and lane k % SUB stores element k.
template <int J, int RLO, int RHI, int MODE, bool GEO = false, int SUB = 1>
__device__ __forceinline__ void ui_rows(const SnapDev& s, double* __restrict__ Ur, double* __restrict__ Ui,
                                        const double* __restrict__ rij, const int* __restrict__ pair_off,
                                        const int* __restrict__ pair_end, const int* __restrict__ perm, const int* __restrict__ ti,
                                        const int* __restrict__ tj, int N, double wself, int elem_sel, int atom,
                                        const double* __restrict__ pgeo = nullptr, int sub = 0) {
    static_assert(SUB == 1 || (GEO && MODE != UI_FULL_WSELF), "lanes share an atom only where pgeo gives the pairs");
    constexpr int NE = rows_elems(J, RLO, RHI);
    double accr[NE], acci[NE];
#pragma unroll
    for (int k = 0; k < NE; ++k) { accr[k] = 0.0; acci[k] = 0.0; }
    auto accumulate = [&](const PairGeom& g, double sf) {
        row_chain<J, 0, RLO, RHI>(g, s.rootpq, [&](auto Jc, auto MBc, auto& pr, auto& pi, auto&, auto&) {
            constexpr int JJ = decltype(Jc)::value, MB = decltype(MBc)::value;
            constexpr int base = rows_slot(J, RLO, JJ, MB, 0);
#pragma unroll
            for (int ma = 0; ma <= JJ; ++ma) {
                accr[base + ma] += sf * pr[ma];
                acci[base + ma] += sf * pi[ma];
            }
        });
    };

    // the next pair's data are loaded while the current pair's recursion runs
    const int q0 = SUB == 1 || atom < N ? pair_off[atom] : 0, q1 = SUB == 1 || atom < N ? pair_end[atom] : 0;
    if constexpr (GEO) {
        double n[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
        if (q0 + sub < q1)
#pragma unroll
            for (int k = 0; k < 5; ++k) n[k] = pgeo[5 * static_cast<size_t>(q0 + sub) + k];
        for (int q = q0 + sub; q < q1; q += SUB) {
            PairGeom g;
            g.ar = n[0];
            g.ai = n[1];
            g.br = n[2];
            g.bi = n[3];
            const double sf = n[4];
            if (q + SUB < q1)
#pragma unroll
                for (int k = 0; k < 5; ++k) n[k] = pgeo[5 * static_cast<size_t>(q + SUB) + k];
            accumulate(g, sf);
        }
    } else {
        double nx = 0.0, ny = 0.0, nz = 0.0;
        int nti = 0, ntj = 0;
        if (q0 < q1) {
            const int p = perm ? perm[q0] : q0;
            nx = rij[3 * p]; ny = rij[3 * p + 1]; nz = rij[3 * p + 2];
            nti = ti[p]; ntj = tj[p];
        }
        for (int q = q0; q < q1; ++q) {
            const double x = nx, y = ny, z = nz;
            const int tip = nti, tjp = ntj;
            if (q + 1 < q1) {
                const int p = perm ? perm[q + 1] : q + 1;
                nx = rij[3 * p]; ny = rij[3 * p + 1]; nz = rij[3 * p + 2];
                nti = ti[p]; ntj = tj[p];
            }
            if (elem_sel >= 0 && s.map[tjp] != elem_sel) continue;
            const double rc = (s.radelem[tip] + s.radelem[tjp]) * s.rcutfac;
            PairGeom g;
            pair_geometry<false>(x, y, z, rc, s.rmin0, s.rfac0, s.switchflag, s.wjelem[tjp], g);
            accumulate(g, g.sfac);
        }
    }

    if constexpr (SUB > 1) {
#pragma unroll
        for (int k = 0; k < NE; ++k) {
            accr[k] = sub_sum<SUB>(accr[k]);
            acci[k] = sub_sum<SUB>(acci[k]);
        }
        if (atom >= N) return;   // lanes past the last atom took part in no other atom's sum
    }
    const size_t n = static_cast<size_t>(N);
    static_for<RLO, RHI + 1>([&](auto MBc) {
        constexpr int MB = decltype(MBc)::value;
        static_for<2 * MB, J + 1>([&](auto Jc) {
            constexpr int JJ = decltype(Jc)::value;
            constexpr int base = rows_slot(J, RLO, JJ, MB, 0);
            constexpr int row = u_block(JJ) + (JJ + 1) * MB;
#pragma unroll
            for (int ma = 0; ma <= JJ; ++ma) {
                const size_t o = static_cast<size_t>(row + ma) * n + atom;
                if constexpr (MODE == UI_ACCUMULATE) {
                    if (SUB > 1 && sub != (base + ma) % SUB) continue;
                    Ur[o] += accr[base + ma];
                    Ui[o] += acci[base + ma];
                } else if constexpr (MODE == UI_HALF_WSELF) {
                    if (SUB > 1 && sub != (base + ma) % SUB) continue;
                    const size_t oh = static_cast<size_t>(h_block(JJ) + (JJ + 1) * MB + ma) * n + atom;
                    Ur[oh] = accr[base + ma] + (ma == MB ? wself : 0.0);
                    Ui[oh] = acci[base + ma];
                } else {
                    const double vr = accr[base + ma] + (ma == MB ? wself : 0.0);
                    const double vi = acci[base + ma];
                    Ur[o] = vr;
                    Ui[o] = vi;
                    if (2 * MB < JJ) {   // mirror into row j-mb: U(j-mb, j-ma) = (-1)^(ma+mb) conj U(mb, ma)
                        const size_t om =
                            static_cast<size_t>(u_block(JJ) + (JJ + 1) * (JJ - MB) + (JJ - ma)) * n + atom;
                        const bool even = ((ma + MB) % 2) == 0;
                        Ur[om] = even ? vr : -vr;
                        Ui[om] = even ? -vi : vi;
                    }
                }
            }
        });
    });
}

// The row groups of twojmax = 8 ({0}, {1}, {2}, {3,4}) and 6 ({0}, {1}, {2,3}) as one launch: workgroup
// b runs group (b / 8) % NG on atom block (b / 8 / NG) * 8 + b % 8, so the groups of one atom block go to
// the same XCD (workgroups are dealt to the 8 XCDs round-robin) and share its L2 for r_ij.
template <int J>
constexpr int ui_ngroups() { return J == 8 ? 4 : (J == 6 ? 3 : 1); }

template <int J, int MODE, bool GEO = false, int SUB = 1>
__global__ __launch_bounds__(64) void k_ui(SnapDev s, double* __restrict__ Ur, double* __restrict__ Ui,
                                           const double* __restrict__ rij, const int* __restrict__ pair_off,
                                           const int* __restrict__ pair_end, const int* __restrict__ perm, const int* __restrict__ ti,
                                           const int* __restrict__ tj, int N, double wself, int elem_sel,
                                           const double* __restrict__ pgeo) {
    constexpr int NG = ui_ngroups<J>();
    const int b = blockIdx.x, k = b / 8;
    const int group = k % NG, ablock = (k / NG) * 8 + b % 8;
    const int atom = ablock * (64 / SUB) + static_cast<int>(threadIdx.x) / SUB, sub = threadIdx.x % SUB;
    if (SUB == 1 && atom >= N) return;
    if constexpr (J == 8) {
        if (group == 0) ui_rows<8, 0, 0, MODE, GEO, SUB>(s, Ur, Ui, rij, pair_off, pair_end, perm, ti, tj, N, wself, elem_sel, atom, pgeo, sub);
        else if (group == 1) ui_rows<8, 1, 1, MODE, GEO, SUB>(s, Ur, Ui, rij, pair_off, pair_end, perm, ti, tj, N, wself, elem_sel, atom, pgeo, sub);
        else if (group == 2) ui_rows<8, 2, 2, MODE, GEO, SUB>(s, Ur, Ui, rij, pair_off, pair_end, perm, ti, tj, N, wself, elem_sel, atom, pgeo, sub);
        else ui_rows<8, 3, 4, MODE, GEO, SUB>(s, Ur, Ui, rij, pair_off, pair_end, perm, ti, tj, N, wself, elem_sel, atom, pgeo, sub);
    } else if constexpr (J == 6) {
        if (group == 0) ui_rows<6, 0, 0, MODE, GEO, SUB>(s, Ur, Ui, rij, pair_off, pair_end, perm, ti, tj, N, wself, elem_sel, atom, pgeo, sub);
        else if (group == 1) ui_rows<6, 1, 1, MODE, GEO, SUB>(s, Ur, Ui, rij, pair_off, pair_end, perm, ti, tj, N, wself, elem_sel, atom, pgeo, sub);
        else ui_rows<6, 2, 3, MODE, GEO, SUB>(s, Ur, Ui, rij, pair_off, pair_end, perm, ti, tj, N, wself, elem_sel, atom, pgeo, sub);
    } else {
        ui_rows<J, 0, J / 2, MODE, GEO, SUB>(s, Ur, Ui, rij, pair_off, pair_end, perm, ti, tj, N, wself, elem_sel, atom, pgeo, sub);
    }
}

template <int J, int MODE, bool GEO = false, int SUB = 1>
static void ui_groups(const SnapDev& s, double* Ur, double* Ui, const double* rij, const int* off, const int* end,
                      const int* perm, const int* ti, const int* tj, int N, double wself, int esel, hipStream_t st,
                      const double* pgeo = nullptr) {
    constexpr int NG = ui_ngroups<J>();
    constexpr int A = 64 / SUB;   // atoms per workgroup
    const int ablocks = ((N + A - 1) / A + 7) / 8 * 8;   // padded to whole XCD rounds; excess blocks return
    hipLaunchKernelGGL((k_ui<J, MODE, GEO, SUB>), dim3(ablocks * NG), dim3(64), 0, st, s, Ur, Ui, rij, off, end, perm, ti,
                       tj, N, wself, esel, pgeo);
}

void launch_ui(const SnapDev& s, UiMode mode, double* Ur, double* Ui, const double* rij, const int* pair_off,
               const int* perm, const int* ti, const int* tj, int N, double wself, int esel, hipStream_t st) {
    if (N <= 0) return;
#define UI_CASE(JV)                                                                                   \
    case JV:                                                                                          \
        if (mode == UI_ACCUMULATE)                                                                    \
            ui_groups<JV, UI_ACCUMULATE>(s, Ur, Ui, rij, pair_off, pair_off + 1, perm, ti, tj, N, wself, esel, st); \
        else if (mode == UI_HALF_WSELF)                                                               \
            ui_groups<JV, UI_HALF_WSELF>(s, Ur, Ui, rij, pair_off, pair_off + 1, perm, ti, tj, N, wself, esel, st); \
        else                                                                                          \
            ui_groups<JV, UI_FULL_WSELF>(s, Ur, Ui, rij, pair_off, pair_off + 1, perm, ti, tj, N, wself, esel, st); \
        break;
    switch (s.J) {
        UI_CASE(2)
        UI_CASE(4)
        UI_CASE(6)
        UI_CASE(8)
        default: break;
    }
#undef UI_CASE
}

// The per-pair geometry that launch_ui_geo reads, pgeo[5q..5q+4] = (a_r, a_i, b_r, b_i, sfac w_j), for the
// pairs of a list whose length is on the device (np_dev): one lane per pair.
__global__ __launch_bounds__(256) void k_pair_geo(SnapDev s, const double* __restrict__ rij,
                                                  const int* __restrict__ ti, const int* __restrict__ tj,
                                                  const int* __restrict__ np_dev, int cap,
                                                  double* __restrict__ pgeo) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (np_dev ? *np_dev : cap)) return;
    const int tjq = tj[q];
    PairGeom g;
    pair_geometry<false>(rij[3 * static_cast<size_t>(q)], rij[3 * static_cast<size_t>(q) + 1],
                         rij[3 * static_cast<size_t>(q) + 2], (s.radelem[ti[q]] + s.radelem[tjq]) * s.rcutfac, s.rmin0,
                         s.rfac0, s.switchflag, s.wjelem[tjq], g);
    double* __restrict__ o = pgeo + 5 * static_cast<size_t>(q);
    o[0] = g.ar;
    o[1] = g.ai;
    o[2] = g.br;
    o[3] = g.bi;
    o[4] = g.sfac;
}

void launch_pair_geo(const SnapDev& s, const double* rij, const int* ti, const int* tj, const int* np_dev, int cap,
                     double* pgeo, hipStream_t st) {
    if (cap <= 0) return;
    hipLaunchKernelGGL(k_pair_geo, dim3((cap + 255) / 256), dim3(256), 0, st, s, rij, ti, tj, np_dev, cap, pgeo);
}

// compute_ui with the per-atom sums in LDS (half layout plus wself, from the pair geometry pgeo).  Lanes are pairs.
// The pairs of `ab` (at most 64) consecutive atoms are contiguous; window b of such a block holds its atoms whose first pair lies in
// [b*UI_PB, (b+1)*UI_PB) of the block, so with at most 96 pairs per atom (UI_NL - UI_PB) a window has at most UI_NL
// pairs, one per lane.  Each lane runs the row-chain recursion of its pair; every finished half row, scaled by
// sfac w_j, goes to LDS; then thread (ma, atom) adds the row entry of the atom's pairs in pair order and writes U, with
// wself added to the diagonal last (upstream adds it first, cpuSnap.cpp:312-542; the sums agree to rounding, as those
// of the per-atom kernel do).  The workgroups are persistent over the blocks; all lanes share the control flow of the
// recursion.
constexpr int UI_PB = 416, UI_NL = 512;

template <int J>
__global__ __launch_bounds__(UI_NL) void k_ui_lds(const double* __restrict__ rootpq, double* __restrict__ Ur,
                                                 double* __restrict__ Ui, const double* __restrict__ pgeo,
                                                 const int* __restrict__ poff, const int* __restrict__ pend, int N,
                                                 double wself, int ab) {
    constexpr int RW = J + 1;
    __shared__ double sr[UI_NL * RW], si[UI_NL * RW];
    __shared__ int s_off[64 + 1];   // pair offsets (relative to the window) of the window's atoms
    const int lane = threadIdx.x;
    const size_t n = static_cast<size_t>(N);
    const int blocks = (N + ab - 1) / ab;
    for (int blk = blockIdx.x; blk < blocks; blk += gridDim.x) {
      const int f0 = ab * blk, f1 = min(f0 + ab, N), base = poff[f0], ptot = pend[f1 - 1] - base;
      for (int b = 0; b * UI_PB <= ptot; ++b) {
        // atoms a0..a1-1: a0 (a1) is the first atom whose pairs start at or behind b*UI_PB ((b+1)*UI_PB)
        auto lower = [&](int v) {
            int lo = f0, hi = f1;
            while (lo < hi) {
                const int mid = lo + (hi - lo) / 2;
                if (poff[mid] - base < v) lo = mid + 1;
                else hi = mid;
            }
            return lo;
        };
        const int a0 = lower(b * UI_PB), a1 = lower((b + 1) * UI_PB);
        const int na = a1 - a0;
        if (na <= 0) continue;   // uniform
        const int q0 = poff[a0], np = pend[a1 - 1] - q0;   // at most UI_NL
        __syncthreads();   // the previous window's readers are done with s_off and the row stage
        for (int k = lane; k <= na; k += UI_NL) s_off[k] = (k < na ? poff[a0 + k] : pend[a1 - 1]) - q0;
        PairGeom g;   // lanes past the block's pairs run the recursion on a zero pair; nothing reads them
        g.ar = g.ai = g.br = g.bi = 0.0;
        double sf = 0.0;
        if (lane < np) {
            const size_t q = static_cast<size_t>(q0 + lane);
            g.ar = pgeo[5 * q];
            g.ai = pgeo[5 * q + 1];
            g.br = pgeo[5 * q + 2];
            g.bi = pgeo[5 * q + 3];
            sf = pgeo[5 * q + 4];
        }
        row_chain<J, 0, 0, J / 2>(g, rootpq, [&](auto Jc, auto MBc, auto& pr, auto& pim, auto&, auto&) {
            constexpr int L = decltype(Jc)::value, MB = decltype(MBc)::value;
            __syncthreads();   // the previous row's sums have read the stage
#pragma unroll
            for (int ma = 0; ma <= L; ++ma) {
                sr[lane * RW + ma] = sf * pr[ma];
                si[lane * RW + ma] = sf * pim[ma];
            }
            __syncthreads();
            constexpr int row = h_block(L) + (L + 1) * MB;
            for (int t = lane; t < na * (L + 1); t += UI_NL) {
                const int ma = t / na, al = t - ma * na;   // consecutive threads: consecutive atoms
                const int p1 = min(s_off[al + 1], UI_NL);   // the bound holds with at most 96 pairs per atom
                double ar = 0.0, ai = 0.0;
                for (int p = s_off[al]; p < p1; ++p) {
                    ar += sr[p * RW + ma];
                    ai += si[p * RW + ma];
                }
                const size_t o = static_cast<size_t>(row + ma) * n + a0 + al;
                Ur[o] = ar + (ma == MB ? wself : 0.0);
                Ui[o] = ai;
            }
        });
      }
    }
}

void launch_ui_geo_lds(const SnapDev& s, double* Ur, double* Ui, const double* pgeo, const int* pair_off,
                       const int* pair_end, int N, double wself, int groups, int ab, hipStream_t st) {
    if (N <= 0) return;
    const int G = groups > 0 ? groups : 512;
    switch (s.J) {
        case 2: hipLaunchKernelGGL((k_ui_lds<2>), dim3(G), dim3(UI_NL), 0, st, s.rootpq, Ur, Ui, pgeo, pair_off, pair_end, N, wself, ab); break;
        case 4: hipLaunchKernelGGL((k_ui_lds<4>), dim3(G), dim3(UI_NL), 0, st, s.rootpq, Ur, Ui, pgeo, pair_off, pair_end, N, wself, ab); break;
        case 6: hipLaunchKernelGGL((k_ui_lds<6>), dim3(G), dim3(UI_NL), 0, st, s.rootpq, Ur, Ui, pgeo, pair_off, pair_end, N, wself, ab); break;
        case 8: hipLaunchKernelGGL((k_ui_lds<8>), dim3(G), dim3(UI_NL), 0, st, s.rootpq, Ur, Ui, pgeo, pair_off, pair_end, N, wself, ab); break;
        default: break;
    }
}

// Measured on displaced BCC crystals, us with 1 / 4 / 16 lanes per atom: twojmax 4, 128 atoms 16 / 9 / 9, 16,000 atoms
// 20 / 15 / 48, 65,536 atoms 27 / 45 / 163; twojmax 6, 128 atoms 17 / 9 / 7, 8,192 atoms 20 / 16 / 34, 31,250 atoms
// 39 / 40 / 102; twojmax 8, 432 atoms 33 / 15 / 14, 8,192 atoms 36 / 32 / 103, 16,000 atoms 39 / 59 / 197.  The lines
// lie where one lane per atom would leave most (24 waves) or half (512 waves) of the 1,024 SIMDs idle.
int ui_lanes_per_atom(int J, int N) {
    const long groups = J == 8 ? 4 : (J == 6 ? 3 : 1);
    const long waves = (N + 63L) / 64 * groups;
    return waves <= 24 ? 16 : (waves <= 512 ? 4 : 1);
}

void launch_ui_geo(const SnapDev& s, double* Ur, double* Ui, const double* pgeo, const int* pair_off,
                   const int* pair_end, int N, double wself, hipStream_t st, int lanes) {
    if (N <= 0) return;
    if (lanes == 0) lanes = ui_lanes_per_atom(s.J, N);
#define UG(JV, SUBV)                                                                                                 \
    ui_groups<JV, UI_HALF_WSELF, true, SUBV>(s, Ur, Ui, nullptr, pair_off, pair_end, nullptr, nullptr, nullptr, N, wself, -1, st, \
                                             pgeo)
#define UG_CASE(JV)                                                        \
    case JV:                                                               \
        if (lanes == 16)                                                   \
            UG(JV, 16);                                                    \
        else if (lanes == 4)                                               \
            UG(JV, 4);                                                     \
        else                                                               \
            UG(JV, 1);                                                     \
        break;
    switch (s.J) {
        UG_CASE(2)
        UG_CASE(4)
        UG_CASE(6)
        UG_CASE(8)
        default: break;
    }
#undef UG_CASE
#undef UG
}

void launch_ui_acc_geo(const SnapDev& s, double* Ur, double* Ui, const double* pgeo, const int* pair_off, int N,
                       hipStream_t st) {
    if (N <= 0) return;
    const int lanes = ui_lanes_per_atom(s.J, N);
#define UA(JV, SUBV)                                                                                                  \
    ui_groups<JV, UI_ACCUMULATE, true, SUBV>(s, Ur, Ui, nullptr, pair_off, pair_off + 1, nullptr, nullptr, nullptr, N, \
                                             0.0, -1, st, pgeo)
#define UA_CASE(JV)         \
    case JV:                \
        if (lanes == 16)    \
            UA(JV, 16);     \
        else if (lanes == 4) \
            UA(JV, 4);      \
        else                \
            UA(JV, 1);      \
        break;
    switch (s.J) {
        UA_CASE(2)
        UA_CASE(4)
        UA_CASE(6)
        UA_CASE(8)
        default: break;
    }
#undef UA_CASE
#undef UA
}

}  // namespace mdp
