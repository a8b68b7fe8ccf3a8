// Training-side kernels of the learned surrogate: the descriptor chain rule that turns per-atom
// energy gradients g = dE_a/dB_a into forces, the adjoint of the force loss with respect to g, and
// the per-configuration energy loss.  All sums are gathers in a fixed order (no atomics), so a
// training step is deterministic.
//
// Layouts (P pairs sorted by centre atom, n atoms, K descriptor components):
//   g, U      [K][n]          dbdr  [K][3][P]  (dB_k(centre)/dr_ij, r_ij = x_j - x_i)
//   s         [3][P]          F, R, Fref  [n][3]
// Pair p = (i = pi[p], j = pj[p]) contributes s_p = sum_k g_ki dbdr_kp to F_i and -s_p to F_j
// (F = -dE/dx with E_i a function of the r_ij of its pairs, as in cpuSnap.cpp:2293-2365).
#include <hip/hip_runtime.h>

#include "sur_launch.hpp"

namespace mdp {

__global__ void k_sur_pair_s(const double* __restrict__ g, const double* __restrict__ dbdr, const int* __restrict__ pi,
                             int K, int n, long P, double* __restrict__ s) {
    const long p = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (p >= P) return;
    const int i = pi[p];
    double sx = 0.0, sy = 0.0, sz = 0.0;
    for (int k = 0; k < K; ++k) {
        const double gk = g[static_cast<size_t>(k) * n + i];
        sx += gk * dbdr[(3 * k) * P + p];
        sy += gk * dbdr[(3 * k + 1) * P + p];
        sz += gk * dbdr[(3 * k + 2) * P + p];
    }
    s[p] = sx;
    s[P + p] = sy;
    s[2 * P + p] = sz;
}

// F and R of every atom: 16 lanes per atom, lane s taking own pairs and incoming entries s, s + 16, ... (an
// atom's own pairs are one contiguous run of each plane), combined by a butterfly in a fixed order.  Bound by
// the latency of the incoming gather, whose pairs belong to the same configuration and hit in L2.  400,000 atoms,
// 9.0 M pairs: 182 us; 756 us with one lane per atom.
constexpr int FSUB = 16;

__global__ __launch_bounds__(256) void k_sur_atom_f(const double* __restrict__ s, const int* __restrict__ own_off,
                                                    const int* __restrict__ in_off, const int* __restrict__ in_idx,
                                                    long P, int n, const double* __restrict__ fref,
                                                    double* __restrict__ F, double* __restrict__ R) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    const int a = t / FSUB, sub = t % FSUB;
    const bool live = a < n;
    double fx = 0.0, fy = 0.0, fz = 0.0;
    if (live) {
        for (int p = own_off[a] + sub; p < own_off[a + 1]; p += FSUB) {
            fx += s[p];
            fy += s[P + p];
            fz += s[2 * P + p];
        }
        for (int q = in_off[a] + sub; q < in_off[a + 1]; q += FSUB) {
            const long p = in_idx[q];
            fx -= s[p];
            fy -= s[P + p];
            fz -= s[2 * P + p];
        }
    }
#pragma unroll
    for (int w = FSUB / 2; w >= 1; w /= 2) {
        fx += __shfl_xor(fx, w);
        fy += __shfl_xor(fy, w);
        fz += __shfl_xor(fz, w);
    }
    if (!live || sub > 2) return;
    const double f = sub == 0 ? fx : (sub == 1 ? fy : fz);
    if (F) F[3 * static_cast<size_t>(a) + sub] = f;
    if (R) R[3 * static_cast<size_t>(a) + sub] = f - fref[3 * static_cast<size_t>(a) + sub];
}

// U[k][i] = coef * sum_{p = (i, j)} (R_i - R_j) . dbdr_kp   (= d(coef/2 sum |R|^2)/dg_ki)
//
// Bound: one read of dbdr (24 K bytes per pair).  A workgroup takes `atoms` consecutive atoms, whose pairs are
// one contiguous run, 256 pairs at a time, lane = pair: each of the 3 K planes is read in full lines.  The K
// products of the 256 pairs go to LDS, and thread (atom, k) adds its atom's share in pair order, so the sum's
// order does not depend on the launch.  (The row length of 257 keeps both sides free of bank conflicts.)
// 400,000 atoms, 9.0 M pairs, K = 14: 556 us, 5.4 TB/s of dbdr.  One lane per atom reading its own pairs touched a
// cache line per value and took 7,437 us.
constexpr int UCH = 256, UKMAX = 16, UATOMS = 32;

__global__ __launch_bounds__(UCH) void k_sur_u(const double* __restrict__ R, const double* __restrict__ dbdr,
                                               const int* __restrict__ own_off, const int* __restrict__ pj, int K,
                                               int n, long P, double coef, double* __restrict__ U, int atoms) {
    extern __shared__ double prod[];   // [K][UCH + 1]
    __shared__ int off[UATOMS + 1];
    const int t = threadIdx.x, a0 = blockIdx.x * atoms, na = min(atoms, n - a0);
    if (t <= na) off[t] = own_off[a0 + t];
    __syncthreads();
    const int p0 = off[0], p1 = off[na];
    // thread t owns the sums (atom, k) numbered t and t + UCH (atoms * K <= 2 UCH)
    double acc[2] = {0.0, 0.0};
    for (int c0 = p0; c0 < p1; c0 += UCH) {
        const int p = c0 + t;
        if (p < p1) {
            int i = 0;   // the centre atom: off[i] <= p < off[i + 1]
#pragma unroll
            for (int step = UATOMS / 2; step > 0; step >>= 1)
                if (i + step < na && off[i + step] <= p) i += step;
            const size_t ri = 3 * static_cast<size_t>(a0 + i), rj = 3 * static_cast<size_t>(pj[p]);
            const double dx = R[ri] - R[rj], dy = R[ri + 1] - R[rj + 1], dz = R[ri + 2] - R[rj + 2];
#pragma unroll
            for (int k = 0; k < UKMAX; ++k)
                if (k < K)
                    prod[k * (UCH + 1) + t] =
                        dx * dbdr[(3 * k) * P + p] + dy * dbdr[(3 * k + 1) * P + p] + dz * dbdr[(3 * k + 2) * P + p];
        }
        __syncthreads();
        const int c1 = min(c0 + UCH, p1);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int id = t + h * UCH;
            if (id < na * K) {
                const int i = id / K, k = id - i * K;
                const int lo = max(off[i], c0), hi = min(off[i + 1], c1);
                const double* __restrict__ row = prod + k * (UCH + 1) - c0;
                for (int q = lo; q < hi; ++q) acc[h] += row[q];
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int id = t + h * UCH;
        if (id < na * K) {
            const int i = id / K, k = id - i * K;
            U[static_cast<size_t>(k) * n + a0 + i] = coef * acc[h];
        }
    }
}

// per configuration: E_c = sum of its atom energies; alpha_a = coef * 2 (E_c - Eref_c) / N_c^2
// (the derivative of coef * ((E_c - Eref_c) / N_c)^2 with respect to each atom energy).  One wave per
// configuration: lane sums of every 64th atom, then a butterfly (1,600 configurations of 250 atoms: 5 us; 63 us
// with one lane per configuration).
__global__ __launch_bounds__(256) void k_sur_energy(const double* __restrict__ e, const int* __restrict__ cfg_off,
                                                    const double* __restrict__ eref, int C, double coef,
                                                    double* __restrict__ Ec, double* __restrict__ alpha) {
    const int c = blockIdx.x * 4 + static_cast<int>(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (c >= C) return;   // uniform over the wave
    const int a0 = cfg_off[c], a1 = cfg_off[c + 1];
    double E = 0.0;
    for (int a = a0 + lane; a < a1; a += 64) E += e[a];
#pragma unroll
    for (int w = 32; w >= 1; w /= 2) E += __shfl_xor(E, w);
    if (lane == 0) Ec[c] = E;
    if (alpha) {
        const double nc = static_cast<double>(a1 - a0);
        const double al = coef * 2.0 * (E - eref[c]) / (nc * nc);
        for (int a = a0 + lane; a < a1; a += 64) alpha[a] = al;
    }
}

// per-block partial sums of v[k]^2 (fixed order within a block)
__global__ __launch_bounds__(256) void k_sumsq(const double* __restrict__ v, long n, double* __restrict__ part) {
    __shared__ double sh[256];
    double s = 0.0;
    for (long k = static_cast<long>(blockIdx.x) * 256 + threadIdx.x; k < n; k += static_cast<long>(gridDim.x) * 256)
        s += v[k] * v[k];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (static_cast<int>(threadIdx.x) < o) sh[threadIdx.x] += sh[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

void launch_sur_pair_s(const double* g, const double* dbdr, const int* pi, int K, int n, long P, double* s,
                       hipStream_t st) {
    if (P > 0) hipLaunchKernelGGL(k_sur_pair_s, dim3((P + 255) / 256), dim3(256), 0, st, g, dbdr, pi, K, n, P, s);
}

void launch_sur_atom_f(const double* s, const int* own_off, const int* in_off, const int* in_idx, long P, int n,
                       const double* fref, double* F, double* R, hipStream_t st) {
    if (n > 0)
        hipLaunchKernelGGL(k_sur_atom_f, dim3(static_cast<unsigned>((static_cast<long>(n) * FSUB + 255) / 256)), dim3(256),
                           0, st, s, own_off, in_off, in_idx, P, n, fref, F, R);
}

void launch_sur_u(const double* R, const double* dbdr, const int* own_off, const int* pj, int K, int n, long P,
                  double coef, double* U, hipStream_t st) {
    if (n <= 0) return;
    // 32 atoms fill nearly three chunks of 256 pairs; small sets take 8 so that more workgroups are in flight
    const int atoms = n >= 16384 ? UATOMS : 8;
    hipLaunchKernelGGL(k_sur_u, dim3((n + atoms - 1) / atoms), dim3(UCH), sizeof(double) * K * (UCH + 1), st, R, dbdr,
                       own_off, pj, K, n, P, coef, U, atoms);
}

void launch_sur_energy(const double* e, const int* cfg_off, const double* eref, int C, double coef, double* Ec,
                       double* alpha, hipStream_t st) {
    if (C > 0)
        hipLaunchKernelGGL(k_sur_energy, dim3((C + 3) / 4), dim3(256), 0, st, e, cfg_off, eref, C, coef, Ec, alpha);
}

void launch_sumsq(const double* v, long n, double* part, int nblocks, hipStream_t st) {
    hipLaunchKernelGGL(k_sumsq, dim3(nblocks), dim3(256), 0, st, v, n, part);
}

}  // namespace mdp
