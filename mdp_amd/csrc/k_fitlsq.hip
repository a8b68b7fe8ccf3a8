// Linear-fit tallies and normal equations over the batched descriptors.
//
// From the per-configuration B and dB/dr of the batch, the kernels below form what the upstream
// fitting driver consumes: per configuration the type-resolved descriptor sum bi
// (cpuSnapTallyBispectrum, cpuSnap.cpp:2265-2291), the per-atom derivative tally bd
// (cpuSnapTallyBispectrumDeriv, :2293-2365) and the virial tally bv (cpuSnapTallyBispectrumVirial,
// :2367-2470), and then the weighted normal equations L = sum_r w_r^2 a_r a_r^T, h = sum_r w_r^2 a_r b_r
// of the energy, force and stress rows (linearfit.jl:168-200, rows as in emldescriptors.jl:80-140).
// Every sum runs in a fixed order, so the results do not depend on scheduling.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "fit_launch.hpp"
#include "runtime.hpp"
#include "snap_launch.hpp"

namespace mdp {

namespace {
inline int nblocks(long n, int b) { return static_cast<int>((n + b - 1) / b); }
}  // namespace

// ---- incoming pairs of every atom (pairs whose neighbour is that atom), ascending pair index ----

__global__ void k_lsq_zero(int* __restrict__ a, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = 0;
}

__global__ void k_lsq_in_count(const int* __restrict__ pj, long P, int* __restrict__ in_cnt) {
    const long p = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (p < P) atomicAdd(in_cnt + pj[p], 1);
}

__global__ void k_lsq_in_fill(const int* __restrict__ pj, long P, const int* __restrict__ in_off,
                              int* __restrict__ cursor, int* __restrict__ in_idx) {
    const long p = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (p >= P) return;
    const int a = pj[p];
    in_idx[in_off[a] + atomicAdd(cursor + a, 1)] = static_cast<int>(p);
}

// The fill order depends on scheduling: each atom's list is put in ascending order, 16 lanes per atom ranking its
// entries from an LDS copy (105,000 atoms of 20 pairs: 13 us; 99 us with one lane per atom sorting by insertion).  A list
// longer than the copy is sorted in place by one lane.
constexpr int SORT_SUB = 16, SORT_MAX = 128;

__global__ __launch_bounds__(256) void k_lsq_in_sort(const int* __restrict__ in_off, int* __restrict__ in_idx, int N) {
    __shared__ int list[256 / SORT_SUB][SORT_MAX];
    const int t = blockIdx.x * 256 + threadIdx.x, a = t / SORT_SUB, sub = t % SORT_SUB;
    const int lo = a < N ? in_off[a] : 0, n = a < N ? in_off[a + 1] - lo : 0;
    int* l = list[threadIdx.x / SORT_SUB];
    int* __restrict__ x = in_idx + lo;
    if (n <= SORT_MAX)
        for (int k = sub; k < n; k += SORT_SUB) l[k] = x[k];
    __syncthreads();
    if (n <= SORT_MAX) {
        for (int k = sub; k < n; k += SORT_SUB) {
            const int v = l[k];
            int rank = 0;
            for (int m = 0; m < n; ++m) rank += l[m] < v;
            x[rank] = v;
        }
    } else if (sub == 0) {
        for (int i = 1; i < n; ++i) {
            const int v = x[i];
            int k = i - 1;
            while (k >= 0 && x[k] > v) {
                x[k + 1] = x[k];
                --k;
            }
            x[k + 1] = v;
        }
    }
}

void launch_lsq_incoming(const int* pj, long P, int N, int* in_cnt, int* in_off, int* cursor, int* in_idx,
                         int* scan_tmp, hipStream_t st) {
    if (N <= 0) return;
    hipLaunchKernelGGL(k_lsq_zero, dim3(nblocks(N, 256)), dim3(256), 0, st, in_cnt, N);
    hipLaunchKernelGGL(k_lsq_zero, dim3(nblocks(N, 256)), dim3(256), 0, st, cursor, N);
    if (P > 0) hipLaunchKernelGGL(k_lsq_in_count, dim3(nblocks(P, 256)), dim3(256), 0, st, pj, P, in_cnt);
    exclusive_scan(in_cnt, in_off, N, scan_tmp, st);
    if (P > 0) hipLaunchKernelGGL(k_lsq_in_fill, dim3(nblocks(P, 256)), dim3(256), 0, st, pj, P, in_off, cursor, in_idx);
    hipLaunchKernelGGL(k_lsq_in_sort, dim3(nblocks(static_cast<long>(N) * SORT_SUB, 256)), dim3(256), 0, st, in_off,
                       in_idx, N);
}

// ---- tallies ------------------------------------------------------------------------------------

// bd of configuration c at bd + 3*a0_c*Kt, element (comp + 3*ii, col) at [comp + 3 ii + 3 N_c col],
// col = (t-1)*IB + k with t the type of the pair's owner: + dB/dr of the atom's own pairs, - dB/dr of the
// pairs whose neighbour it is.  Thread = (atom, k), atoms fastest.
__global__ void k_lsq_bd(const double* __restrict__ dblist, const int* __restrict__ poff,
                         const int* __restrict__ in_off, const int* __restrict__ in_idx, const int* __restrict__ pti,
                         const int* __restrict__ type, const int* __restrict__ cfg_of, const int* __restrict__ cfg_a0,
                         const int* __restrict__ cfg_p0, int N, int IB, int ntypes, double* __restrict__ bd) {
    const long t = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= static_cast<long>(N) * IB) return;
    const int g = static_cast<int>(t % N), k = static_cast<int>(t / N);
    const int c = cfg_of[g], a0 = cfg_a0[c], nc = cfg_a0[c + 1] - a0, p0 = cfg_p0[c];
    const long pc = cfg_p0[c + 1] - p0;
    const double* __restrict__ db = dblist + static_cast<size_t>(p0) * 3 * IB;
    const int kt = ntypes * IB, tg = type[g];
    double* __restrict__ out = bd + 3 * static_cast<size_t>(a0) * kt + 3 * (g - a0);
    const int q0 = poff[g], q1 = poff[g + 1], i0 = in_off[g], i1 = in_off[g + 1];
    for (int ty = 1; ty <= ntypes; ++ty) {
        double s0 = 0.0, s1 = 0.0, s2 = 0.0;
        if (tg == ty)
            for (int q = q0; q < q1; ++q) {
                const size_t e = static_cast<size_t>(q - p0) + 3 * pc * k;
                s0 += db[e];
                s1 += db[e + pc];
                s2 += db[e + 2 * pc];
            }
        for (int m = i0; m < i1; ++m) {
            const int q = in_idx[m];
            if (pti[q] != ty) continue;
            const size_t e = static_cast<size_t>(q - p0) + 3 * pc * k;
            s0 -= db[e];
            s1 -= db[e + pc];
            s2 -= db[e + 2 * pc];
        }
        const size_t col = static_cast<size_t>(ty - 1) * IB + k;
        out[3 * nc * col] = s0;
        out[3 * nc * col + 1] = s1;
        out[3 * nc * col + 2] = s2;
    }
}

// The tallies of dB/dr for one element type: bd (as above) and the virial v = -r (x) dB/dr in one pass over dB/dr.
// Bound: that one read (24 IB bytes per pair).  One workgroup per (configuration, k): it streams the three planes
// of k through LDS in tiles of BD_TILE pairs, adds each pair's virial on the way, and then every atom adds its own
// pairs of the tile and subtracts its incoming ones (both ascending), in registers of the thread that owns it: up to
// H atoms per thread.  The indices of an atom's next two incoming pairs are kept loaded: a tile without one costs no
// memory access, and one load's latency passes behind the other's pair.  Configurations come largest first (cfg_ord), those
// of more than BD_TH and of more than 4 BD_TH atoms in launches of their own, so that small ones don't carry the registers of
// large ones.  105,000 atoms, 2.1 M pairs, twojmax 8:
// 1,312 us (2.1 TB/s); a pass per plane for bd and a second read of dB/dr for the virial took 1,841 + 813 us.
// bv[c*6*Kt + 6*k + m], components m = (xx, yy, zz, xy, xz, yz); as[(6c + m')*Kt + k] are the same as the stress rows of
// the fit, in the upstream row order m' -> m = (0, 1, 2, 5, 4, 3) (snapcpp.jl:660-662).
constexpr int BD_TILE = 1280, BD_TH = 512, BD_MAXH = 6;

template <int H>
__global__ __launch_bounds__(BD_TH) void k_lsq_bd_bv(const double* __restrict__ dblist, const double* __restrict__ rij,
                                                     const int* __restrict__ poff, const int* __restrict__ in_off,
                                                     const int* __restrict__ in_idx, const int* __restrict__ cfg_a0,
                                                     const int* __restrict__ cfg_p0, const int* __restrict__ cfg_ord,
                                                     int IB, double* __restrict__ bd, double* __restrict__ bv,
                                                     double* __restrict__ as) {
    __shared__ double tile[3][BD_TILE];
    __shared__ double red[BD_TH / 64][6];
    const int c = cfg_ord[blockIdx.x / IB], k = blockIdx.x % IB, t = threadIdx.x;
    const int a0 = cfg_a0[c], nc = cfg_a0[c + 1] - a0, p0 = cfg_p0[c], pc = cfg_p0[c + 1] - p0;
    const double* __restrict__ db = dblist + static_cast<size_t>(p0) * 3 * IB + 3 * static_cast<size_t>(pc) * k;
    const double* __restrict__ r = rij + 3 * static_cast<size_t>(p0);
    double s[H][3], v[6] = {0, 0, 0, 0, 0, 0};
    int q0[H], q1[H], m[H], mend[H], next[H], after[H];   // own pairs; incoming list position and end, next two pairs
#pragma unroll
    for (int h = 0; h < H; ++h) {
        const int a = t + h * BD_TH;
        const bool live = a < nc;
        s[h][0] = s[h][1] = s[h][2] = 0.0;
        q0[h] = live ? poff[a0 + a] - p0 : 0;
        q1[h] = live ? poff[a0 + a + 1] - p0 : 0;
        m[h] = live ? in_off[a0 + a] : 0;
        mend[h] = live ? in_off[a0 + a + 1] : 0;
        next[h] = m[h] < mend[h] ? in_idx[m[h]] - p0 : pc;
        after[h] = m[h] + 1 < mend[h] ? in_idx[m[h] + 1] - p0 : pc;
    }
    for (int t0 = 0; t0 < pc; t0 += BD_TILE) {
        const int t1 = min(pc, t0 + BD_TILE);
        __syncthreads();   // the previous tile's readers are done
        for (int q = t0 + t; q < t1; q += BD_TH) {
            const double bx = db[q], by = db[q + static_cast<size_t>(pc)], bz = db[q + 2 * static_cast<size_t>(pc)];
            const double dx = -r[3 * q], dy = -r[3 * q + 1], dz = -r[3 * q + 2];
            tile[0][q - t0] = bx;
            tile[1][q - t0] = by;
            tile[2][q - t0] = bz;
            v[0] += dx * bx;
            v[1] += dy * by;
            v[2] += dz * bz;
            v[3] += dx * by;
            v[4] += dx * bz;
            v[5] += dy * bz;
        }
        __syncthreads();
#pragma unroll
        for (int h = 0; h < H; ++h) {
            const int lo = max(q0[h], t0) - t0, hi = min(q1[h], t1) - t0;
#pragma unroll 4
            for (int q = lo; q < hi; ++q) {
                s[h][0] += tile[0][q];
                s[h][1] += tile[1][q];
                s[h][2] += tile[2][q];
            }
            while (next[h] < t1) {
                const int q = next[h] - t0;
                ++m[h];
                next[h] = after[h];
                after[h] = m[h] + 1 < mend[h] ? in_idx[m[h] + 1] - p0 : pc;
                s[h][0] -= tile[0][q];
                s[h][1] -= tile[1][q];
                s[h][2] -= tile[2][q];
            }
        }
    }
    double* __restrict__ out = bd + 3 * static_cast<size_t>(a0) * IB + 3 * static_cast<size_t>(nc) * k;
#pragma unroll
    for (int h = 0; h < H; ++h) {
        const int a = t + h * BD_TH;
        if (a < nc) {
            out[3 * a] = s[h][0];
            out[3 * a + 1] = s[h][1];
            out[3 * a + 2] = s[h][2];
        }
    }
#pragma unroll
    for (int w = 32; w >= 1; w /= 2)
#pragma unroll
        for (int i = 0; i < 6; ++i) v[i] += __shfl_xor(v[i], w);
    if ((t & 63) == 0)
#pragma unroll
        for (int i = 0; i < 6; ++i) red[t >> 6][i] = v[i];
    __syncthreads();
    if (t < 6) {
        constexpr int ord[6] = {0, 1, 2, 5, 4, 3};
        double raw = 0.0, row = 0.0;
        for (int w = 0; w < BD_TH / 64; ++w) {
            raw += red[w][t];
            row += red[w][ord[t]];
        }
        bv[static_cast<size_t>(c) * 6 * IB + 6 * k + t] = raw;
        as[(static_cast<size_t>(c) * 6 + t) * IB + k] = row;
    }
}

// bi[c*Kt + col] = sum of B_k over the atoms of type t of configuration c: one block per (c, col), its
// threads over the atoms (coalesced), fixed-order tree reduction
__global__ __launch_bounds__(256) void k_lsq_bi(const double* __restrict__ blist, const int* __restrict__ type,
                                                const int* __restrict__ cfg_a0, int IB, int ntypes,
                                                double* __restrict__ bi) {
    const int kt = ntypes * IB;
    const int c = blockIdx.x / kt, col = blockIdx.x % kt;
    const int ty = col / IB + 1, k = col % IB;
    const int a0 = cfg_a0[c], nc = cfg_a0[c + 1] - a0;
    const double* __restrict__ b = blist + static_cast<size_t>(a0) * IB + static_cast<size_t>(nc) * k;
    double s = 0.0;
    for (int ii = threadIdx.x; ii < nc; ii += 256)
        if (type[a0 + ii] == ty) s += b[ii];
    __shared__ double red[256];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (static_cast<int>(threadIdx.x) < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) bi[blockIdx.x] = red[0];
}

// virial tally of configuration c and column col (one block; several element types, or configurations too large for
// k_lsq_bd_bv): v = -r (x) dB/dr summed over the pairs
// whose owner has the column's type, components (xx, yy, zz, xy, xz, yz) as upstream; written raw,
// bv[c*6*Kt + 6*col + m], and as the stress rows of the fit, as[(6c + m')*Kt + col] with the upstream
// row order m' -> m = (0, 1, 2, 5, 4, 3) (snapcpp.jl:660-662).  Fixed-order tree reduction.
__global__ __launch_bounds__(256) void k_lsq_bv(const double* __restrict__ dblist, const double* __restrict__ rij,
                                                const int* __restrict__ pti, const int* __restrict__ cfg_p0, int IB,
                                                int ntypes, double* __restrict__ bv, double* __restrict__ as) {
    const int kt = ntypes * IB;
    const int c = blockIdx.x / kt, col = blockIdx.x % kt;
    const int ty = col / IB + 1, k = col % IB;
    const int p0 = cfg_p0[c];
    const long pc = cfg_p0[c + 1] - p0;
    const double* __restrict__ db = dblist + static_cast<size_t>(p0) * 3 * IB + 3 * pc * k;
    double v[6] = {0, 0, 0, 0, 0, 0};
    for (long lp = threadIdx.x; lp < pc; lp += 256) {
        const long q = p0 + lp;
        if (pti[q] != ty) continue;
        const double dx = -rij[3 * q], dy = -rij[3 * q + 1], dz = -rij[3 * q + 2];
        const double bx = db[lp], by = db[lp + pc], bz = db[lp + 2 * pc];
        v[0] += dx * bx;
        v[1] += dy * by;
        v[2] += dz * bz;
        v[3] += dx * by;
        v[4] += dx * bz;
        v[5] += dy * bz;
    }
    __shared__ double red[6][256];
#pragma unroll
    for (int m = 0; m < 6; ++m) red[m][threadIdx.x] = v[m];
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (static_cast<int>(threadIdx.x) < w)
#pragma unroll
            for (int m = 0; m < 6; ++m) red[m][threadIdx.x] += red[m][threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x < 6) {
        const int m = threadIdx.x;
        bv[static_cast<size_t>(c) * 6 * kt + 6 * col + m] = red[m][0];
        constexpr int ord[6] = {0, 1, 2, 5, 4, 3};
        as[(static_cast<size_t>(c) * 6 + m) * kt + col] = red[ord[m]][0];
    }
}

void launch_lsq_tallies(const double* blist, const double* dblist, const double* rij, const int* poff,
                        const int* in_off, const int* in_idx, const int* pti, const int* type, const int* cfg_of,
                        const int* cfg_a0, const int* cfg_p0, const int* cfg_ord, const int* sizes, int C, int N,
                        int IB, int ntypes, double* bi, double* bd, double* bv, double* as, hipStream_t st) {
    const int kt = ntypes * IB;
    // One element type and at most BD_MAXH atoms per thread (3,072 atoms) in any configuration: one read of dB/dr for both
    // tallies.  24 configurations of 2,500 atoms, twojmax 8, tallies and the energy row: 970 us, against 6,990 with the thread
    // per atom and descriptor and the second read that larger ones take; 200 of 250 atoms and one of 2,500: 900 against 6,240.
    const bool fused = ntypes == 1 && (C == 0 || sizes[0] <= BD_MAXH * BD_TH);
    if (fused) {
        // configurations of more than `atoms` atoms: the first so many of cfg_ord
        auto above = [&](int atoms) {
            return static_cast<int>(std::partition_point(sizes, sizes + C, [&](int n) { return n > atoms; }) - sizes);
        };
        const int n4 = above(4 * BD_TH), n1 = above(BD_TH);
        auto launch = [&](auto kernel, int first, int end) {
            if (first < end)
                hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(end - first) * IB), dim3(BD_TH), 0, st, dblist, rij, poff,
                                   in_off, in_idx, cfg_a0, cfg_p0, cfg_ord + first, IB, bd, bv, as);
        };
        launch(k_lsq_bd_bv<BD_MAXH>, 0, n4);
        launch(k_lsq_bd_bv<4>, n4, n1);
        launch(k_lsq_bd_bv<1>, n1, C);
    } else {
        hipLaunchKernelGGL(k_lsq_bd, dim3(nblocks(static_cast<long>(N) * IB, 256)), dim3(256), 0, st, dblist, poff,
                           in_off, in_idx, pti, type, cfg_of, cfg_a0, cfg_p0, N, IB, ntypes, bd);
    }
    hipLaunchKernelGGL(k_lsq_bi, dim3(static_cast<unsigned>(C) * kt), dim3(256), 0, st, blist, type, cfg_a0, IB, ntypes,
                       bi);
    if (!fused)
        hipLaunchKernelGGL(k_lsq_bv, dim3(static_cast<unsigned>(C) * kt), dim3(256), 0, st, dblist, rij, pti, cfg_p0, IB,
                           ntypes, bv, as);
}

// ---- weighted normal equations --------------------------------------------------------------------

// Chunk ch covers rows r < nrows <= 64: a(r, k) = A[abase + r*rs + k*cs], target T[tbase + r], weight
// W[wbase + r / wdiv].  Outputs e < K(K+1)/2 are L(k, l), k <= l (row-major upper triangle), then K entries of h.
//
// The sum over rows of w^2 [a | b]^T [a | b] on the FP64 matrix cores: the K + 1 columns of a chunk are staged column
// by column in LDS (row length 66: the operand reads of a half wave cover all banks), and each wave owns every
// fourth of the upper 16 x 16 tiles, one v_mfma_f64_16x16x4 per tile and four rows (operands A[m][k], B[k][n] at lanes
// m + 16k, n + 16k; the accumulator's register i of lane (m, g) is row 4i + g, column m).  Workgroup b takes chunks b,
// b + G, ... in order and writes its partial sums to part[b].  Bound: one read of the rows; the three groups of a batch
// with 315,000 force rows of 55 columns take 100 us, 430 us with one output per thread.
typedef double f64x4 __attribute__((ext_vector_type(4)));
constexpr int GR_LD = 66, GR_MAXT = 5;   // at most 5 x 16 columns (K <= 79)

template <int NT>
__global__ __launch_bounds__(256) void k_lsq_gram(const LsqChunk* __restrict__ chunks, int nchunks,
                                                  const double* __restrict__ A, const double* __restrict__ T,
                                                  const double* __restrict__ W, int K, double* __restrict__ part) {
    constexpr int TILES = NT * (NT + 1) / 2, PER = (TILES + 3) / 4;
    __shared__ double tile[NT * 16 * GR_LD];
    __shared__ double w2[64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, m16 = lane & 15, g4 = lane >> 4;
    const int nout = K * (K + 1) / 2 + K;
    int ti[PER], tj[PER];   // this wave's tiles, (row, column) of the upper triangle in row-major order
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        int id = min(wave + 4 * u, TILES - 1), i = 0;
        while (id >= NT - i) id -= NT - i++;
        ti[u] = i;
        tj[u] = i + id;
    }
    f64x4 acc[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u) acc[u] = f64x4{0.0, 0.0, 0.0, 0.0};
    for (int i = threadIdx.x; i < NT * 16 * GR_LD; i += 256) tile[i] = 0.0;   // the columns past K stay zero
    for (int ch = blockIdx.x; ch < nchunks; ch += gridDim.x) {
        const LsqChunk q = chunks[ch];
        __syncthreads();
        for (int i = threadIdx.x; i < 64 * K; i += 256) {   // rows fastest: contiguous reads when rs == 1
            const int k = i / 64, r = i % 64;
            tile[k * GR_LD + r] =
                r < q.nrows ? A[q.abase + static_cast<long>(r) * q.rs + static_cast<long>(k) * q.cs] : 0.0;
        }
        if (threadIdx.x < 64) {
            const int r = threadIdx.x;
            const double w = r < q.nrows ? W[q.wbase + r / q.wdiv] : 0.0;
            w2[r] = w * w;
            tile[K * GR_LD + r] = r < q.nrows ? T[q.tbase + r] : 0.0;
        }
        __syncthreads();
#pragma unroll 4
        for (int st = 0; st < 16; ++st) {
            const int r = 4 * st + g4;
            const double w = w2[r];
#pragma unroll
            for (int u = 0; u < PER; ++u) {
                const double a = w * tile[(16 * ti[u] + m16) * GR_LD + r];
                const double b = tile[(16 * tj[u] + m16) * GR_LD + r];
                acc[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc[u], 0, 0, 0);
            }
        }
    }
    double* __restrict__ o = part + static_cast<size_t>(blockIdx.x) * nout;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        if (wave + 4 * u >= TILES) continue;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int k = 16 * ti[u] + 4 * i + g4, l = 16 * tj[u] + m16;
            if (k < K && l == K) o[K * (K + 1) / 2 + k] = acc[u][i];
            if (k <= l && l < K) o[k * K - k * (k - 1) / 2 + l - k] = acc[u][i];
        }
    }
}

// out[e] = sum over b = 0..G-1 of part[b][e]: 64 outputs per workgroup, wave w adds partials w, w + 16, ... and the 16
// sums are added in wave order (1,024 partials: 7 us; 245 us when one lane added a whole output)
__global__ __launch_bounds__(1024) void k_lsq_gram_sum(const double* __restrict__ part, int G, int nout,
                                                       double* __restrict__ out) {
    __shared__ double sum[16][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, e = blockIdx.x * 64 + lane;
    double s = 0.0;
    if (e < nout) {
#pragma unroll 8
        for (int b = w; b < G; b += 16) s += part[static_cast<size_t>(b) * nout + e];
    }
    sum[w][lane] = s;
    __syncthreads();
    if (w != 0 || e >= nout) return;
    s = sum[0][lane];
#pragma unroll
    for (int k = 1; k < 16; ++k) s += sum[k][lane];
    out[e] = s;
}

int lsq_gram_max_columns() { return 77; }

void launch_lsq_gram(const LsqChunk* chunks, int nchunks, const double* A, const double* T, const double* W, int K,
                     double* part, int G, double* out, hipStream_t st) {
    const int nout = K * (K + 1) / 2 + K, NT = (K + 1 + 15) / 16;
    static_assert(GR_MAXT * 16 >= 78, "the columns and the target fit the tiles");
    G = G < nchunks ? G : nchunks;
    switch (NT) {
#define GRAM(NTV)                                                                                                       case NTV:                                                                                                               hipLaunchKernelGGL(k_lsq_gram<NTV>, dim3(G), dim3(256), 0, st, chunks, nchunks, A, T, W, K, part);                   break;
        GRAM(1)
        GRAM(2)
        GRAM(3)
        GRAM(4)
        GRAM(5)
#undef GRAM
        default: return;
    }
    hipLaunchKernelGGL(k_lsq_gram_sum, dim3(nblocks(nout, 64)), dim3(1024), 0, st, part, G, nout, out);
}

}  // namespace mdp
