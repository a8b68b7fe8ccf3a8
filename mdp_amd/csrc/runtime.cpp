// Host runtime shared by the drop-in entry points and the MD engine.
#include "runtime.hpp"

#include <algorithm>
#include <cstring>

namespace mdp {

namespace {
thread_local std::string g_error;
}

void set_error(const std::string& msg) { g_error = msg; }
void clear_error() { g_error.clear(); }
const char* get_error() { return g_error.c_str(); }

hipStream_t library_stream() {
    static hipStream_t s = [] {
        hipStream_t st = nullptr;
        if (hipStreamCreateWithFlags(&st, hipStreamNonBlocking) != hipSuccess) st = nullptr;
        return st;
    }();
    if (!s) throw Error("could not create the library HIP stream (no GPU?)");
    return s;
}

hipStream_t stream_after_callers() {
    MDP_HIP(hipDeviceSynchronize());
    return library_stream();
}

std::mutex& library_mutex() {
    static std::mutex m;
    return m;
}

void DevTables::upload(const SnapIndex& ix, const double* rootpq_h, const double* cg_h, const double* radelem_h,
                       const double* wjelem_h, const int* map_h, int ntypes, hipStream_t st) {
    std::vector<char> h;
    auto put = [&](const void* p, size_t bytes) {   // a null table is zeros
        const size_t o = h.size();
        h.resize(o + (bytes + 63) / 64 * 64, 0);
        if (p && bytes) std::memcpy(h.data() + o, p, bytes);
        return o;
    };
    const int jd = ix.J + 1;
    const size_t rootpq = put(rootpq_h ? rootpq_h : ix.rootpq.data(), sizeof(double) * (ix.J + 2) * (ix.J + 2));
    const size_t cg = put(cg_h ? cg_h : ix.cglist.data(), sizeof(double) * ix.idxcg_max);
    const size_t radelem = put(radelem_h, sizeof(double) * (ntypes + 1));
    const size_t wjelem = put(wjelem_h, sizeof(double) * (ntypes + 1));
    const size_t map = put(map_h, sizeof(int) * (ntypes + 1));
    const size_t idxz = put(ix.idxz.data(), sizeof(int) * ix.idxz.size());
    const size_t idxb = put(ix.idxb.data(), sizeof(int) * ix.idxb.size());
    const size_t idxu_block = put(ix.idxu_block.data(), sizeof(int) * jd);
    const size_t idxz_block = put(ix.idxz_block.data(), sizeof(int) * jd * jd * jd);
    const size_t idxb_block = put(ix.idxb_block.data(), sizeof(int) * jd * jd * jd);
    const size_t idxcg_block = put(ix.idxcg_block.data(), sizeof(int) * jd * jd * jd);
    if (idx.J != ix.J || h != content) {
        content.clear();
        idx = ix;
        buf.ensure(h.size());
        MDP_HIP(hipMemcpyAsync(buf.p, h.data(), h.size(), hipMemcpyHostToDevice, st));
        MDP_HIP(hipStreamSynchronize(st));
        content.swap(h);
    }
    char* const d = buf.as<char>();
    view.J = ix.J;
    view.idxu_max = ix.idxu_max;
    view.idxz_max = ix.idxz_max;
    view.idxb_max = ix.idxb_max;
    view.idxcg_max = ix.idxcg_max;
    view.rootpq = reinterpret_cast<double*>(d + rootpq);
    view.cg = reinterpret_cast<double*>(d + cg);
    view.radelem = reinterpret_cast<double*>(d + radelem);
    view.wjelem = reinterpret_cast<double*>(d + wjelem);
    view.map = reinterpret_cast<int*>(d + map);
    view.idxz = reinterpret_cast<int*>(d + idxz);
    view.idxb = reinterpret_cast<int*>(d + idxb);
    view.idxu_block = reinterpret_cast<int*>(d + idxu_block);
    view.idxz_block = reinterpret_cast<int*>(d + idxz_block);
    view.idxb_block = reinterpret_cast<int*>(d + idxb_block);
    view.idxcg_block = reinterpret_cast<int*>(d + idxcg_block);
}

std::vector<double> y_beta_table(const SnapIndex& ix, const double* beta, int e1, int e2, int e3, int ne, int ielem,
                                 int ncoeffall, int bnorm) {
    const int J = ix.J, jd = J + 1;
    std::vector<double> out;
    for (int j1 = 0; j1 <= J; ++j1)
        for (int j2 = 0; j2 <= j1; ++j2)
            for (int j = j1 - j2; j <= std::min(J, j1 + j2); j += 2) {
                double w;
                if (j >= j1) {
                    const int jjb = ix.idxb_block[j + j2 * jd + j1 * jd * jd];
                    const int it = ((e1 * ne + e2) * ne + e3) * ix.idxb_max + jjb + 1 + ielem * ncoeffall;
                    w = (j1 == j) ? ((j2 == j) ? 3 * beta[it] : 2 * beta[it]) : beta[it];
                } else if (j >= j2) {
                    const int jjb = ix.idxb_block[j1 + j2 * jd + j * jd * jd];
                    const int it = ((e3 * ne + e2) * ne + e1) * ix.idxb_max + jjb + 1 + ielem * ncoeffall;
                    w = (j2 == j) ? 2 * beta[it] : beta[it];
                } else {
                    const int jjb = ix.idxb_block[j1 + j * jd + j2 * jd * jd];
                    const int it = ((e2 * ne + e3) * ne + e1) * ix.idxb_max + jjb + 1 + ielem * ncoeffall;
                    w = beta[it];
                }
                if (!bnorm && j1 > j) w *= (j1 + 1) / (j + 1.0);
                if (bnorm) w /= (j + 1);
                out.push_back(w);
            }
    return out;
}

void y_triple_weights(const SnapIndex& ix, int bnorm, std::vector<int>& jjb, std::vector<double>& fac) {
    // read off the weight table with one-hot coefficient vectors
    const int nc = ix.idxb_max + 1;
    jjb.clear();
    fac.clear();
    for (int k = 0; k < ix.idxb_max; ++k) {
        std::vector<double> beta(nc, 0.0);
        beta[1 + k] = 1.0;
        const std::vector<double> t = y_beta_table(ix, beta.data(), 0, 0, 0, 1, 0, nc, bnorm);
        if (jjb.empty()) {
            jjb.assign(t.size(), -1);
            fac.assign(t.size(), 0.0);
        }
        for (size_t q = 0; q < t.size(); ++q)
            if (t[q] != 0.0) {
                if (jjb[q] >= 0) throw Error("coupling triple with two bispectrum coefficients");
                jjb[q] = k;
                fac[q] = t[q];
            }
    }
    for (int q : jjb)
        if (q < 0) throw Error("coupling triple without a bispectrum coefficient");
}

}  // namespace mdp
