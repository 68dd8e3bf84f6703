// Host-side multigrid lists of a batch of boxes, for test_cpu_amg_lists.py:
//   amg_lists_check threads sx sy sz limit element_limit nx ny nz [nx ny nz ...]
// builds the hierarchy for the coupling strengths s and the A P lists over the
// element values with the given limits (0: the defaults) and prints their
// lengths and hashes, or what the builder refused.  The builder asks for the
// number of host threads; this program's answer takes the place of the library's.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <thread>

#include "mhs_amg.h"
#include "mhs_ebe.h"
#include "mhs_kernels.h"
#include "mhs_structure.h"

using namespace mhs;

static unsigned g_threads = 1, g_asked = 0;
unsigned std::thread::hardware_concurrency() noexcept {
    ++g_asked;
    return g_threads;
}

static unsigned long long g_hash = 1469598103934665603ull;
template <class V>
static void mix(const V &v) {
    for (auto x : v) g_hash = (g_hash ^ (unsigned long long)(long long)x) * 1099511628211ull;
    g_hash = (g_hash ^ v.size()) * 1099511628211ull;
}

int main(int argc, char **argv) {
    g_threads = (unsigned)std::atoi(argv[1]);
    const Strength st = {std::atof(argv[2]), std::atof(argv[3]), std::atof(argv[4])};
    const size_t limit = std::strtoull(argv[5], nullptr, 10), elimit = std::strtoull(argv[6], nullptr, 10);
    std::vector<int> icp{0}, fp{0}, nb, ijk, family;
    for (int a = 7; a + 2 < argc; a += 3) {
        const int nx = std::atoi(argv[a]), ny = std::atoi(argv[a + 1]), nz = std::atoi(argv[a + 2]), c0 = icp.back();
        for (int c = 0; c < nx * ny * nz; ++c) {
            const int q[3] = {c % nx, c / nx % ny, c / (nx * ny)}, n[3] = {nx, ny, nz}, step[3] = {1, nx, nx * ny};
            ijk.insert(ijk.end(), q, q + 3);
            for (int d = 0; d < 3; ++d)
                for (int up = 0; up < 2; ++up) {
                    const bool in = up ? q[d] + 1 < n[d] : q[d] > 0;
                    nb.push_back(in ? c0 + c + (up ? step[d] : -step[d]) : -1);
                    family.push_back(d * 8 + (q[0] & 1));
                }
            fp.push_back((int)nb.size());
        }
        icp.push_back(c0 + nx * ny * nz);
    }
    Topology T;
    std::string e = build_topology(T, (int)icp.size() - 1, icp.data(), icp.back(), fp.data(), nb.data(), nullptr, nullptr,
                                   family.data());
    EbeLayout E;
    if (e.empty()) e = build_ebe(E, T, ijk.data());
    AmgHierarchy H;
    if (e.empty()) e = build_amg(H, T, ijk, st, true, limit ? limit : kMaxList);
    std::printf("asked %u\namg %s\n", g_asked, e.empty() ? "ok" : e.c_str());
    if (!e.empty()) return 0;
    size_t longest = H.ap.src.size();
    for (const AmgLevel &l : H.lev) {
        longest = std::max({longest, l.src.size(), l.t_pa.size(), l.p_src.size()});
        mix(l.row_ptr); mix(l.col); mix(l.diag); mix(l.src_ptr); mix(l.src); mix(l.agg); mix(l.agg2);
        mix(l.child_ptr); mix(l.child); mix(l.src2); mix(l.p_ptr); mix(l.p_col); mix(l.p_own); mix(l.p_src_ptr);
        mix(l.p_src); mix(l.pt_ptr); mix(l.pt_col); mix(l.pt_map); mix(l.p_tpos); mix(l.t_ptr); mix(l.t_col);
        mix(l.t_pair_ptr); mix(l.t_pa); mix(l.t_pb); mix(l.t_p);
    }
    mix(H.ap.slice_ptr); mix(H.ap.col); mix(H.ap.src_ptr); mix(H.ap.src); mix(H.ap.slice);
    mix(H.tail.tab); mix(H.tail.idx);
    std::printf("matrix %lld\nap %zu\nlongest %zu\n", (long long)T.slice_ptr[T.nslices], H.ap.src.size(), longest);
    std::vector<ListEnd> ptr;
    std::vector<int> src;
    e = ebe_ap_lists(E, T, H.ap, H.lev[1].agg, H.lev[1].agg2, ptr, src, elimit ? elimit : kMaxList);
    mix(ptr); mix(src);
    std::printf("element %s\nelement_list %zu\nhash %llx\n", e.empty() ? "ok" : e.c_str(), src.size(), g_hash);
    // what the autotuner would time: per right-hand sides and value size the first
    // level of every candidate's tail
    DevAmg A{};
    A.nlev = H.nlev();
    A.tail_first = H.tail.first;
    A.tail_lds = kTailBytes;
    for (int l = 0; l < A.nlev; ++l) {
        A.tail_iend[l] = H.tail.iend[l];
        A.tail_vend[l] = H.tail.vend[l];
        A.tail_vec[l] = H.tail.vec[l];
        for (size_t t = 0; l > 0 && t + 1 < H.lev[l].inst_ptr.size(); ++t)
            A.max_rows[l] = std::max(A.max_rows[l], H.lev[l].inst_ptr[t + 1] - H.lev[l].inst_ptr[t]);
    }
    for (int vsize : {4, 8})
        for (int nrhs : {1, 3}) {
            std::printf("tail_%d_%d", vsize, nrhs);
            for (int r : tail_candidates(A, nrhs, vsize)) std::printf(" %d", tail_level(A, r, nrhs, vsize));
            std::printf(" | %d\n", tail_level(A, 32768, nrhs, vsize));
        }
    return 0;
}
