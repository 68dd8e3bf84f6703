// Aggregation multigrid hierarchy (host-side set-up); see mhs_amg.h.
#include "mhs_amg.h"
#include "mhs_lists.h"

#include <algorithm>
#include <array>
#include <cmath>
#include <numeric>

namespace mhs {

namespace {

void children(AmgLevel &C, int nf) {
    const bool two = !C.agg2.empty();
    C.child_ptr.assign(C.n + 1, 0);
    for (int i = 0; i < nf; ++i) {
        if (C.agg[i] >= 0) C.child_ptr[C.agg[i] + 1]++;
        if (two && C.agg2[i] >= 0) C.child_ptr[C.agg2[i] + 1]++;
    }
    for (int I = 0; I < C.n; ++I) C.child_ptr[I + 1] += C.child_ptr[I];
    C.child.assign(C.child_ptr[C.n], 0);
    std::vector<int> fill(C.child_ptr.begin(), C.child_ptr.end() - 1);
    for (int i = 0; i < nf; ++i) {
        const bool half = two && C.agg2[i] >= 0;
        if (C.agg[i] >= 0) C.child[fill[C.agg[i]]++] = half ? ~i : i;
        if (half) C.child[fill[C.agg2[i]]++] = ~i;
    }
}

// Position of each row's diagonal entry (-1: none).
void find_diagonal(AmgLevel &C) {
    C.diag.assign(C.n, -1);
    for (int I = 0; I < C.n; ++I)
        for (int e = C.row_ptr[I]; e < C.row_ptr[I + 1]; ++e)
            if (C.col[e] == I) C.diag[I] = e;
}

// Sparsity of P'AP and the gather lists, coarse row by coarse row: the
// entries (agg(j), pos) of the coarse row's children by column.
// row_entries(i, emit) must call emit(j, pos) for every stored entry of
// finer row i (COARSE: j is already the coarse column, the entries being
// those of A P).  Requires children() to have run.
template <bool COARSE = false, class RowEntries>
bool galerkin_pattern(AmgLevel &C, size_t max_list, RowEntries row_entries) {
    const bool ok = build_rows(C.n, C.row_ptr, C.col, C.src_ptr, C.src, nullptr, max_list, [&]() {
        return [&, rows = ByColumn<int>(C.n)](int I, RowPart &R) mutable {
            rows.start();
            for (int k = C.child_ptr[I]; k < C.child_ptr[I + 1]; ++k)
                row_entries(C.child[k], [&](int j, int pos) {
                    const int J = COARSE ? j : C.agg[j];
                    if (J >= 0) rows.put(J, pos);
                });
            rows.finish([&](int J, int *e, int n) {
                // by position whatever its weight (from CSR rows they come so)
                if constexpr (COARSE)
                    std::sort(e, e + n, [](int x, int y) { return std::max(x, ~x) < std::max(y, ~y); });
                R.col.push_back(J);
                R.src.insert(R.src.end(), e, e + n);
                R.end.push_back(ListEnd(R.src.size()));
            });
        };
    });
    if (ok) find_diagonal(C);
    return ok;
}

// naggs: rows of level 1.  False: too long.
bool build_ap(ApPattern &P, const Topology &T, int naggs, const std::vector<int> &agg, const std::vector<int> &agg2,
              size_t max_list) {
    const int ns = T.nslices, nt = ranges(ns, 32);
    P.slice_ptr.assign(ns + 1, 0);
    // slice by slice: the rows' entries (aggregate, position; ~position: half the
    // entry), sorted, then the slots and their lists in slot order
    struct Run { int J, n, at; };
    struct Part { std::vector<int> slice, col, src; std::vector<ListEnd> end; };
    std::vector<Part> parts(nt);
    std::vector<int> width(ns, 0);
    in_ranges(ns, nt, [&](int t, int b, int e) {
        Part &Q = parts[t];
        ByColumn<int> row(naggs);
        std::vector<std::vector<Run>> runs(kSlice);
        std::vector<int> pos;
        for (int sl = b; sl < e; ++sl) {
            size_t w = 0;
            pos.clear();
            for (int l = 0; l < kSlice; ++l) {
                const int f = sl * kSlice + l;
                const long long base = T.slice_ptr[sl] + l;
                row.start();
                for (int k = 0; k < T.row_len[f]; ++k) {
                    const long long p = base + (long long)k * kSlice;
                    const int j = T.col[p], J = agg[j], J2 = agg2[j];
                    if (J >= 0) row.put(J, J2 >= 0 ? ~int(p) : int(p));
                    if (J2 >= 0) row.put(J2, ~int(p));
                }
                auto &r = runs[l];
                r.clear();
                row.finish([&](int J, int *e, int n) {
                    std::sort(e, e + n);
                    r.push_back({J, n, int(pos.size())});
                    pos.insert(pos.end(), e, e + n);
                });
                w = std::max(w, r.size());
            }
            width[sl] = int(w);
            for (size_t k = 0; k < w; ++k) {
                Q.slice.push_back(sl);
                for (int l = 0; l < kSlice; ++l) {
                    const bool in = k < runs[l].size();
                    Q.col.push_back(in ? runs[l][k].J : 0);
                    if (in)
                        Q.src.insert(Q.src.end(), pos.begin() + runs[l][k].at,
                                     pos.begin() + runs[l][k].at + runs[l][k].n);
                    Q.end.push_back(ListEnd(Q.src.size()));
                }
            }
        }
    });
    for (int sl = 0; sl < ns; ++sl) P.slice_ptr[sl + 1] = P.slice_ptr[sl] + (long long)width[sl] * kSlice;
    std::vector<std::vector<int>> slices(nt), cols(nt), srcs(nt);
    std::vector<std::vector<ListEnd>> ends(nt);
    for (int t = 0; t < nt; ++t) {
        slices[t].swap(parts[t].slice);
        cols[t].swap(parts[t].col);
        ends[t].swap(parts[t].end);
        srcs[t].swap(parts[t].src);
    }
    if (too_long(total(cols), total(srcs), max_list)) return false;
    P.slice.clear();
    P.col.clear();
    P.src.clear();
    append(P.slice, slices);
    append(P.col, cols);
    const std::vector<size_t> at = append(P.src, srcs);
    for (int t = 0; t < nt; ++t)
        for (ListEnd &e : ends[t]) e += ListEnd(at[t]);
    P.src_ptr.assign(1, 0);
    append(P.src_ptr, ends);
    return true;
}

// Smoothed-aggregation transfer F -> C (C.agg set, F's CSR pattern known):
// the patterns of P, P', T = A_F P and A_C = P' T, with the gather / pair
// lists that let every solve fill their values on the device.
bool sa_transfer(AmgLevel &F, AmgLevel &C, size_t max_list) {
    const int n = F.n;
    F.sa_out = true;
    F.p_own.assign(n, -1);
    if (!build_rows(n, F.p_ptr, F.p_col, F.p_src_ptr, F.p_src, nullptr, max_list, [&]() {
        return [&, row = ByColumn<int>(C.n)](int i, RowPart &R) mutable {
            row.start();
            for (int k = F.row_ptr[i]; k < F.row_ptr[i + 1]; ++k) row.put(C.agg[F.col[k]], k);
            row.finish([&](int J, int *e, int m) {
                R.col.push_back(J);
                R.src.insert(R.src.end(), e, e + m);
                R.end.push_back(ListEnd(R.src.size()));
            });
        };
    })) return false;
    for (int i = 0; i < n; ++i)
        for (int q = F.p_ptr[i]; q < F.p_ptr[i + 1]; ++q)
            if (F.p_col[q] == C.agg[i]) F.p_own[i] = q;
    // P' (rows of C)
    F.pt_ptr.assign(C.n + 1, 0);
    for (int J : F.p_col) F.pt_ptr[J + 1]++;
    for (int I = 0; I < C.n; ++I) F.pt_ptr[I + 1] += F.pt_ptr[I];
    F.pt_col.assign(F.p_col.size(), 0);
    F.pt_map.assign(F.p_col.size(), 0);
    {
        std::vector<int> fill(F.pt_ptr.begin(), F.pt_ptr.end() - 1);
        for (int i = 0; i < n; ++i)
            for (int q = F.p_ptr[i]; q < F.p_ptr[i + 1]; ++q) {
                const int e = fill[F.p_col[q]]++;
                F.pt_col[e] = i;
                F.pt_map[e] = q;
            }
        F.p_tpos.assign(F.p_col.size(), 0);
        for (size_t e = 0; e < F.pt_map.size(); ++e) F.p_tpos[F.pt_map[e]] = int(e);
    }
    // T = A P, then A_C = P' T: per column the pairs of the two factors' positions,
    // which come in ascending order
    using Pair = std::pair<int, int>;
    auto emit = [](ByColumn<Pair> &row, RowPart &R) {
        row.finish([&](int J, const Pair *e, int m) {
            R.col.push_back(J);
            for (int k = 0; k < m; ++k) {
                R.src.push_back(e[k].first);
                R.src2.push_back(e[k].second);
            }
            R.end.push_back(ListEnd(R.src.size()));
        });
    };
    if (!build_rows(n, F.t_ptr, F.t_col, F.t_pair_ptr, F.t_pa, &F.t_pb, max_list, [&]() {
        return [&, row = ByColumn<Pair>(C.n)](int i, RowPart &R) mutable {
            row.start();
            for (int k = F.row_ptr[i]; k < F.row_ptr[i + 1]; ++k) {
                const int j = F.col[k];
                for (int q = F.p_ptr[j]; q < F.p_ptr[j + 1]; ++q) row.put(F.p_col[q], {k, q});
            }
            emit(row, R);
        };
    })) return false;
    C.sa_in = true;
    if (!build_rows(C.n, C.row_ptr, C.col, C.src_ptr, C.src, &C.src2, max_list, [&]() {
        return [&, row = ByColumn<Pair>(C.n)](int I, RowPart &R) mutable {
            row.start();
            for (int e = F.pt_ptr[I]; e < F.pt_ptr[I + 1]; ++e) {
                const int i = F.pt_col[e], q = F.pt_map[e];
                for (int t = F.t_ptr[i]; t < F.t_ptr[i + 1]; ++t) row.put(F.t_col[t], {q, t});
            }
            emit(row, R);
        };
    })) return false;
    find_diagonal(C);
    return true;
}

// Block factors for one transfer: 2 along the coarsenable directions whose
// strength is at least theta times the strongest coarsenable one.
std::array<int, 3> choose_blocks(const Strength &s, double theta, const std::vector<int> &cur) {
    const int ninst = int(cur.size() / 3);
    bool can[3] = {false, false, false};
    for (int t = 0; t < ninst; ++t)
        for (int d = 0; d < 3; ++d) can[d] = can[d] || cur[3 * t + d] > 1;
    double smax = 0.0;
    for (int d = 0; d < 3; ++d)
        if (can[d]) smax = std::max(smax, s[d]);
    std::array<int, 3> b{1, 1, 1};
    for (int d = 0; d < 3; ++d)
        if (can[d] && (!(smax > 0.0) || s[d] >= theta * smax)) b[d] = 2;
    return b;
}

// Index blocks and offsets of the one-workgroup tail (see TailLayout), from the
// coarsest level up to the finest that still fits: 16-bit local indices, at
// most 4096 rows of an instance and index and FP64 value prefixes of at most
// kTailBytes.  Level prefixes are padded to 16 bytes for the vector copies.
void build_tail(AmgHierarchy &H) {
    TailLayout &T = H.tail;
    const int L = int(H.lev.size()), ninst = int(H.lev.back().inst_ptr.size()) - 1;
    T = TailLayout();
    T.tab.assign((size_t)ninst * L * TL_K, 0);
    T.iend.assign(L, 0);
    T.vend.assign(L, 0);
    T.vec.assign(L, 0);
    // sizes first: the finest level every instance can hold
    T.first = L - 1;
    for (int l = L - 1; l >= 1; --l) {
        const AmgLevel &F = H.lev[l];
        bool fits = true;
        for (int s = 0; s < ninst; ++s) {
            int *t = &T.tab[((size_t)s * L + l) * TL_K];
            const int *up = l + 1 < L ? t + TL_K : nullptr;
            t[TL_R0] = F.inst_ptr[s];
            const long long n = t[TL_N] = F.inst_ptr[s + 1] - F.inst_ptr[s];
            long long ni = up ? up[TL_IEND] : 0, nv = up ? up[TL_VEND] : 0;
            t[TL_VEC] = up ? up[TL_VEC] + (l + 2 < L ? 3 : 2) * up[TL_N] : 0;
            auto take = [](long long &at, long long k) { const long long o = at; at += k; return (int)o; };
            if (!up) {
                t[TL_VAL] = take(nv, n * n);
            } else {
                const long long nC = up[TL_N];
                t[TL_E0] = F.row_ptr[t[TL_R0]];
                t[TL_NNZ] = F.row_ptr[t[TL_R0] + n] - t[TL_E0];
                t[TL_RP] = take(ni, n + 1);
                t[TL_COL] = take(ni, t[TL_NNZ]);
                t[TL_VAL] = take(nv, t[TL_NNZ]);
                t[TL_WD] = take(nv, n);
                if (F.sa_out) {
                    t[TL_PT0] = F.pt_ptr[up[TL_R0]];
                    t[TL_NPT] = F.pt_ptr[up[TL_R0] + nC] - t[TL_PT0];
                    t[TL_T0] = F.t_ptr[t[TL_R0]];
                    t[TL_NT] = F.t_ptr[t[TL_R0] + n] - t[TL_T0];
                    t[TL_PTP] = take(ni, nC + 1);
                    t[TL_PTC] = take(ni, t[TL_NPT]);
                    t[TL_TP] = take(ni, n + 1);
                    t[TL_TC] = take(ni, t[TL_NT]);
                    t[TL_PTV] = take(nv, t[TL_NPT]);
                    t[TL_MV] = take(nv, t[TL_NT]);
                } else {
                    t[TL_CP] = take(ni, nC + 1);
                    t[TL_CH] = take(ni, n);
                    t[TL_AGG] = take(ni, n);
                }
            }
            ni = (ni + 7) / 8 * 8;
            nv = (nv + 3) / 4 * 4;
            // (the coarsest level always fits: at most kMaxCoarsest rows)
            if (up && (n > 4096 || t[TL_NNZ] > 65535 || t[TL_NPT] > 65535 || t[TL_NT] > 65535 ||
                       2 * ni + 8 * nv > kTailBytes))
                fits = false;
            t[TL_IEND] = (int)std::min<long long>(ni, 1 << 30);
            t[TL_VEND] = (int)std::min<long long>(nv, 1 << 30);
            T.iend[l] = std::max(T.iend[l], t[TL_IEND]);
            T.vend[l] = std::max(T.vend[l], t[TL_VEND]);
            T.vec[l] = std::max(T.vec[l], t[TL_VEC] + (up ? 3 : 2) * (int)n);
        }
        if (!fits) break;
        T.first = l;
    }
    long long ni = 0, nv = 0;
    for (int s = 0; s < ninst; ++s) {
        int *t0 = &T.tab[(size_t)s * L * TL_K];
        t0[0] = int(ni);
        t0[1] = int(nv);
        ni += t0[T.first * TL_K + TL_IEND];
        nv += t0[T.first * TL_K + TL_VEND];
    }
    if (ni > 0x7fffffffLL || nv > 0x7fffffffLL) {   // 32-bit offsets: the coarsest level alone
        T.first = L - 1;
        ni = nv = 0;
        for (int s = 0; s < ninst; ++s) {
            int *t0 = &T.tab[(size_t)s * L * TL_K];
            t0[0] = 0;
            t0[1] = int(nv);
            nv += t0[(L - 1) * TL_K + TL_VEND];
        }
    }
    T.nval = nv;
    T.idx.assign(std::max<long long>(ni, 8), 0);
    for (int s = 0; s < ninst; ++s)
        for (int l = T.first; l + 1 < L; ++l) {
            const AmgLevel &F = H.lev[l], &C = H.lev[l + 1];
            const int *t = &T.tab[((size_t)s * L + l) * TL_K], *up = t + TL_K;
            uint16_t *o = &T.idx[T.tab[(size_t)s * L * TL_K]];
            const int r0 = t[TL_R0], n = t[TL_N], c0 = up[TL_R0], nC = up[TL_N];
            for (int i = 0; i <= n; ++i) o[t[TL_RP] + i] = uint16_t(F.row_ptr[r0 + i] - t[TL_E0]);
            for (int e = 0; e < t[TL_NNZ]; ++e) o[t[TL_COL] + e] = uint16_t(F.col[t[TL_E0] + e] - r0);
            if (F.sa_out) {
                for (int i = 0; i <= nC; ++i) o[t[TL_PTP] + i] = uint16_t(F.pt_ptr[c0 + i] - t[TL_PT0]);
                for (int e = 0; e < t[TL_NPT]; ++e) o[t[TL_PTC] + e] = uint16_t(F.pt_col[t[TL_PT0] + e] - r0);
                for (int i = 0; i <= n; ++i) o[t[TL_TP] + i] = uint16_t(F.t_ptr[r0 + i] - t[TL_T0]);
                for (int e = 0; e < t[TL_NT]; ++e) o[t[TL_TC] + e] = uint16_t(F.t_col[t[TL_T0] + e] - c0);
            } else {
                const int k0 = C.child_ptr[c0];
                for (int i = 0; i <= nC; ++i) o[t[TL_CP] + i] = uint16_t(C.child_ptr[c0 + i] - k0);
                for (int k = k0; k < C.child_ptr[c0 + nC]; ++k) o[t[TL_CH] + k - k0] = uint16_t(C.child[k] - r0);
                for (int i = 0; i < n; ++i) o[t[TL_AGG] + i] = uint16_t(C.agg[r0 + i] - c0);
            }
        }
}

}  // namespace

std::string instance_dims(const Topology &T, const std::vector<int> &ijk, std::vector<int> &dims) {
    const int ninst = T.ninst;
    if ((int)ijk.size() != 3 * T.nc) return "logical cell indices: need 3 per cell";
    dims.assign(3 * ninst, 0);
    for (int t = 0; t < ninst; ++t)
        for (int c = T.inst_cellpos[t]; c < T.inst_cellpos[t + 1]; ++c)
            for (int d = 0; d < 3; ++d) {
                if (ijk[3 * c + d] < 0) return "logical cell indices must be non-negative";
                dims[3 * t + d] = std::max(dims[3 * t + d], ijk[3 * c + d] + 1);
            }
    return "";
}

std::vector<std::array<int, 3>> coarsening_plan(const Strength &strength, const std::vector<int> &dims) {
    const int ninst = int(dims.size() / 3);
    Strength s = strength;
    for (double &v : s)
        if (!(v > 0.0) || !std::isfinite(v)) v = 0.0;
    std::vector<int> cur = dims;
    std::vector<std::array<int, 3>> plan;
    for (;;) {
        if (!plan.empty()) {
            long long mx = 0;
            for (int t = 0; t < ninst; ++t)
                mx = std::max(mx, (long long)cur[3 * t] * cur[3 * t + 1] * cur[3 * t + 2]);
            if (mx <= kMaxCoarsest || plan.size() >= 40) break;
        }
        const std::array<int, 3> b = choose_blocks(s, plan.empty() ? 0.5 : 0.25, cur);
        plan.push_back(b);
        for (int t = 0; t < ninst; ++t)
            for (int d = 0; d < 3; ++d) cur[3 * t + d] = (cur[3 * t + d] + b[d] - 1) / b[d];
        const Strength s0 = s;
        for (int d = 0; d < 3; ++d) s[d] = s0[d] * b[(d + 1) % 3] * b[(d + 2) % 3] / b[d];
    }
    return plan;
}

std::string build_amg(AmgHierarchy &H, const Topology &T, const std::vector<int> &ijk, const Strength &strength,
                      bool smoothed, size_t max_list) {
    H = AmgHierarchy();
    const char *const kTooLong = "grid too large for the 32-bit multigrid gather lists";
    const int ninst = T.ninst;
    if (T.slice_ptr[T.nslices] > 0x7fffffffLL)
        return "face matrix too large for the 32-bit multigrid gather lists";
    std::vector<int> dims;
    std::string ed = instance_dims(T, ijk, dims);
    if (!ed.empty()) return ed;
    H.blocks = coarsening_plan(strength, dims);
    H.lev.emplace_back();  // level 0 is the SELL face matrix
    // ---- level 1: faces -> blocks of their cells.  A face inside a block takes
    // the block's value, a face between two blocks the mean of both (a periodic
    // pair's faces those of the two cells across it): linear pressures are
    // interpolated exactly from block means, so the coarse operator is not
    // too stiff across the blocks as it is with the owner's block alone
    // (51 -> 35 iterations at 128x128x64).
    {
        const std::array<int, 3> &b0 = H.blocks[0];
        AmgLevel L1;
        L1.inst_ptr.assign(ninst + 1, 0);
        L1.dims.resize(3 * ninst);
        for (int t = 0; t < ninst; ++t) {
            long long m = 1;
            for (int d = 0; d < 3; ++d) {
                L1.dims[3 * t + d] = (dims[3 * t + d] + b0[d] - 1) / b0[d];
                m *= L1.dims[3 * t + d];
            }
            L1.inst_ptr[t + 1] = L1.inst_ptr[t] + int(m);
        }
        L1.n = L1.inst_ptr[ninst];
        L1.agg.assign(T.nfp, -1);
        L1.agg2.assign(T.nfp, -1);
        std::vector<int> inst_of_cell(T.nc);
        for (int t = 0; t < ninst; ++t)
            for (int c = T.inst_cellpos[t]; c < T.inst_cellpos[t + 1]; ++c) inst_of_cell[c] = t;
        auto block = [&](int c) {
            const int t = inst_of_cell[c], *bd = &L1.dims[3 * t];
            const int I = ijk[3 * c] / b0[0], J = ijk[3 * c + 1] / b0[1], K = ijk[3 * c + 2] / b0[2];
            return L1.inst_ptr[t] + I + bd[0] * (J + bd[1] * K);
        };
        for (int f = 0; f < T.nfp; ++f) {
            const int h = T.dof_hf[f];
            if (h < 0) continue;
            L1.agg[f] = block(T.hf_cell[h]);
            const int twin = T.hf_twin[h];   // the face's other side, or its periodic partner
            const int g = twin >= 0 ? block(T.hf_cell[twin]) : L1.agg[f];
            if (g != L1.agg[f]) L1.agg2[f] = g;
        }
        children(L1, T.nfp);
        // A_1 = P' (A P): each entry sums the A P slots of its row's faces
        // (about 7 per face row) instead of the face matrix's entries (11)
        if (!build_ap(H.ap, T, L1.n, L1.agg, L1.agg2, max_list)) return kTooLong;
        const ApPattern &ap = H.ap;
        const bool fits = galerkin_pattern<true>(L1, max_list, [&](int child, auto emit) {
            const bool half = child < 0;
            const int f = half ? ~child : child;
            const long long base = ap.slice_ptr[f / kSlice] + f % kSlice;
            const int w = int((ap.slice_ptr[f / kSlice + 1] - ap.slice_ptr[f / kSlice]) / kSlice);
            for (int e = 0; e < w; ++e) {
                const long long q = base + (long long)e * kSlice;
                if (ap.src_ptr[q + 1] > ap.src_ptr[q]) emit(ap.col[q], half ? ~int(q) : int(q));   // padding slots sum nothing
            }
        });
        if (!fits) return kTooLong;
        H.lev.push_back(std::move(L1));
    }
    // ---- coarser levels: group the blocks again until every instance is small
    bool sa_done = false;
    for (size_t l = 1; l < H.blocks.size(); ++l) {
        const AmgLevel &F = H.lev.back();
        const std::array<int, 3> &bl = H.blocks[l];
        AmgLevel C;
        C.inst_ptr.assign(ninst + 1, 0);
        C.dims.resize(3 * ninst);
        for (int t = 0; t < ninst; ++t) {
            long long m = 1;
            for (int d = 0; d < 3; ++d) {
                C.dims[3 * t + d] = (F.dims[3 * t + d] + bl[d] - 1) / bl[d];
                m *= C.dims[3 * t + d];
            }
            C.inst_ptr[t + 1] = C.inst_ptr[t] + int(m);
        }
        C.n = C.inst_ptr[ninst];
        C.agg.assign(F.n, -1);
        for (int t = 0; t < ninst; ++t) {
            const int *fd = &F.dims[3 * t], *cd = &C.dims[3 * t];
            for (int r = F.inst_ptr[t]; r < F.inst_ptr[t + 1]; ++r) {
                const int loc = r - F.inst_ptr[t];
                const int i = loc % fd[0], j = (loc / fd[0]) % fd[1], k = loc / (fd[0] * fd[1]);
                C.agg[r] = C.inst_ptr[t] + i / bl[0] + cd[0] * (j / bl[1] + cd[1] * (k / bl[2]));
            }
        }
        AmgLevel &Fr = H.lev.back();
        children(C, F.n);
        // smooth one transfer: the first from a level with at most an eighth
        // as many rows as there are faces (cheap next to the face level),
        // most of the gain in iterations, while the other levels keep the
        // sparse stencils of piecewise-constant aggregation (smoothing widens
        // every stencil)
        if (smoothed && !sa_done && 8LL * Fr.n <= (long long)T.nf_total) {
            sa_done = true;
            if (!sa_transfer(Fr, C, max_list)) return kTooLong;
            // the up-sweep stores M = P - w D^-1 T on T's pattern, which holds
            // P's (A holds its diagonal; both rows sorted)
            Fr.t_p.assign(Fr.t_col.size(), -1);
            for (int i = 0; i < Fr.n; ++i) {
                int t = Fr.t_ptr[i];
                for (int q = Fr.p_ptr[i]; q < Fr.p_ptr[i + 1]; ++q) {
                    while (t < Fr.t_ptr[i + 1] && Fr.t_col[t] < Fr.p_col[q]) ++t;
                    if (t == Fr.t_ptr[i + 1] || Fr.t_col[t] != Fr.p_col[q])
                        return "smoothed transfer: a row of P outside the pattern of A P";
                    Fr.t_p[t] = q;
                }
            }
        } else {
            const bool fits = galerkin_pattern(C, max_list, [&](int r, auto emit) {
                for (int k = Fr.row_ptr[r]; k < Fr.row_ptr[r + 1]; ++k) emit(Fr.col[k], k);
            });
            if (!fits) return kTooLong;
        }
        H.lev.push_back(std::move(C));
    }
    const AmgLevel &Lc = H.lev.back();
    for (int t = 0; t < ninst; ++t)
        if (Lc.inst_ptr[t + 1] - Lc.inst_ptr[t] > kMaxCoarsest) return "multigrid hierarchy does not coarsen";
    H.coarse_off.assign(ninst + 1, 0);
    for (int t = 0; t < ninst; ++t) {
        const int m = Lc.inst_ptr[t + 1] - Lc.inst_ptr[t];
        H.coarse_off[t + 1] = H.coarse_off[t] + m * m;
    }
    for (size_t l = 1; l < H.lev.size(); ++l)
        for (int I = 0; I < H.lev[l].n; ++I)
            if (H.lev[l].diag[I] < 0) return "coarse row without a diagonal entry";
    build_tail(H);
    return "";
}

}  // namespace mhs
