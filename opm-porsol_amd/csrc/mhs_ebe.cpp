// Element-by-element layout of the level-0 face operator.  See mhs_ebe.h.
#include "mhs_ebe.h"

#include "mhs_kernels.h"
#include "mhs_lists.h"

#include <algorithm>
#include <numeric>

namespace mhs {

int greedy_colours(int nc, const int *facepos, const int *nb, std::vector<int> &colour, const int *ijk) {
    if (ijk) {
        colour.assign(nc, 0);
        for (int c = 0; c < nc; ++c) colour[c] = (ijk[3 * (size_t)c] + ijk[3 * (size_t)c + 1] + ijk[3 * (size_t)c + 2]) & 1;
        int ncol = nc > 0 ? 1 : 0;
        for (int c = 0; c < nc; ++c) {
            bool clash = false;
            unsigned long long used = 0;
            for (int h = facepos[c]; h < facepos[c + 1]; ++h) {
                const int o = nb[h];
                if (o < 0) continue;
                if (o < c && colour[o] == colour[c]) clash = true;
                if (colour[o] < 64) used |= 1ull << colour[o];
            }
            if (clash) {
                int k = 2;
                while (k < 64 && (used & (1ull << k))) ++k;
                colour[c] = k;
            }
            ncol = std::max(ncol, colour[c] + 1);
        }
        return ncol;
    }
    colour.assign(nc, -1);
    int ncol = 0;
    for (int c = 0; c < nc; ++c) {
        unsigned long long used = 0;
        for (int h = facepos[c]; h < facepos[c + 1]; ++h) {
            const int o = nb[h];
            if (o >= 0 && colour[o] >= 0 && colour[o] < 64) used |= 1ull << colour[o];
        }
        int k = 0;
        while (k < 64 && (used & (1ull << k))) ++k;
        colour[c] = k;
        ncol = std::max(ncol, k + 1);
    }
    return ncol;
}

std::string ebe_ap_lists(const EbeLayout &E, const Topology &T, const ApPattern &ap, const std::vector<int> &agg,
                         const std::vector<int> &agg2, std::vector<ListEnd> &ptr, std::vector<int> &src,
                         size_t max_list) {
    const long long slots = (long long)ap.col.size();
    if (slots >= 0x7fffffffLL || E.nval >= 0x7fffffffLL) return "too many values for 32-bit lists";
    // row by row (each row's slots depend on its own cells, in ascending order),
    // the lists in slot order
    const int ns = T.nslices, nt = ranges(ns, 32);
    struct Part {
        std::vector<int> src;
        std::vector<ListEnd> end;
        bool outside = false;
    };
    std::vector<Part> parts(nt);
    in_ranges(ns, nt, [&](int t, int b, int e) {
        Part &Q = parts[t];
        std::vector<std::pair<int, int>> in;   // (slot of the slice, position)
        std::vector<int> J, end;
        for (int sl = b; sl < e; ++sl) {
            const long long base = ap.slice_ptr[sl];
            const int w = int((ap.slice_ptr[sl + 1] - base) / kSlice);
            in.clear();
            end.assign((size_t)w * kSlice + 1, 0);
            for (int l = 0; l < kSlice; ++l) {
                const int f = sl * kSlice + l;
                if (agg[f] < 0) continue;
                // the row's aggregates (about 7; padding slots list nothing)
                J.clear();
                for (int q = 0; q < w; ++q) {
                    const long long at = base + l + (long long)q * kSlice;
                    if (ap.src_ptr[at + 1] > ap.src_ptr[at]) J.push_back(ap.col[at]);
                }
                for (int r = 0; r < 2; ++r) {
                    const int c = T.row_cell[2 * (size_t)f + r];
                    if (c < 0) continue;
                    const int f0 = T.facepos[c], n = T.facepos[c + 1] - f0, np = n * (n + 1) / 2;
                    const int i = T.row_loc[2 * (size_t)f + r], s = E.cell_seg[c], loc = E.cell_local[c];
                    for (int j = 0; j < n; ++j) {
                        const int rj = T.hf_dof[f0 + j];
                        const int v = int(E.seg_val[s] + ebe_slot(loc, i <= j ? pidx(i, j, n) : pidx(j, i, n), np));
                        for (int a : {agg[rj], agg2[rj]}) {
                            if (a < 0) continue;
                            const auto at = std::find(J.begin(), J.end(), a);
                            if (at == J.end()) {
                                Q.outside = true;
                                continue;
                            }
                            const int q = int(at - J.begin()) * kSlice + l;
                            in.emplace_back(q, agg2[rj] >= 0 ? ~v : v);
                            ++end[q + 1];
                        }
                    }
                }
            }
            const size_t s0 = Q.src.size();
            for (int q = 0; q < w * kSlice; ++q) end[q + 1] += end[q];
            Q.src.resize(s0 + in.size());
            for (const auto &x : in) Q.src[s0 + end[x.first]++] = x.second;
            // (each end has moved to where the next slot starts)
            for (int q = 0; q < w * kSlice; ++q) Q.end.push_back(ListEnd(s0 + end[q]));
        }
    });
    std::vector<std::vector<int>> srcs(nt);
    std::vector<std::vector<ListEnd>> ends(nt);
    for (int t = 0; t < nt; ++t) {
        if (parts[t].outside) return "a cell entry outside the A P pattern";
        srcs[t].swap(parts[t].src);
        ends[t].swap(parts[t].end);
    }
    if (too_long(0, total(srcs), max_list)) return "too many entries for 32-bit lists";
    src.clear();
    const std::vector<size_t> at = append(src, srcs);
    for (int t = 0; t < nt; ++t)
        for (ListEnd &e : ends[t]) e += ListEnd(at[t]);
    ptr.assign(1, 0);
    append(ptr, ends);
    return "";
}

std::string build_ebe(EbeLayout &E, const Topology &T, const int *ijk) {
    E = EbeLayout();
    if (T.has_periodic) return "periodic faces";
    if ((long long)T.nfp > (long long)kEbeRow) return "too many face rows";
    const int nc = T.nc;
    std::vector<int> colour;
    const int ncol = greedy_colours(nc, T.facepos.data(), T.nb.data(), colour, ijk);
    if (ncol > kMaxColours) return "more than 8 colours";
    // instance of every cell
    std::vector<int> inst(nc);
    for (int t = 0; t < T.ninst; ++t)
        for (int c = T.inst_cellpos[t]; c < T.inst_cellpos[t + 1]; ++c) inst[c] = t;
    // segments: cells sorted by (colour, hexahedron or not, instance, face
    // count, index), so that each colour's hexahedra form one block range
    // (launched with the 6-face kernel) followed by the other cells
    auto key = [&](int c) {
        const int n = T.facepos[c + 1] - T.facepos[c];
        return (((long long)colour[c] * 2 + (n == 6 ? 0 : 1)) * T.ninst + inst[c]) * (kMaxFaces + 1) + n;
    };
    std::vector<int> order(nc);
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return key(a) < key(b); });
    E.ncolours = ncol;
    E.colour_blk.assign(ncol + 1, 0);
    E.cell_seg.assign(nc, -1);
    E.cell_local.assign(nc, -1);
    std::vector<int> seg_colour;
    for (size_t i = 0; i < order.size();) {
        size_t j = i;
        const long long k = key(order[i]);
        while (j < order.size() && key(order[j]) == k) ++j;
        const int c0 = order[i];
        const int n = T.facepos[c0 + 1] - T.facepos[c0];
        const int count = (int)(j - i);
        const int len = (count + kEbeBlock - 1) / kEbeBlock * kEbeBlock;
        const int s = E.nseg++;
        E.seg_n.push_back(n);
        E.seg_inst.push_back(inst[c0]);
        E.seg_count.push_back(count);
        E.seg_len.push_back(len);
        E.seg_blk0.push_back(E.nblk);
        E.seg_val.push_back(E.nval);
        E.seg_dof.push_back(E.ndof);
        seg_colour.push_back(colour[c0]);
        for (int b = 0; b < len / kEbeBlock; ++b) E.blk_seg.push_back(s);
        E.nblk += len / kEbeBlock;
        E.nval += (long long)n * (n + 1) / 2 * len;
        E.ndof += (long long)n * len;
        for (size_t q = i; q < j; ++q) {
            E.cell_seg[order[q]] = s;
            E.cell_local[order[q]] = (int)(q - i);
        }
        i = j;
    }
    for (int k = 0, b = 0; k <= ncol; ++k) {
        while (b < E.nblk && seg_colour[E.blk_seg[b]] < k) ++b;
        E.colour_blk[k] = b;
    }
    E.colour_split.assign(ncol, 0);
    for (int k = 0; k < ncol; ++k) {
        int b = E.colour_blk[k];
        while (b < E.colour_blk[k + 1] && E.seg_n[E.blk_seg[b]] == 6) ++b;
        E.colour_split[k] = b;
    }
    // face rows with the first/last-writer flags, in the 64-cell tiles of the values
    E.dof.assign((size_t)E.ndof, 0u);
    for (int c = 0; c < nc; ++c) {
        const int s = E.cell_seg[c], l = E.cell_local[c];
        const int f0 = T.facepos[c], n = T.facepos[c + 1] - f0;
        for (int j = 0; j < n; ++j) {
            const int h = f0 + j, o = T.nb[h];
            uint32_t d = (uint32_t)T.hf_dof[h];
            if (o < 0 || colour[c] < colour[o]) d |= kEbeFirst;
            if (o < 0 || colour[c] > colour[o]) d |= kEbeLast;
            E.dof[(size_t)E.seg_dof[s] + (size_t)ebe_slot(l, j, n)] = d;
        }
    }
    // partial-sum slots: each instance's blocks (over all colours) contiguous
    std::vector<int> per_inst(T.ninst + 1, 0);
    for (int b = 0; b < E.nblk; ++b) ++per_inst[E.seg_inst[E.blk_seg[b]] + 1];
    E.inst_slot.assign(T.ninst + 1, 0);
    for (int t = 0; t < T.ninst; ++t) E.inst_slot[t + 1] = E.inst_slot[t] + per_inst[t + 1];
    std::vector<int> next(E.inst_slot.begin(), E.inst_slot.end() - 1);
    E.blk_slot.resize(E.nblk);
    for (int b = 0; b < E.nblk; ++b) E.blk_slot[b] = next[E.seg_inst[E.blk_seg[b]]]++;
    E.nslots = E.nblk;
    E.blk_info.resize(4 * (size_t)E.nblk);
    E.blk_base.resize(2 * (size_t)E.nblk);
    for (int b = 0; b < E.nblk; ++b) {
        const int s = E.blk_seg[b], n = E.seg_n[s], local0 = (b - E.seg_blk0[s]) * kEbeBlock;
        E.blk_info[4 * b] = n;
        E.blk_info[4 * b + 1] = E.seg_inst[s];
        E.blk_info[4 * b + 2] = std::min(kEbeBlock, E.seg_count[s] - local0);
        E.blk_info[4 * b + 3] = E.blk_slot[b];
        E.blk_base[2 * b] = E.seg_val[s] + ebe_slot(local0, 0, n * (n + 1) / 2);
        E.blk_base[2 * b + 1] = E.seg_dof[s] + ebe_slot(local0, 0, n);
    }
    return "";
}

}  // namespace mhs
