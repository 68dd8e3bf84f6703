// Host-side list building for the multigrid set-up: contiguous ranges of rows on
// several threads, their lists appended in order.
#pragma once

#include <algorithm>
#include <exception>
#include <thread>
#include <utility>
#include <vector>

#include "mhs_amg.h"

namespace mhs {

// Host threads for the row loops below (each row's lists depend on that row
// alone): fn(t, begin, end) on contiguous ranges of [0, n), at least `least`
// items each.  The hierarchy of 128x128x64 cells is 100M list entries.
constexpr int kMaxThreads = 8;
inline int ranges(int n, int least) {
    const int hw = std::max(1u, std::thread::hardware_concurrency());
    return std::max(1, std::min({n / std::max(1, least), hw, kMaxThreads}));
}
template <class Fn>
void in_ranges(int n, int nt, Fn fn) {
    std::vector<std::exception_ptr> err(nt);
    auto run = [&](int t) {
        try {
            fn(t, int((long long)n * t / nt), int((long long)n * (t + 1) / nt));
        } catch (...) {
            err[t] = std::current_exception();
        }
    };
    std::vector<std::thread> pool;
    pool.reserve(nt);
    int t = 1;
    try {
        for (; t < nt; ++t) pool.emplace_back(run, t);
    } catch (...) {   // no more threads to be had: the rest runs here
    }
    run(0);
    for (int u = t; u < nt; ++u) run(u);
    for (auto &th : pool) th.join();
    for (auto &e : err)
        if (e) std::rethrow_exception(e);
}
// Appends the ranges' lists in order; returns where each one starts.
template <class I>
std::vector<size_t> append(std::vector<I> &out, const std::vector<std::vector<I>> &parts) {
    std::vector<size_t> at(parts.size() + 1, out.size());
    for (size_t t = 0; t < parts.size(); ++t) at[t + 1] = at[t] + parts[t].size();
    out.resize(at.back());
    in_ranges(int(parts.size()), int(parts.size()), [&](int, int b, int e) {
        for (int t = b; t < e; ++t) std::copy(parts[t].begin(), parts[t].end(), out.begin() + at[t]);
    });
    return at;
}

inline size_t total(const std::vector<std::vector<int>> &parts) {
    size_t n = 0;
    for (const auto &p : parts) n += p.size();
    return n;
}
// What the lists of one pattern may hold: positions of its entries are 32-bit
// signed (~pos marks a half entry), the ends of its lists 32-bit unsigned.
inline bool too_long(size_t entries, size_t list, size_t max_list) {
    return entries > std::min<size_t>(max_list, 0x7fffffff) || list > std::min(max_list, kMaxList);
}

// A row's entries by column: columns ascending, each one's entries in the order
// they were put.  A place per column instead of a sort: a row of a triple product
// has some hundred entries in a few dozen columns, and sorting them took half of
// the hierarchy's time (128x128x64 with 2x2x1 blocks: 2.3 -> 1.7 s on 8 threads,
// 7.9 -> 4.4 s on one; 20x20x10: 22 -> 9 ms, 9^3: 4.9 -> 2.2 ms).
template <class E>
class ByColumn {
    struct Col {
        int col, n, at;
    };
    std::vector<int> place_;   // of a column in cols_, where cols_ holds that column there
    std::vector<Col> cols_;
    std::vector<std::pair<int, E>> in_;
    std::vector<std::pair<int, int>> order_;
    std::vector<E> out_;

public:
    explicit ByColumn(int ncols) : place_(ncols, 0) {}
    void start() {
        cols_.clear();
        in_.clear();
    }
    void put(int col, const E &e) {
        int &p = place_[col];
        if ((size_t)p >= cols_.size() || cols_[p].col != col) {
            p = (int)cols_.size();
            cols_.push_back({col, 0, 0});
        }
        ++cols_[p].n;
        in_.emplace_back(p, e);
    }
    // each(column, entries, how many)
    template <class Fn>
    void finish(Fn each) {
        order_.clear();
        for (size_t p = 0; p < cols_.size(); ++p) order_.emplace_back(cols_[p].col, (int)p);
        std::sort(order_.begin(), order_.end());
        int at = 0;
        for (const auto &o : order_) {
            cols_[o.second].at = at;
            at += cols_[o.second].n;
        }
        out_.resize(in_.size());
        for (const auto &i : in_) out_[cols_[i.first].at++] = i.second;
        for (const auto &o : order_) {
            const Col &c = cols_[o.second];
            each(c.col, out_.data() + (c.at - c.n), c.n);
        }
    }
};

// Rows of a CSR pattern whose entries each carry a list, built range by range, each
// range with a row = make() of its own: row(i, R) appends the row's columns to R.col and, per entry, its sources to
// R.src (and R.src2) and their end to R.end.  False: too long.
struct RowPart {
    std::vector<int> col, src, src2, len;
    std::vector<ListEnd> end;
};
template <class Make>
bool build_rows(int n, std::vector<int> &ptr, std::vector<int> &col, std::vector<ListEnd> &src_ptr,
                std::vector<int> &src, std::vector<int> *src2, size_t max_list, Make make) {
    const int nt = ranges(n, 2048);
    std::vector<RowPart> P(nt);
    in_ranges(n, nt, [&](int t, int b, int e) {
        RowPart &R = P[t];
        auto row = make();
        R.len.reserve(e - b);
        for (int i = b; i < e; ++i) {
            const size_t c0 = R.col.size();
            row(i, R);
            R.len.push_back(int(R.col.size() - c0));
        }
    });
    std::vector<std::vector<int>> cols(nt), srcs(nt), srcs2(nt);
    std::vector<std::vector<ListEnd>> ends(nt);
    for (int t = 0; t < nt; ++t) {
        cols[t].swap(P[t].col);
        srcs[t].swap(P[t].src);
        srcs2[t].swap(P[t].src2);
        ends[t].swap(P[t].end);
    }
    if (too_long(total(cols), total(srcs), max_list)) return false;
    ptr.assign(n + 1, 0);
    for (int t = 0, i = 0; t < nt; ++t)
        for (int l : P[t].len) {
            ptr[i + 1] = ptr[i] + l;
            ++i;
        }
    col.clear();
    src.clear();
    append(col, cols);
    const std::vector<size_t> at = append(src, srcs);
    for (int t = 0; t < nt; ++t)
        for (ListEnd &e : ends[t]) e += ListEnd(at[t]);
    src_ptr.assign(1, 0);
    append(src_ptr, ends);
    if (src2) {
        src2->clear();
        append(*src2, srcs2);
    }
    return true;
}

}  // namespace mhs
