// Aggregation multigrid hierarchy for the face system (host-side set-up).
//
// Aggregates are geometric: a face takes the mean of its two cells, and cells are
// grouped in blocks of their logical (i, j, k) indices, 2 or 1 cells along each direction depending on the coupling
// strength along it (semi-coarsening of anisotropic problems); every coarser
// level groups the blocks again.  The coarse operators are algebraic,
// A_{l+1} = P' A_l P with that averaging P from the faces and the
// piecewise-constant P of the aggregates below (smoothed on one transfer).  Their sparsity and, for every coarse entry,
// the list of finer entries that sum into it are built here once per
// structure, so that each solve forms the Galerkin products with a pure gather.
#pragma once

#include <array>
#include <cstddef>
#include <cstdint>
#include <string>
#include <vector>

#include "mhs_structure.h"

namespace mhs {

constexpr int kMaxCoarsest = 64;  // largest coarsest system per instance (dense inverse)

// Ends of the gather lists.  Positions in the lists fit 31 bits, but a list is
// longer than the array it gathers from: a face between two blocks is in both
// blocks' lists, so A P's hold up to twice the face matrix's entries (which
// stay below 2^31), level 1's about 1.6 times and level 2's pairs 1.5 times.
// kMaxList leaves room below 2^32 for the widest step of the kernels' loops.
using ListEnd = uint32_t;
constexpr size_t kMaxList = 0xffff0000u;

struct AmgLevel {
    int n = 0;                      // rows (all instances, unpadded)
    std::vector<int> inst_ptr;      // [ninst+1] first row of each instance
    std::vector<int> dims;          // [3 * ninst] block dimensions per instance
    std::vector<int> row_ptr, col;  // CSR pattern (columns sorted)
    std::vector<int> diag;          // position of the diagonal in each row
    std::vector<ListEnd> src_ptr;   // [nnz+1] gather list ranges
    std::vector<int> src;           // positions in the finer level's value array (level 1, ~pos: half of it)
    std::vector<int> agg;           // [n_finer] row of this level each finer row feeds (-1: none)
    // level 1: second aggregate of a face between two blocks (-1: the face lies
    // inside one block); the transfer gives such a face the mean of both
    std::vector<int> agg2;
    std::vector<int> child_ptr;     // [n+1]
    std::vector<int> child;         // finer rows of each row (level 1: ~f for a face with two aggregates)
    // Levels built by smoothed aggregation take their values as sums of
    // products over pairs (P position, T position) of the finer level's
    // transfer: src holds the P positions, src2 the T positions.
    bool sa_in = false;
    std::vector<int> src2;
    // Smoothed-aggregation transfer to the next coarser level (when sa_out):
    // P = (I - w_p D^-1 A) P_t with the tentative aggregates agg of the next
    // level, T = A P, and P transposed for the restriction.
    bool sa_out = false;
    std::vector<int> p_ptr, p_col, p_own;      // P rows; p_own[i]: entry of row i in its own aggregate
    std::vector<ListEnd> p_src_ptr;
    std::vector<int> p_src;                    // per P entry: positions of this level's values
    std::vector<int> pt_ptr, pt_col, pt_map;   // rows of the coarser level: fine row, P position
    std::vector<int> p_tpos;                   // per P entry: its position in the P' rows (inverse of pt_map)
    std::vector<int> t_ptr, t_col;             // T = A P
    std::vector<ListEnd> t_pair_ptr;
    std::vector<int> t_pa, t_pb;               // per T entry: (value position, P position)
    std::vector<int> t_p;                      // per T entry: the P entry of the same row and column, or -1
};

// A P with the level-1 aggregates: the fine-row by aggregate matrix of the
// post-smoothing sweep, (A P)_{iJ} = sum of a_ij P_jJ over the columns j that
// touch aggregate J (P_jJ 1, or 1/2 for a face between two).  Stored in the SELL-64 layout of the face matrix (lane-major
// slices; padding slots have column 0 and value 0), with, for every slot, the
// list of face-matrix positions that sum into it.
struct ApPattern {
    std::vector<long long> slice_ptr;  // [nslices+1]
    std::vector<int> col;              // level-1 row of each slot
    std::vector<ListEnd> src_ptr;      // [slots+1]
    std::vector<int> src;              // face-matrix SELL positions (~pos: half the entry)
    std::vector<int> slice;            // [slots/64] slice of each group of 64 slots
};

// The small levels of one V-cycle as the one-workgroup tail kernel reads them
// (k_vcycle_tail): per instance one block of 16-bit indices and one block of
// values, each ordered from the coarsest level to finer ones, so that a tail
// starting at level lt copies a prefix of both into LDS.  The index block is
// static; the values are gathered into theirs once per solve.
enum {
    TL_R0 = 0, TL_N,                   // first row, rows of the instance on this level
    TL_E0, TL_NNZ,                     // entries of those rows in the level's matrix
    TL_RP, TL_COL,                     // index block: local row pointers and columns
    TL_CP, TL_CH, TL_AGG,              // tentative transfer to the next level: children, aggregates
    TL_PTP, TL_PTC, TL_TP, TL_TC,      // smoothed transfer: rows of P' and of M
    TL_PT0, TL_NPT, TL_T0, TL_NT,      // their entries in the level's arrays
    TL_VAL, TL_WD, TL_PTV, TL_MV,      // value block: matrix, w D^-1, P', M (coarsest: the dense inverse)
    TL_VEC,                            // vectors: b, x, res (coarsest: b, x), in rows
    TL_IEND, TL_VEND,                  // lengths of the prefixes that include this level
    TL_K
};                                     // (row 0 of an instance: offsets of its blocks in TL_R0, TL_N)
struct TailLayout {
    int first = 0;                     // finest level the blocks hold
    std::vector<int> tab;              // [ninst][nlev][TL_K]
    std::vector<uint16_t> idx;
    long long nval = 0;                // values over all instances
    std::vector<int> iend, vend, vec;  // per level: longest prefixes and most vector rows of an instance
};
constexpr int kTailBytes = 152 * 1024; // LDS the tail may take

struct AmgHierarchy {
    std::vector<AmgLevel> lev;      // lev[0] unused placeholder, lev[1..] coarse levels
    std::vector<std::array<int, 3>> blocks;  // logical block factors of each transfer (l -> l+1)
    std::vector<int> coarse_off;    // [ninst+1] offsets of the dense coarsest inverses
    ApPattern ap;
    TailLayout tail;
    int nlev() const { return int(lev.size()); }
};

// Coupling strength along the three logical directions, e.g. the mean
// two-point transmissibility of the faces between logical neighbours.  The
// aggregates of every transfer are blocks of the finer level's logical grid,
// 2 or 1 cells along each direction: a direction is coarsened when its
// strength is at least half the strongest (a quarter below level 1), and the
// strengths then scale like those of the coarse blocks (cross-section over
// length).  Directions of extent 1 in every instance are never coarsened.
using Strength = std::array<double, 3>;

// Block factors of each transfer for these strengths and per-instance
// logical dimensions dims[3 * ninst], until every instance has at most
// kMaxCoarsest rows.
std::vector<std::array<int, 3>> coarsening_plan(const Strength &strength, const std::vector<int> &dims);

// Logical dimensions of every instance from ijk[3*nc] (instance-local,
// 0-based).  Returns an empty string on success.
std::string instance_dims(const Topology &T, const std::vector<int> &ijk, std::vector<int> &dims);

// Builds the hierarchy from logical cell indices ijk[3*nc] (instance-local,
// 0-based) with the blocks of coarsening_plan.  The transfer from the face
// matrix to level 1 is the tentative (piecewise-constant) one; with smoothed
// = true one coarse transfer is smoothed (the first from a level with at most
// an eighth as many rows as faces), the others stay tentative.  Returns an
// empty string on success.  A grid whose lists would pass max_list entries is
// refused.
std::string build_amg(AmgHierarchy &H, const Topology &T, const std::vector<int> &ijk,
                      const Strength &strength = {1.0, 1.0, 1.0}, bool smoothed = true,
                      size_t max_list = kMaxList);

}  // namespace mhs
