// Plan of the one-workgroup-per-system kernels (sys_kernels.hip): a system
// small enough that its factors, the fronts being factored and the network's
// state fit one workgroup's LDS is factored, solved and stepped by one
// workgroup per scenario.
//
// LDS layout of the factors (elements of the front type, per front p of fs
// rows and K pivots, uc = fs - K, us = fs | 1, ls = K | 1):
//   fo + i * us + j                     pivot rows (i < K, j < fs): L11\U11, U12
//   fo + K * us + (i - K) * ls + j      rows below (i >= K, j < K): L21
// and in the scratch region, live from the front's level to its parent's:
//   co + (i - K) * uc + (j - K)         contribution block
// The odd strides keep a wave's accesses down a column free of bank conflicts.
// The solve sweeps reuse the scratch region for the fronts' work vectors
// (wo + position).
#pragma once

#include "analyze.hpp"

#include <cstddef>
#include <cstdint>
#include <vector>

namespace cupf {

// Contribution blocks are added by destination: a front's destinations are cut
// into slices of 16 (a lane each), a slice holding its destinations and then
// `width` rows of 16 sources, padded with the element that holds zero.  Every
// destination has one owner, so a front is assembled without a barrier between
// children and in a fixed order.

// One front, 32 bytes (the order the kernels read).
struct SysFront {
    int fo = 0, co = 0, wo = 0;
    int size = 0;        // fs | K << 16
    int first = 0;       // first pivot (permuted index); the pivots are consecutive
    int rows = 0;        // its positions in the row and gather lists
    int slice0 = 0, slices = 0;
};

// A slice: offset of its destinations in the add list in units of 16 | width
// << 20.
constexpr int kSysSliceShift = 20;

struct SysPlan {
    bool ok = false;                 // the pattern qualifies (sizes of the fields below)
    int n = 0, nnz = 0;
    int fac = 0, scratch = 0;        // elements: factors; contribution blocks / work vectors and the zero
    std::vector<int> blob;           // packed tables, copied to LDS as they are
    std::vector<uint16_t> adds;      // the slices' destinations and sources (element numbers)
    // offsets into the blob: ints for fronts, levels and slices, u16 elements for the lists
    int num_fronts = 0, num_levels = 0;
    int o_level = 0, o_slice = 0, o_task = 0, o_rows = 0, o_gptr = 0, o_gsrc = 0, o_perm = 0;
    std::vector<int> slot_pos;       // A value slot -> factor element
};

// Levels: per level four ints {first task, quads, wave fronts, shared fronts}; tasks
// (u16 front ids, in the order wave fronts, quads, shared fronts): a quad is four
// fronts of at most 16 rows, one per 16 lanes of a wave (0xffff: none); a wave
// front is one wave's, a shared front the whole workgroup's.
constexpr int kSysLevelInts = 4;
constexpr int kSysSmallRows = 16;
// largest front (the shared fronts' register tiles)
constexpr int kSysMaxRows = 112;

// Panel cap of the one-workgroup plan, whatever the caller's (which shapes the
// level sweeps): a workgroup eliminates a front pivot by pivot at any width, so
// narrow panels only add levels and assemblies (118 buses: 9 levels at 8, 5 at
// 64).
constexpr int kSysCap = 64;

// most_elems: elements (factors and scratch) that may fit the LDS at all.
SysPlan make_sys_plan(const LuPlan& P, size_t most_elems);

// The one-workgroup plan (ok false: the system does not qualify) of the pattern
// rp/ci, whose analysis and plan at the caller's cap are sym and P.
SysPlan find_sys_plan(const LuPlan& P, const Symbolic& sym, const int* rp, const int* ci, size_t most_elems);

}  // namespace cupf
