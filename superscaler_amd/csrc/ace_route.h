// Which kernel scores a batch: the rule of launch_score, as host code that the CPU tests walk as it is.
#pragma once
#include <algorithm>

#include "ace_many.h"

// The first five defer the evaluation of stage tails to records in a workspace.
enum AceKernelId { ACE_K_SPREAD, ACE_K_DUO, ACE_K_DENSE, ACE_K_MANY, ACE_K_DEFERRED, ACE_K_IN_PLACE };

struct AceRouteTables {         // what a handle's tables allow
    int32_t ops;
    bool spread;                // the kernel of small batches (its position table was made)
    bool dense;                 // the dense tables
    int32_t dense_windows;      // ... windows of their rows (0: resident)
    int32_t dense_lanes;        // ... lanes of a workgroup of large batches
    bool many;                  // the assembly loop over the table compiler's rows
    int32_t windows;            // ... windows of those (1: resident)
    bool deferred;              // the C++ loop with deferred stage tails
};

// Up to this many plans a batch takes the kernel of small batches.  Its time grows with the number of plans once every CU has six workgroups
// (1,536 plans); that of the others, where a lane or a few walk a plan, hardly does until the chip is full, and they cross
// where that time is reached.  That place depends on the graph: both times grow with the ops, but not alike.  A path has one
// limit or one line in the ops, at or below the first crossing of the graphs measured for it (or within 3 % of its time), so a graph that crosses later has a jump
// there.  By what else would take the batch, in us per launch at the limit and where the graph crosses (plan per workgroup / the other):
//   PLAIN    the mid-sized kernel                    limit  4,096: 315 ops  31 / 32, crosses at  4,400 plans; 523 ops  45 /  51,  4,850;
//                                                                  821 ops  56 / 67,  5,000; 1,251 ops  82 /  79,  3,950; 134 ops  18 / 21, 5,250
//   WINDOWED large, windowed rows (dense tables)     6,000 and 4 per op: 118 ops  26 / 30, crosses at 7,700 plans; 134 ops 28 / 32, 7,450 to 8,850 by what is in
//            the windows; 182 ops 32 / 38, 8,450; 230 ops 36 / 44, 8,600; 270 ops 46 / 48, 7,500; 315 ops 48 / 48, 7,300; 523 ops 80 / 93, 9,700; 1,251 ops 195 / 210, 11,900
//   ROWS     large, the table compiler's rows        limit  8,800: windows 118 ops  33 / 41, crosses at 11,400 plans; 134 ops 35 / 44, 11,500; 230 ops 43 / 62, 12,900;
//                                                                  315 ops  57 / 86, 13,450; 523 ops 87 / 151, 16,450; 821 ops in two windows 107 / 120, 9,900; 1,251 ops
//                                                                  161 / 341, 19,700; resident 118 ops 32 / 32, 8,800; 134 ops 33 / 35, 9,050 to 9,450
//   ... and both of these at most 1,500, 48 per op and 700 per window, for short graphs: 38 ops in two windows cross at 4,730 over dense tables and at 4,860
//            over the others, in five at 7,050
//   SLOW     no assembly loop (memory of collectives, more than 256 rows)
//                                                    limit 18,432: 315 ops 134 / 163, 22,300; 523 ops 197 / 456, above 32,768; 134 ops  87 / 140, 30,200
//   RECORDS  stage records                           limit 14,336: 315 ops 134 / 136, 14,500; 523 ops 199 / 316, 23,000; 134 ops 81 / 148, above 24,576
//            single-stage queries                           14,336: 315 ops  85 / 103, 18,000; 523 ops 80 / 179, 134 ops 53 / 124, both above 24,576
//   DEFERRED the C++ loop, rows resident or in windows that no assembly loop fetches
//                                                    100 per op, 2,500 per window after the first, 4,096 to 16,384: resident 118 ops 42 / 56, crosses at 16,700; 134 ops
//                                                                  48 / 62, 17,450; windows 16 ops  14 / 24, 9,000; 29 ops 30 / 41, 15,100; 55 ops 48 / 73, 25,750; 134 ops 57 / 68,
//                                                                  19,000; 107 ops  56 / 131, 315 ops 102 / 352, 1,251 ops 286 / 1,442, all above 32,768
// and at one plan 8 to 26 where a lane needs 49 to 169 (13 to 20 us is what the host needs for a launch).
constexpr int kSpreadMaxPlain = 4096, kSpreadMaxRows = 8800, kSpreadMaxSlow = 18432, kSpreadMaxRecords = 14336;
inline long long ace_spread_max_windowed(long long ops) { return 6000 + 4 * ops; }
inline long long ace_spread_max_deferred(long long ops, long long windows) { return std::min(16384ll, std::max(4096ll, 100 * ops + 2500 * (windows - 1))); }
inline long long ace_spread_max_short(long long ops, long long windows) { return 1500 + 48 * ops + 700 * windows; }

// Workgroups of large batches over dense tables: slices of 64 plans each, and how many of them.
struct AceShares { uint32_t slices; size_t groups; };
inline AceShares ace_dense_shares(const AceRouteTables &t, long long plans) {
    const uint32_t slices = ace_dense_slices(plans, t.dense_lanes / 64, 256 * (kDenseWinLanes / t.dense_lanes));
    return {slices, ((size_t)plans + 64u * slices - 1) / (64u * slices)};
}
inline AceShares ace_many_shares(long long plans) {
    const uint32_t slices = ace_many_slices(plans);
    return {slices, ((size_t)plans + 64u * slices - 1) / (64u * slices)};
}

constexpr size_t kWsPlan = (size_t)ACE_MAX_STAGES * ACE_WS_REC * sizeof(double);    // workspace bytes per plan of all kernels but the dense one (kDensePlan)

// Bytes of workspace that plain scoring of so many plans asks for (0: none), at most kWsMost.  The dense tables' records are the larger
// ones: a batch that fits only without them goes over the table compiler's rows, one that does not fit either way has its stage tails
// evaluated where they end.
constexpr size_t kWsMost = 64ull << 30;
// (a block more than the plans: the kernels of large batches round the share of every CU up)
inline size_t ace_workspace_plans(long long plans) { return ((size_t)plans + 1023) / 1024 * 1024 + 1024; }
inline size_t ace_workspace(const AceRouteTables &t, long long plans) {
    const size_t rounded = ace_workspace_plans(plans);
    if (t.dense && rounded * kDensePlan <= kWsMost) return rounded * kDensePlan;
    return t.deferred && rounded * kWsPlan <= kWsMost ? rounded * kWsPlan : 0;
}

// `records`: stage records or single-stage queries; `workspace`: how many bytes of it there are.
inline AceKernelId ace_route(const AceRouteTables &t, long long plans, bool records, size_t workspace) {
    const bool plain = !records && workspace != 0;
    const int L = plain && t.dense && t.dense_windows == 0 ? ace_duo_lanes(plans) : 0;
    AceKernelId other = ACE_K_IN_PLACE;
    if (L && (size_t)((plans + L - 1) / L) * (size_t)L * kWsPlan <= workspace) other = ACE_K_DUO;
    else if (plain && t.dense && ace_dense_shares(t, plans).groups * ace_dense_shares(t, plans).slices * kDenseWave <= workspace) other = ACE_K_DENSE;
    else if (plain && t.many && ace_many_shares(plans).groups * ace_many_shares(plans).slices * 64u * kWsPlan <= workspace) other = ACE_K_MANY;
    else if (plain && t.deferred && (size_t)(plans + 1023) / 1024 * 1024 * kWsPlan <= workspace) other = ACE_K_DEFERRED;
    const long long most = records ? kSpreadMaxRecords : other == ACE_K_DUO ? kSpreadMaxPlain : other == ACE_K_IN_PLACE ? kSpreadMaxSlow :
                           other == ACE_K_DENSE ? std::min(ace_spread_max_windowed(t.ops), ace_spread_max_short(t.ops, t.dense_windows)) :
                           other == ACE_K_DEFERRED ? ace_spread_max_deferred(t.ops, t.windows) :
                           std::min((long long)kSpreadMaxRows, ace_spread_max_short(t.ops, t.windows));
    return t.spread && plans <= most ? ACE_K_SPREAD : other;
}
