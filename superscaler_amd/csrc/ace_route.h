// Which kernel scores a batch: the rule of launch_score, as host code that the CPU tests walk as it is.
#pragma once
#include "ace_many.h"

// The first five defer the evaluation of stage tails to records in a workspace.
enum AceKernelId { ACE_K_SPREAD, ACE_K_DUO, ACE_K_DENSE, ACE_K_MANY, ACE_K_DEFERRED, ACE_K_IN_PLACE };

struct AceRouteTables {         // what a handle's tables allow
    int32_t ops;
    bool spread;                // the kernel of small batches (its position table was made)
    bool dense, dense_windows;  // the dense tables; their rows in windows
    int32_t dense_lanes;        // ... of a workgroup of large batches
    bool many, many_windows;    // the assembly loop over the table compiler's rows; those in windows
    bool deferred;              // the C++ loop with deferred stage tails
};

// Up to this many plans a batch takes the kernel of small batches.  Its time grows with the number of plans once every CU has six workgroups
// (1,536 plans); that of the others, where a lane or a few walk a plan, hardly does until the chip is full, and they cross
// where that time is reached.  That place depends on the graph: both times grow with the ops, but not alike.  A path has one
// limit all the same, at or below the first crossing of the graphs measured for it, so a graph that crosses later has a jump
// there.  By what else would take the batch, in us per launch at the limit and where the graph crosses (plan per workgroup / the other):
//   PLAIN    the mid-sized kernel                    limit  4,096: 315 ops  30 / 32, crosses at  4,300 plans; 523 ops  44 /  50,  4,650;
//                                                                  821 ops  56 / 67,  5,000; 1,251 ops  82 /  81,  4,050
//   WINDOWED large, windowed rows (dense tables)     limit  6,144: 118 ops  29 / 30, crosses at  6,700 plans; 134 ops 31 / 33, 6,600; 182 ops 35 / 39, 7,150;
//                                                                  230 ops  40 / 44, 7,050; 270 ops 48 / 49, 6,150
//   SLOW     no assembly loop (memory of collectives, more than 256 rows)
//                                                    limit 18,432: 315 ops 161 / 161, 18,400; 523 ops 238 / 459, above 24,576 (313 / 460);
//                                                                  134 ops  97 / 140, above 24,576 (128 / 140)
//   RECORDS  stage records                           limit 14,336: 315 ops 134 / 136, 14,500; 523 ops 199 / 316, 23,000; 134 ops 81 / 148, above 24,576
//            single-stage queries                           14,336: 315 ops  85 / 103, 18,000; 523 ops 80 / 179, 134 ops 53 / 124, both above 24,576
//   OTHER    the C++ loop with deferred stage tails  limit  4,096:  62 ops  18 / 41, 11,500; 134 ops  22 / 83, 20,000
// and at one plan 8 to 26 where a lane needs 49 to 169 (13 to 20 us is what the host needs for a launch).
constexpr int kSpreadMaxPlain = 4096, kSpreadMaxWindowed = 6144, kSpreadMaxSlow = 18432, kSpreadMaxRecords = 14336;
constexpr int kSpreadMaxOther = 4096;    // (tables that no assembly loop walks)

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
    const int L = plain && t.dense && !t.dense_windows ? ace_duo_lanes(plans) : 0;
    AceKernelId other = ACE_K_IN_PLACE;
    if (L && (size_t)((plans + L - 1) / L) * (size_t)L * kWsPlan <= workspace) other = ACE_K_DUO;
    else if (plain && t.dense && ace_dense_shares(t, plans).groups * ace_dense_shares(t, plans).slices * kDenseWave <= workspace) other = ACE_K_DENSE;
    else if (plain && t.many && ace_many_shares(plans).groups * ace_many_shares(plans).slices * 64u * kWsPlan <= workspace) other = ACE_K_MANY;
    else if (plain && t.deferred && (size_t)(plans + 1023) / 1024 * 1024 * kWsPlan <= workspace) other = ACE_K_DEFERRED;
    const int most = records ? kSpreadMaxRecords : other == ACE_K_DUO ? kSpreadMaxPlain : other == ACE_K_IN_PLACE ? kSpreadMaxSlow :
                     other == ACE_K_DENSE || (other == ACE_K_MANY && t.many_windows) ? kSpreadMaxWindowed : kSpreadMaxOther;
    return t.spread && plans <= most ? ACE_K_SPREAD : other;
}
