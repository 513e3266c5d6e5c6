// Launches of as many workgroups as a batch needs.  A grid's size in work items is a 32-bit number, and a larger grid may run cut
// short without an error; kernels with several lanes per plan reach that long before a batch's own limit (2^31 - 1 plans).
#pragma once
#include <cstdint>

constexpr uint64_t kMaxWorkItems = 1ull << 31;

// f(first workgroup, workgroups) for the parts of a grid of `groups` workgroups of `lanes` lanes, in order.
template <class F> void ace_grid_parts(uint64_t groups, uint32_t lanes, F f) {
    const uint64_t most = kMaxWorkItems / lanes;
    for (uint64_t at = 0; at < groups; at += most) f(at, (uint32_t)(groups - at < most ? groups - at : most));
}
