// Workgroup ids by XCD.
#pragma once

#include <hip/hip_runtime.h>

/// Consecutive workgroups of a grid of `total` go to the 8 XCDs in turn, each
/// with an L2 of its own. The workgroup's place where every XCD has a
/// contiguous share of 0 .. total - 1 (the first total % 8 one more).
__device__ __forceinline__ int xcdShare(int id, int total) {
    const int xcd = id % 8, each = total / 8;
    return xcd * each + min(xcd, total % 8) + id / 8;
}
