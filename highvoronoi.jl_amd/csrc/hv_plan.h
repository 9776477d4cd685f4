// hv_plan.h -- sizes the walk plans its launches with: plain C++ without device code, so that a host
// program can go through them.
#pragma once
#include <stdint.h>
#include <algorithm>

// The buckets a level's nr rays are counted into (k_tent_group): position p of the n generators' gaps,
// HV_BUCKET_SUB positions a gap, lies in bucket (p >> shift) + m of mesh m, whose positions start at
// (goff[m] + m) HV_BUCKET_SUB.  As many as two a ray, at least 2048 and at most 2^21 (8 MiB of
// counts), and one more a mesh: the meshes' own are outside the limit, which no shift could meet
// with more meshes than that.
constexpr int HV_BUCKET_SUB = 16;
struct HvBuckets {
    int shift, count;   // bucket count - 1 is empty: its offset is the number of rays placed
};
inline HvBuckets hv_buckets(int64_t n, int64_t nmesh, int64_t nr) {
    const int64_t positions = (n + nmesh) * HV_BUCKET_SUB;
    const int64_t limit = std::max<int64_t>(2048, std::min<int64_t>(2 * nr, 1 << 21));
    int shift = 0;
    while ((positions >> shift) > limit) ++shift;
    return {shift, (int)((positions >> shift) + nmesh + 1)};
}

// Levels of internal nodes of the 8-ary tree, and k_knn's waiting nodes.  A tree has at most 2^29
// leaves (leaves of one point; node numbers of the binary tree are 32-bit), so at most ten levels.
// A step takes the topmost eight nodes, of whatever levels, and puts their internal children, at
// most 64, in their place.  A node of level l then never waits above position 63 l: the root waits at
// 0, and a child of a taken node of level l lands at most 63 above the lowest taken position, which
// is no higher than that node's own.
constexpr int HV_TREE_LEVELS = 10;
constexpr int HV_KNN_STACK = 576;
static_assert(HV_KNN_STACK > 63 * (HV_TREE_LEVELS - 1), "room for the deepest node's highest position");
