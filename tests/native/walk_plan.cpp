// Host checks of hv_plan.h: exit status 0 when every one holds.
#include "hv_plan.h"
#include <cstdio>
#include <random>
#include <vector>

// hv_buckets over k meshes of n generators each and a level of nr rays: the shift is one a 64-bit
// number can be shifted by, and the meshes' buckets are disjoint, ascending and below the empty one
static int buckets(int64_t k, int64_t n, int64_t nr) {
    const HvBuckets b = hv_buckets(k * n, k, nr);
    if (b.shift < 0 || b.shift > 62 || b.count < k + 1) return 1;
    if ((int64_t)b.count > (1 << 21) + k + 1) return 2;
    int64_t last = -1;
    for (int64_t m = 0; m < k; ++m) {
        const int64_t first = (m * n + m) * HV_BUCKET_SUB;                        // position of the gap before generator 0
        const int64_t end = (m * n + m + n) * HV_BUCKET_SUB + HV_BUCKET_SUB - 1;   // last of the gap behind the last one
        const int64_t lo = (first >> b.shift) + m, hi = (end >> b.shift) + m;
        if (lo <= last || hi < lo) return 3;
        last = hi;
    }
    const int64_t past = ((k * n + k) * HV_BUCKET_SUB >> b.shift) + k;   // where the packets' plan ends
    return last < b.count - 1 && past == b.count - 1 ? 0 : 4;
}

// the steps of k_knn over a tree of all levels, children kept at random: no waiting node above its level's
// position, and the stack's room not passed
static int knn_stack(unsigned seed, double keep) {
    std::mt19937 rng(seed);
    std::bernoulli_distribution kept(keep);
    std::vector<int> level{0};
    for (int step = 0; step < 200000 && !level.empty(); ++step) {
        const size_t nb = level.size() < 8 ? level.size() : 8;
        const std::vector<int> taken(level.end() - nb, level.end());
        level.resize(level.size() - nb);
        for (size_t grp = 0; grp < nb; ++grp) {   // the topmost node's children first
            const int l = taken[nb - 1 - grp];
            for (int c = 0; c < 8; ++c)
                if (l + 1 < HV_TREE_LEVELS && kept(rng)) level.push_back(l + 1);
        }
        if (level.size() > (size_t)HV_KNN_STACK) return 1;
        for (size_t p = 0; p < level.size(); ++p)
            if (p > 63 * (size_t)level[p]) return 2;
    }
    return 0;
}

int main() {
    const int64_t meshes[] = {1, 2, 2047, 2048, 2049, 5000, 50000}, sizes[] = {3, 200, 4097};
    const int64_t rays[] = {1, 2, 50, 1023, 1024, 1025, 3000, 100000, 1 << 20, (1 << 20) + 1, 100000000};
    for (int64_t k : meshes)
        for (int64_t n : sizes)
            for (int64_t nr : rays)
                if (int e = buckets(k, n, nr)) {
                    std::printf("buckets: %lld meshes of %lld, %lld rays: check %d\n", (long long)k, (long long)n, (long long)nr, e);
                    return 1;
                }
    if (int e = buckets(1, (1 << 30) - 1, 5)) {
        std::printf("buckets: one mesh of 2^30 - 1: check %d\n", e);
        return 1;
    }
    for (unsigned seed = 0; seed < 8; ++seed)
        for (double keep : {1.0, 0.95, 0.8, 0.5, 0.3})
            if (int e = knn_stack(seed, keep)) {
                std::printf("waiting nodes: seed %u, %g kept: check %d\n", seed, keep, e);
                return 1;
            }
    return 0;
}
