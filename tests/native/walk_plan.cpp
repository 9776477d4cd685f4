// Host checks of hv_plan.h: exit status 0 when every one holds.
#include "hv_plan.h"
#include <cstdio>

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
    return 0;
}
