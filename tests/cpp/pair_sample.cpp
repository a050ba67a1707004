// The sample sort of pair lists on lists whose order follows the sample's stride:
// the keys of its largest bucket. (Buckets of about n / nb keys; a workgroup sorts
// 4,096 in LDS, and one that holds more takes many times longer.)
#include <cstdio>

#include "oibvh_internal.h"

// as the sort takes its splitters: every 8th key of a ranked sample of 8 per bucket
static uint32_t largest_bucket(const std::vector<uint32_t>& keys)
{
    const uint32_t n = (uint32_t)keys.size(), nb = std::min(1024u, n / 256u), S = 8u * nb;
    std::vector<uint32_t> sample(S);
    for (uint32_t i = 0; i < S; i++) {
        const uint32_t at = oi_sample_at(i, n, S);
        if (at < (uint64_t)i * n / S || at >= (uint64_t)(i + 1) * n / S) {
            std::printf("n %u: sample %u at %u, outside its stride\n", n, i, at);
            return ~0u;
        }
        sample[i] = keys[at];
    }
    std::sort(sample.begin(), sample.end());
    std::vector<uint32_t> count(nb, 0u);
    for (uint32_t k : keys) {
        uint32_t b = 0;
        for (uint32_t step = 1024; step; step >>= 1)
            if (b + step < nb && sample[8u * (b + step)] <= k) b += step;
        count[b]++;
    }
    return *std::max_element(count.begin(), count.end());
}

int main()
{
    int bad = 0;
    for (uint32_t n : {9217u, 10240u, 16384u, 65536u, 262144u, 300000u, 1u << 20}) {
        // groups of `len` hits, as a workgroup appends them: the first `low` of each
        // group come from one end of the key range and the others from the other
        for (uint32_t len : {2u, 16u, 32u, 33u, 64u, 128u, 256u, 512u})
            for (uint32_t low : {1u, len / 2u, len - 1u}) {
                std::vector<uint32_t> keys(n);
                for (uint32_t i = 0; i < n; i++) keys[i] = i % len < low ? i : (1u << 24) + i;
                const uint32_t most = largest_bucket(keys);
                if (most > 4096u) std::printf("n %u, groups of %u, %u low: %u keys\n", n, len, low, most), bad = 1;
            }
        std::vector<uint32_t> ordered(n), reverse(n);
        for (uint32_t i = 0; i < n; i++) ordered[i] = i, reverse[i] = n - i;
        if (largest_bucket(ordered) > 4096u || largest_bucket(reverse) > 4096u) std::printf("n %u ordered\n", n), bad = 1;
    }
    return bad;
}
