// oibvh_pairs.hip -- the hit list in get_pairs order (meshA, meshB, triA, triB,
// lexicographic) on the device; the reference downloads its list unsorted
// (scene.cu:414-416).
//
// A hit is one (mesh pair, leaf pair), so no two hits of a query are equal: the
// place of a hit is the number of hits below it, and no stability is needed.
//   k_pairs_rank          short lists: every hit counts the hits below it, one
//                         launch;
//   k_pairs_split, k_pairs_bucket, k_pairs_scatter, k_pairs_sort
//                         longer ones: a sample sort. Splitters from a ranked
//                         sample, a bucket and a place in it per hit, the keys
//                         gathered by bucket, each bucket sorted in LDS.
// Keys are the four words packed into 64 bits by the bits that mesh and face ids
// can have. Where they do not fit, short lists compare 128 bits and long ones
// take the LSD passes (k_hits_digits, k_sort_pass, k_hits_gather).
#include <hip/hip_runtime.h>

#include "oibvh_common.h"

typedef unsigned long long u64;

// ---------------------------------------------------------------------------
// keys
// ---------------------------------------------------------------------------
struct Key64 {
    u64 k;
    __device__ __forceinline__ static Key64 of(const uint4& h, oi_pair_bits b)
    {
        // shifts of 32 at most: mesh bits <= 32, face bits <= 24
        const u64 m = ((u64)h.x << b.mesh) | h.y;
        const u64 t = ((u64)h.z << b.tri) | h.w;
        return Key64{b.tri ? (m << (2u * b.tri)) | t : m};
    }
    __device__ __forceinline__ static Key64 top() { return Key64{~0ull}; }
    __device__ __forceinline__ bool operator<(const Key64& o) const { return k < o.k; }
};
struct Key128 {
    u64 m, t;
    __device__ __forceinline__ static Key128 of(const uint4& h, oi_pair_bits)
    {
        return Key128{((u64)h.x << 32) | h.y, ((u64)h.z << 32) | h.w};
    }
    __device__ __forceinline__ static Key128 top() { return Key128{~0ull, ~0ull}; }
    __device__ __forceinline__ bool operator<(const Key128& o) const { return m < o.m || (m == o.m && t < o.t); }
};

__device__ __forceinline__ uint4 hit_of(u64 k, oi_pair_bits b)
{
    const uint32_t tm = (uint32_t)((1ull << b.tri) - 1ull);
    const u64 m = k >> (2u * b.tri);  // 2 b.tri <= 48
    return make_uint4((uint32_t)(m >> b.mesh), (uint32_t)(m & ((1ull << b.mesh) - 1ull)), (uint32_t)(k >> b.tri) & tm,
                      (uint32_t)k & tm);
}

__device__ __forceinline__ uint4 load_hit(const uint4* hits, uint32_t i)
{
    typedef uint32_t v4u __attribute__((ext_vector_type(4)));
    const v4u h = *((const OI_GLOBAL v4u*)oi_g(hits) + i);
    return make_uint4(h.x, h.y, h.z, h.w);
}

// ---------------------------------------------------------------------------
// counting the keys of a list below some own ones
// ---------------------------------------------------------------------------
#define PR_THREADS 512
#define PR_TILE 4096

// A workgroup owns 2 H keys, H = 2^lgh <= 32 (lane l of every wave holds keys
// l mod H and H + l mod H, so that one LDS read serves two compares) and splits
// the list over its 512 / H slices (slice s reads keys s, s + S, ... of each LDS
// tile, one address per slice and read: no bank conflict). load(i) gives list
// key i < n. Returns the counts below own0 and own1 in s_rank[l mod H] and
// s_rank[H + l mod H].
template <class K, class Load>
__device__ __forceinline__ void count_below(const Load& load, uint32_t n, const K& own0, const K& own1, uint32_t lgh,
                                            K* s_key, uint32_t* s_rank)
{
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t S = (PR_THREADS >> lgh), H = 1u << lgh;
    const uint32_t slice = wave * (64u >> lgh) + (lane >> lgh);
    if (tid < 2u * H) s_rank[tid] = 0u;
    uint32_t below0 = 0, below1 = 0;
    constexpr uint32_t J = PR_TILE / PR_THREADS;
    K next[J];
#pragma unroll
    for (uint32_t j = 0; j < J; j++) next[j] = load(min(j * PR_THREADS + tid, n - 1u));
    for (uint32_t t0 = 0; t0 < n; t0 += PR_TILE) {
        __syncthreads();
#pragma unroll
        for (uint32_t j = 0; j < J; j++) {
            const uint32_t i = j * PR_THREADS + tid;
            s_key[i] = t0 + i < n ? next[j] : K::top();  // the top key is below none
        }
        __syncthreads();
        // the next tile's keys arrive while this one is counted
        if (t0 + PR_TILE < n) {
#pragma unroll
            for (uint32_t j = 0; j < J; j++) next[j] = load(min(t0 + PR_TILE + j * PR_THREADS + tid, n - 1u));
        }
        const uint32_t m = min((uint32_t)PR_TILE, n - t0);
#pragma unroll 8
        for (uint32_t j = 0; j < m; j += S) {
            const K k = s_key[j + slice];
            below0 += k < own0 ? 1u : 0u;
            below1 += k < own1 ? 1u : 0u;
        }
    }
    atomicAdd(&s_rank[lane & (H - 1u)], below0);
    atomicAdd(&s_rank[H + (lane & (H - 1u))], below1);
    __syncthreads();
}

// One launch for a short list: n^2 compares, spread over n / 2H workgroups. It
// takes 4.0 us for 107 hits and 4.6 us for 1,500 (the launch and one pass over
// the list per workgroup, L2 hits) and 11 us for 5,100, where the compares bound
// it. The LSD passes in one workgroup that it replaces took 32, 44 and 51 us (one
// CU, a barrier chain per pass).
template <class K>
__global__ void __launch_bounds__(PR_THREADS)
k_pairs_rank(const uint4* __restrict__ hits, uint32_t n, oi_pair_bits bits, uint32_t lgh, uint4* __restrict__ out,
             uint4* __restrict__ host)
{
    __shared__ K s_key[PR_TILE];
    __shared__ uint32_t s_rank[64];
    const uint32_t H = 1u << lgh, i0 = blockIdx.x * 2u * H + (threadIdx.x & (H - 1u));
    const uint4 h0 = load_hit(hits, min(i0, n - 1u)), h1 = load_hit(hits, min(i0 + H, n - 1u));
    count_below<K>([&](uint32_t i) { return K::of(load_hit(hits, i), bits); }, n, K::of(h0, bits), K::of(h1, bits), lgh,
                   s_key, s_rank);
    if (threadIdx.x < H) {
        const uint32_t r0 = s_rank[threadIdx.x], r1 = s_rank[H + threadIdx.x];
        if (i0 < n) out[r0] = h0;
        if (i0 + H < n) out[r1] = h1;
        if (host) {
            if (i0 < n) host[r0] = h0;
            if (i0 + H < n) host[r1] = h1;
        }
    }
}

// ---------------------------------------------------------------------------
// sample sort: five launches whatever the key bits are, where the LSD passes over
// the ids' bytes need 9 to 13. Kernel times, all launches: 15,800 hits 27 us
// (LSD 115), 40,000 27 us (95), 175,000 41 us (125), 800,000 74 us (about 200).
// ---------------------------------------------------------------------------
#define PS_THREADS 512
#define PS_ITEMS 4
#define PS_TILE (PS_THREADS * PS_ITEMS)
#define PS_BUCKETS 1024  // at most
#define PS_OVER 8        // sample keys per bucket
#define PS_CAP 4096      // keys a bucket sorts in LDS

// one hit on its way to its bucket
struct PairRec {
    u64 key;
    uint32_t bucket, at;
};

// the keys of S hits (oi_sample_at) side by side (every workgroup of
// k_pairs_split reads them all: 512 of them gathering 8192 lines of hits took
// 32 us), and zeroed bucket counts
__global__ void __launch_bounds__(256)
k_pairs_sample(const uint4* __restrict__ hits, uint32_t n, oi_pair_bits bits, uint32_t S, u64* __restrict__ sample,
               uint32_t nb, uint32_t* __restrict__ counts)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i < S) sample[i] = Key64::of(load_hit(hits, oi_sample_at(i, n, S)), bits).k;
    if (i < nb) counts[i] = 0u;
}

// splitters[b - 1], b = 1 .. nb - 1: the sample key of rank b * over of the
// S = nb * over; bucket b holds the keys from splitter b - 1 on
__global__ void __launch_bounds__(PR_THREADS)
k_pairs_split(const u64* __restrict__ sample, uint32_t S, uint32_t over, uint32_t lgh, u64* __restrict__ splitters)
{
    __shared__ Key64 s_key[PR_TILE];
    __shared__ uint32_t s_rank[64];
    const uint32_t H = 1u << lgh, i0 = blockIdx.x * 2u * H + (threadIdx.x & (H - 1u));
    const Key64 k0{sample[min(i0, S - 1u)]}, k1{sample[min(i0 + H, S - 1u)]};
    count_below<Key64>([&](uint32_t i) { return Key64{sample[i]}; }, S, k0, k1, lgh, s_key, s_rank);
    if (threadIdx.x < 2u * H) {
        const bool second = threadIdx.x >= H;
        const uint32_t r = s_rank[threadIdx.x];
        if ((second ? i0 + H : i0) < S && r && r % over == 0) splitters[r / over - 1u] = second ? k1.k : k0.k;
    }
}

// bucket of every hit (a binary search over the splitters in LDS) and its place
// there: LDS counts per tile, one fetch_add per tile and bucket in use
__global__ void __launch_bounds__(PS_THREADS)
k_pairs_bucket(const uint4* __restrict__ hits, uint32_t n, oi_pair_bits bits, uint32_t nb,
               const u64* __restrict__ splitters, uint32_t* __restrict__ counts, PairRec* __restrict__ rec)
{
    __shared__ u64 s_split[PS_BUCKETS];
    __shared__ uint32_t s_cnt[PS_BUCKETS];
    const uint32_t tid = threadIdx.x;
    for (uint32_t i = tid; i < nb; i += PS_THREADS) {
        s_split[i] = i + 1u < nb ? splitters[i] : ~0ull;
        s_cnt[i] = 0u;
    }
    u64 key[PS_ITEMS];
    uint32_t b[PS_ITEMS], at[PS_ITEMS];
    const uint32_t i0 = blockIdx.x * PS_TILE + tid;
#pragma unroll
    for (int j = 0; j < PS_ITEMS; j++) {
        const uint32_t i = i0 + j * PS_THREADS;
        key[j] = Key64::of(load_hit(hits, i < n ? i : 0u), bits).k;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PS_ITEMS; j++) {
        uint32_t lo = 0, hi = nb - 1u;  // splitters at or below the key, 0 .. nb - 1
        while (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            if (s_split[mid] <= key[j])
                lo = mid + 1u;
            else
                hi = mid;
        }
        b[j] = lo;
        at[j] = i0 + j * PS_THREADS < n ? atomicAdd(&s_cnt[lo], 1u) : 0u;
    }
    __syncthreads();
    for (uint32_t i = tid; i < nb; i += PS_THREADS) {
        const uint32_t c = s_cnt[i];
        if (c) s_cnt[i] = __hip_atomic_fetch_add(counts + i, c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PS_ITEMS; j++) {
        const uint32_t i = i0 + j * PS_THREADS;
        if (i < n) rec[i] = PairRec{key[j], b[j], s_cnt[b[j]] + at[j]};
    }
}

// keys gathered by bucket: every workgroup scans the counts for the buckets'
// first places (workgroup 0 writes them out, nb + 1 of them)
__global__ void __launch_bounds__(PS_THREADS)
k_pairs_scatter(const PairRec* __restrict__ rec, uint32_t n, uint32_t nb, const uint32_t* __restrict__ counts,
                uint32_t* __restrict__ starts, u64* __restrict__ keys)
{
    __shared__ uint32_t s_start[PS_BUCKETS];
    __shared__ uint32_t s_wsum[PS_THREADS / 64];
    static_assert(PS_BUCKETS == 2 * PS_THREADS, "two counts per thread");
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    PairRec r[PS_ITEMS];
    const uint32_t i0 = blockIdx.x * PS_TILE + tid;
#pragma unroll
    for (int j = 0; j < PS_ITEMS; j++) {
        const uint32_t i = i0 + j * PS_THREADS;
        r[j] = rec[i < n ? i : 0u];
    }
    const uint32_t c0 = 2u * tid < nb ? counts[2u * tid] : 0u, c1 = 2u * tid + 1u < nb ? counts[2u * tid + 1u] : 0u;
    const uint32_t x = oi_wave_scan_incl(c0 + c1);
    if (lane == 63u) s_wsum[wave] = x;
    __syncthreads();
    uint32_t s = x - (c0 + c1);
#pragma unroll
    for (uint32_t w = 0; w < PS_THREADS / 64; w++) s += w < wave ? s_wsum[w] : 0u;
    s_start[2u * tid] = s;
    s_start[2u * tid + 1u] = s + c0;
    if (blockIdx.x == 0) {
        if (2u * tid < nb) starts[2u * tid] = s;
        if (2u * tid + 1u < nb) starts[2u * tid + 1u] = s + c0;
        if (tid == 0) starts[nb] = n;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PS_ITEMS; j++)
        if (i0 + j * PS_THREADS < n) keys[s_start[r[j].bucket] + r[j].at] = r[j].key;
}

// places a < b of a list of m, ascending (places from m on hold the top key)
__device__ __forceinline__ void order_pair(u64* g, uint32_t a, uint32_t b, uint32_t m)
{
    if (b >= m) return;
    const u64 x = g[a], y = g[b];
    if (x > y) {
        g[a] = y;
        g[b] = x;
    }
}

// One bucket per workgroup, bitonic in LDS; a wave's 64 compare-exchanges of a
// stage of distance <= 64 cover 128 consecutive keys in every such stage, so
// only wider ones need a barrier. A bucket that outgrew LDS (the sample missed
// badly) is sorted in place in memory, every merge ascending (its first stage
// compares mirrored places) so that the places past its end never move: all of
// 40,000 keys in one bucket 1.4 ms, of 175,000 7.1, where ranking them against each
// other took the square of their number.
__global__ void __launch_bounds__(PS_THREADS)
k_pairs_sort(u64* keys, const uint32_t* __restrict__ starts, oi_pair_bits bits, uint4* __restrict__ out)
{
    __shared__ u64 s[PS_CAP];
    const uint32_t tid = threadIdx.x, p0 = starts[blockIdx.x], m = starts[blockIdx.x + 1u] - p0;
    if (m > PS_CAP) {
        u64* g = keys + p0;
        uint32_t P = PS_CAP;
        while (P < m) P <<= 1;  // m <= 2^30
        for (uint32_t k = 2; k <= P; k <<= 1) {
            for (uint32_t i = tid; i < (P >> 1); i += PS_THREADS) {
                const uint32_t a = 2u * i - (i & ((k >> 1) - 1u));
                order_pair(g, a, a ^ (k - 1u), m);
            }
            __syncthreads();
            for (uint32_t j = k >> 2; j; j >>= 1) {
                for (uint32_t i = tid; i < (P >> 1); i += PS_THREADS) {
                    const uint32_t a = 2u * i - (i & (j - 1u));
                    order_pair(g, a, a + j, m);
                }
                __syncthreads();
            }
        }
        for (uint32_t i = tid; i < m; i += PS_THREADS) out[p0 + i] = hit_of(g[i], bits);
        return;
    }
    uint32_t P = 128;
    while (P < m) P <<= 1;
    for (uint32_t i = tid; i < P; i += PS_THREADS) s[i] = i < m ? keys[p0 + i] : ~0ull;
    __syncthreads();
    for (uint32_t k = 2; k <= P; k <<= 1) {
        for (uint32_t j = k >> 1; j; j >>= 1) {
            for (uint32_t i = tid; i < (P >> 1); i += PS_THREADS) {
                const uint32_t a = 2u * i - (i & (j - 1u)), b = a + j;
                const u64 x = s[a], y = s[b];
                if ((x > y) == ((a & k) == 0u)) {
                    s[a] = y;
                    s[b] = x;
                }
            }
            // the next stage: j / 2, or k when this was the last of its merge
            const uint32_t next = j > 1u ? j >> 1 : k;
            if (j > 64u || next > 64u)
                __syncthreads();
            else
                oi_wave_fence();
        }
    }
    for (uint32_t i = tid; i < m; i += PS_THREADS) out[p0 + i] = hit_of(s[i], bits);
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
// half the own keys per workgroup, log2: few enough for about two workgroups
// per CU
static uint32_t rank_lgh(uint32_t n)
{
    uint32_t lg = 2;
    while (lg < 5 && (n >> (lg + 1u)) > 512u) lg++;
    return lg;
}

extern "C" {

// wide: the keys' bits do not fit into 64
// host: pinned memory that receives the list too, or null
hipError_t oi_launch_pairs_rank(hipStream_t st, const uint4* hits, uint32_t n, oi_pair_bits bits, int wide, uint4* out,
                                uint4* host)
{
    if (n == 0) return hipSuccess;
    const uint32_t lgh = rank_lgh(n), grid = (n + (2u << lgh) - 1u) >> (lgh + 1u);
    if (wide)
        hipLaunchKernelGGL(k_pairs_rank<Key128>, dim3(grid), dim3(PR_THREADS), 0, st, hits, n, bits, lgh, out,
                           host);
    else
        hipLaunchKernelGGL(k_pairs_rank<Key64>, dim3(grid), dim3(PR_THREADS), 0, st, hits, n, bits, lgh, out,
                           host);
    return hipGetLastError();
}

// bytes of scratch of a sample sort of n hits: records, keys, splitters, counts
// and starts
uint64_t oi_pairs_sort_bytes(uint32_t n)
{
    return (uint64_t)n * (sizeof(PairRec) + sizeof(u64)) + PS_BUCKETS * sizeof(u64) +
           (2ull * PS_BUCKETS + 1u) * sizeof(uint32_t);
}

hipError_t oi_launch_pairs_sort(hipStream_t st, const uint4* hits, uint32_t n, oi_pair_bits bits, void* scratch,
                                uint4* out)
{
    if (n < PS_BUCKETS * PS_OVER / 2u || n > 1u << 30 || 2u * (bits.mesh + bits.tri) > 64u) return hipErrorInvalidValue;
    PairRec* rec = (PairRec*)scratch;
    u64* keys = (u64*)(rec + n);
    u64* splitters = keys + n;
    uint32_t* counts = (uint32_t*)(splitters + PS_BUCKETS);
    uint32_t* starts = counts + PS_BUCKETS;
    // buckets of about 256 keys, at most PS_BUCKETS of them; the sample lies
    // where the keys go later
    uint32_t nb = n / 256u;
    if (nb > PS_BUCKETS) nb = PS_BUCKETS;
    const uint32_t S = nb * PS_OVER, lgh = rank_lgh(S), tiles = (n + PS_TILE - 1u) / PS_TILE;
    hipLaunchKernelGGL(k_pairs_sample, dim3((S + 255u) / 256u), dim3(256), 0, st, hits, n, bits, S, keys, nb, counts);
    hipLaunchKernelGGL(k_pairs_split, dim3((S + (2u << lgh) - 1u) >> (lgh + 1u)), dim3(PR_THREADS), 0, st, keys, S, PS_OVER,
                       lgh, splitters);
    hipLaunchKernelGGL(k_pairs_bucket, dim3(tiles), dim3(PS_THREADS), 0, st, hits, n, bits, nb, splitters, counts, rec);
    hipLaunchKernelGGL(k_pairs_scatter, dim3(tiles), dim3(PS_THREADS), 0, st, rec, n, nb, counts, starts, keys);
    hipLaunchKernelGGL(k_pairs_sort, dim3(nb), dim3(PS_THREADS), 0, st, keys, starts, bits, out);
    return hipGetLastError();
}

}  // extern "C"
