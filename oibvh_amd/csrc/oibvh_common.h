// oibvh_common.h -- device descriptors and device helpers shared by host code
// and kernels; the layout math lives in oibvh_layout.h.
#pragma once
#include "oibvh_layout.h"

#if defined(__HIPCC__) || defined(__HIP__)
// Pointers read from descriptor tables are generic to the compiler, which
// then emits flat memory instructions; these views make them global so that
// loads and stores are global_* and adjacent words combine into one
// multi-dword access (indices are 64-bit so adjacency is provable).
#define OI_GLOBAL __attribute__((address_space(1)))
template <class T>
__device__ __forceinline__ const OI_GLOBAL T* oi_g(const T* p)
{
    return (const OI_GLOBAL T*)p;
}
template <class T>
__device__ __forceinline__ OI_GLOBAL T* oi_gw(T* p)
{
    return (OI_GLOBAL T*)p;
}
// three consecutive 32-bit words at base + 3 i (a vertex or a face)
__device__ __forceinline__ void oi_ld3(const float* base, uint32_t i, float* o)
{
    const OI_GLOBAL float* q = oi_g(base) + 3ull * i;
    o[0] = q[0];
    o[1] = q[1];
    o[2] = q[2];
}
__device__ __forceinline__ void oi_ld3(const uint32_t* base, uint32_t i, uint32_t* o)
{
    const OI_GLOBAL uint32_t* q = oi_g(base) + 3ull * i;
    o[0] = q[0];
    o[1] = q[1];
    o[2] = q[2];
}
// orders a wave's LDS accesses (its lanes exchange values through LDS)
__device__ __forceinline__ void oi_wave_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// inclusive prefix sum over the 64 lanes of a wave (every lane active) with
// DPP moves instead of LDS permutes: a Kogge-Stone scan inside each row of
// 16 lanes (row_shr 1, 2, 4, 8; a lane shifted in from outside its row
// reads 0), then rows 1 and 3 add the last lane of the row before them
// (row_bcast:15), then rows 2 and 3 add lane 31 (row_bcast:31)
__device__ __forceinline__ uint32_t oi_wave_scan_incl(uint32_t x)
{
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, true);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, true);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, true);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, true);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, false);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xc, 0xf, false);
    return x;
}
#endif

#define OI_HIST_WORDS 3072u  // one copy of a build's digit histograms: 8 x 256 or 3 x 1024 bins
#define OI_HIST_REPS 8u      // copies of them
#define OI_SORT_WGS 256u     // tiles a sort pass is divided into, if it has keys enough
#define OI_SORT_GROUP 8u     // tiles of a look-back group

// ---------------------------------------------------------------------------
// device descriptors
// ---------------------------------------------------------------------------

// p' = M * vec4(p, 1) with glm's evaluation order for mat4 * vec4
// (type_mat4x4.inl:561-573): (m[0] x + m[1] y) + (m[2] z + m[3] * 1), m[c] the
// c-th column, stored column-major like glm::mat4 (xf[4c + r]). This is the
// vertex transform of Mesh::transform (mesh.cpp:189-214, transform.cu:35-41).
OI_HD void oi_xform(const float* xf, float x, float y, float z, float* o)
{
    for (int r = 0; r < 3; r++) {
        const float a = xf[r] * x;
        const float b = xf[4 + r] * y;
        const float c = xf[8 + r] * z;
        const float d = xf[12 + r] * 1.0f;
        o[r] = (a + b) + (c + d);
    }
}

// One mesh as the build and refit kernels see it.
struct oi_build_desc {
    const float* pos;        // V*3 vertex positions
    const float* xf;         // model matrix applied to pos (oi_xform), or null
    const uint32_t* faces;   // F*3 original faces (vertex ids local to the mesh)
    uint32_t* sfaces;        // F*3 faces in leaf order (written by the build, read by the refit)
    uint32_t* perm;          // F: leaf -> original face id
    float* nodes;            // N*6 floats, real order
    float* box;              // 6 floats: the Morton quantisation box (written by the build)
    uint32_t F, V, L, vl;
    uint32_t fbase;          // offset in the concatenated per-face sort arrays
    uint32_t pbase;          // first mesh-box partial of this mesh
    uint32_t nparts;         // mesh-box partials (1..256)
    uint32_t vchunk;         // vertices per mesh-box partial
};

// One mesh as the traversal sees it. `ibase` is the mesh's offset in the
// scene's concatenated implicit-index space (each mesh spans 2^(L+1) - 1).
struct oi_mesh_desc {
    const float* nodes;      // N*6 floats, real order: min.xyz, max.xyz
    const uint32_t* sfaces;  // F*3, faces in leaf (Morton) order
    const float* pos;        // V*3 vertex positions
    const uint32_t* perm;    // F: leaf position -> original face id
    const float* xf;         // model matrix applied to pos, or null
    uint32_t F, L, vl, N;
    uint32_t ibase;
    uint32_t pad0;
};

// A mesh table is either a scene's (d_meshes / h_meshes, n_meshes) or, when
// chunk_mesh is not null, a batch's (d_meshes indexed through chunk_mesh).
struct oi_tab_args {
    const oi_mesh_desc* d_meshes;
    const oi_mesh_desc* h_meshes;
    uint32_t n_meshes;
    const uint32_t* chunk_mesh;
    uint32_t shift;
};

// Statistics of a detect, in shards: workgroup b adds to shard b % OI_STAT_SHARDS
// and the shards are summed when the counters are read. A thousand workgroups
// that end together and add to one cache line take 10 us about it (a walk launch
// of 16 us took 35).
#define OI_STAT_SHARDS 64
struct alignas(128) oi_detect_stat {
    unsigned long long tests;  // BVTT box pair tests
    unsigned long long adj;    // leaf pairs dropped as adjacent (self mode)
    unsigned long long fp64;   // SAT axis comparisons re-evaluated in double
    uint32_t cands;            // leaf pairs tested where they were found
};

// Detect counters, reset by the seed kernel before each detect; those that hand
// out places in a list lie on lines of their own.
struct oi_detect_ctl {
    alignas(128) uint32_t n_hits;    // hits found (may exceed capacity)
    alignas(128) uint32_t cands;     // leaf pairs put into the candidate list (may exceed capacity)
    alignas(128) uint32_t deferred;  // FP64 fallback: candidates the FP32 filter left undecided
    alignas(128) uint32_t error;     // OI_ERR_* bits of this detect
    uint32_t sticky;                 // OI_ERR_* bits of earlier asynchronous detects not checked since
    oi_detect_stat stat[OI_STAT_SHARDS];
};

#if defined(__HIPCC__) || defined(__HIP__)
// thread tid of a workgroup of at least OI_STAT_SHARDS threads resets ctl; errors
// of the previous detect move to `sticky` unless the caller checked it
// synchronously
__device__ __forceinline__ void oi_reset_ctl(oi_detect_ctl* ctl, uint32_t tid, uint32_t reset_sticky)
{
    if (tid == 0) {
        ctl->sticky = reset_sticky ? 0u : (ctl->sticky | ctl->error);
        ctl->error = 0;
        ctl->n_hits = 0;
        ctl->cands = 0;
        ctl->deferred = 0;
    }
    if (tid < OI_STAT_SHARDS) {
        oi_detect_stat* s = ctl->stat + tid;
        s->tests = 0;
        s->adj = 0;
        s->fp64 = 0;
        s->cands = 0;
    }
}
#endif

// What a check reads of a query, in pinned host memory that k_publish writes:
// the current counter set's counters and front lengths, the error words of the
// other unchecked sets, and last the sequence number that the host waits for
#define OI_PUB_SETS 4
#define OI_PUB_COUNTS 256
struct oi_published {
    uint32_t n_hits, cands, deferred, error, sticky;
    uint32_t earlier;  // error and sticky bits of the other sets
    unsigned long long tests, adj, fp64;
    uint32_t counts[OI_PUB_COUNTS];
    uint32_t seq;
};
struct oi_publish_args {
    oi_detect_ctl* ctl[OI_PUB_SETS];  // n_sets sets, the current one first; their error and sticky words are cleared
    uint32_t n_sets;
    const uint32_t* counts;           // n_counts <= OI_PUB_COUNTS
    uint32_t n_counts;
    oi_published* out;
    uint32_t seq;
};

// a detect's counter reset (zeroed level counts and result counters), done
// by the last workgroup of a refit's apex launch when a detect follows it in
// the same frame call, instead of a launch of its own
struct oi_seed_args {
    uint32_t* counts;  // null: no reset in this launch
    oi_detect_ctl* ctl;
    uint32_t n0, n_counts, reset_sticky, pad;
};

#define OI_ERR_QUEUE_OVERFLOW 1u  // a BVTT front exceeded its buffer
#define OI_ERR_TIMEOUT 2u
#define OI_ERR_CORRUPT 4u
#define OI_ERR_HITS_OVERFLOW 8u
#define OI_ERR_CAND_OVERFLOW 16u
#define OI_ERR_LOCAL_OVERFLOW 32u  // a workgroup's front outgrew its LDS queue (head local walk)
#define OI_ERR_TAIL_OVERFLOW 64u   // the same in the tail local walk

// one launch of the workgroup-local walk (k_bvtt_local)
struct oi_local_args {
    const uint2* front_in;
    const uint32_t* count_in;  // device length of front_in (null: n_in, one workgroup per chunk)
    uint32_t n_in;
    uint32_t cap_in;           // entries front_in holds (with count_in)
    uint32_t chunk;            // entries per workgroup and pass, at most 2048
    uint32_t levels;           // steps walked; the last one's non-leaf pairs go to front_out
    uint32_t grid;             // with count_in: at most this many workgroups (0: one per chunk of cap_in)
    uint32_t test_entries;     // test the input pairs themselves (the initial front)
    uint32_t overflow_bit;     // error bit set on an LDS front overflow
    uint2* front_out;
    uint32_t* count_out;
    uint32_t cap_out;
    hipEvent_t done;           // recorded when the launch completes (null: none)
};

// one launch of k_bvtt_walk
struct oi_walk_args {
    const uint2* front_in;
    const uint32_t* count_in;  // device length of front_in (null: n_in)
    uint32_t n_in;
    uint32_t cap_in;           // entries front_in holds (with count_in)
    uint32_t e1, e2;           // levels of the first and the second step (e2 = 0: one step)
    uint32_t test_entries;     // test the input pairs themselves (the initial front)
    uint2* front_out;
    uint32_t* count_mid;       // with e2: counts the first step's kept pairs
    uint32_t* count_out;
    uint32_t cap_out;
    uint32_t wgs_long;         // workgroups for a long front (0: as for a short one)
    hipEvent_t done;           // recorded when the launch completes (null: none)
};

// the bytes a device sort of the hit list visits, least significant first:
// digit p is byte shift[p] / 8 of word word[p] (0 meshA, 1 meshB, 2 triA,
// 3 triB)
#define OI_HIT_DIGITS 16
struct oi_hit_digits {
    uint32_t nd;
    uint8_t word[OI_HIT_DIGITS];
    uint8_t shift[OI_HIT_DIGITS];
};

// The place in a list of n hits of its sample's i-th of S <= n keys: anywhere in the
// i-th of S even strides, by a multiplicative hash of i. (Evenly spaced, a list whose
// order repeats with the stride gave a sample of one kind of its hits: one bucket then
// held nearly all the others.)
OI_HD uint32_t oi_sample_at(uint32_t i, uint32_t n, uint32_t S)
{
    const uint32_t lo = (uint32_t)((uint64_t)i * n / S), hi = (uint32_t)((uint64_t)(i + 1u) * n / S);
    uint32_t h = (i + 1u) * 2654435769u;  // 2^32 over the golden ratio
    h = (h ^ (h >> 16)) * 2654435769u;
    h ^= h >> 15;
    return lo + (uint32_t)((uint64_t)h * (hi - lo) >> 32);
}

// bits that the mesh ids and the face ids of a hit list can have (a sort key
// holds two of each)
struct oi_pair_bits {
    uint32_t mesh, tri;
};

// a scene's concatenated implicit index space must stay below this bound
#define OI_IMPLICIT_LIMIT 0xfffffffeu

// detect flags (mirror include/oibvh.h)
#define OI_DETECT_SELF 1u
#define OI_DETECT_FP64_FALLBACK 2u
