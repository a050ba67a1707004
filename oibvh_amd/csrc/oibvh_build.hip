// oibvh_build.hip -- gfx950 kernels for oibvh tree build and refit.
//
// Build (OibvhTree::build, oibvhTree.cu:237-388):
//   k_mesh_box     per-block vertex AABBs (the Morton quantisation box,
//                  Mesh::setupAABB mesh.cpp:91-98); also clears the sort's
//                  scratch counters
//   k_morton       folds the block boxes, then leaf AABB centroid -> 30-bit
//                  Morton key per face
//                  (calculate_aabb_and_morton_kernel, oibvh.cu:42-70) and the
//                  three 10-bit digit histograms of the keys (8-bit digits
//                  for 63-bit keys and batches)
//   k_sort_pass x3 onesweep LSD radix pass with decoupled look-back; stable,
//                  so the permutation equals thrust::stable_sort_by_key's
//                  (oibvhTree.cu:287-297)
//   k_reduce       leaves in sorted order + bottom-up AABB reduce, one subtree
//                  per workgroup; k_reduce_apex climbs the rest in one workgroup
//                  (oibvh_tree_construction_kernel2, oibvh.cu:156-219)
// Refit (OibvhTree::refit, oibvhTree.cu:193-235) is k_reduce alone over the
// already sorted faces (calculate_aabb_kernel + oibvh_tree_construction_kernel,
// oibvh.cu:24-40, 80-154).
//
// Every kernel is table-driven: a BuildTab names the meshes (oi_build_desc)
// and maps each workgroup to a (mesh, chunk) work item, so one launch per
// stage serves one tree or a batch of hundreds of trees. Vertex positions go
// through the mesh's model matrix when it has one (Mesh::transform,
// mesh.cpp:189-214), evaluated on the fly wherever a position is read.
//
// Compiled with -ffp-contract=off. min/max are compare-selects with glm's tie
// rules: min(a,b) = b < a ? b : a, max(a,b) = a < b ? b : a.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include "oibvh_common.h"

#define OI_BLOCK 256
#define OI_MORTON_T 1024    // threads of k_morton

__device__ __forceinline__ float gmin(float a, float b) { return (b < a) ? b : a; }
__device__ __forceinline__ float gmax(float a, float b) { return (a < b) ? b : a; }

__device__ __forceinline__ uint32_t ld_acq_relaxed(const uint32_t* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_relaxed(uint32_t* p, uint32_t v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ---------------------------------------------------------------------------
// mesh tables
// ---------------------------------------------------------------------------
// Meshes come from a device table with a work list, or (d = null) travel in
// the kernel arguments: up to OI_INLINE_MESHES meshes, mesh m owning the
// workgroups [boff[m], boff[m + 1]).
// The mesh is read by its index with scalar loads, from the table or from the
// argument segment (the table is the kernel's first argument): indexing the argument
// itself would put a copy of it into scratch memory, and picked from copies in
// registers the descriptor took 28 VGPRs of k_reduce_w (109 -> 81, so that six waves
// a SIMD fit instead of four: 128 instanced scenes, 4 frames, 5,136 -> 4,923 us).
typedef const __attribute__((address_space(4))) uint32_t* args_t;
__device__ __forceinline__ oi_build_desc uniform_desc(args_t a)
{
    uint32_t w[sizeof(oi_build_desc) / 4u];
#pragma unroll
    for (uint32_t k = 0; k < sizeof(oi_build_desc) / 4u; k++) w[k] = a[k];
    oi_build_desc d;
    __builtin_memcpy(&d, w, sizeof d);
    return d;
}

#define OI_INLINE_MESHES 4
struct BuildTab {
    const oi_build_desc* d;  // device table, or null
    const uint2* work;       // workgroup -> (mesh, chunk) for the device table
    uint32_t n_inl;
    uint32_t boff[OI_INLINE_MESHES + 1];
    oi_build_desc inl[OI_INLINE_MESHES];
    __device__ __forceinline__ uint2 item() const { return item_at(blockIdx.x, gridDim.x); }
    // work item of virtual workgroup v of n (a launch of fewer workgroups
    // than items loops v over b, b + gridDim.x, ...: with gridDim.x a
    // multiple of 8, v stays on workgroup b's XCD)
    __device__ __forceinline__ uint2 item_at(uint32_t v, uint32_t n) const
    {
        const uint32_t w = oi_xcd_remap(v, n);
        if (work) return work[w];
        uint32_t m = 0;
#pragma unroll
        for (uint32_t k = 1; k < OI_INLINE_MESHES; k++)
            if (k < n_inl && w >= boff[k]) m = k;
        return make_uint2(m, w - boff[m]);
    }
    __device__ __forceinline__ oi_build_desc mesh(uint32_t m) const
    {
        m = (uint32_t)__builtin_amdgcn_readfirstlane((int)m);
        return uniform_desc(d ? (args_t)(d + m) : (args_t)__builtin_amdgcn_kernarg_segment_ptr() +
                                                      (offsetof(BuildTab, inl) + m * sizeof(oi_build_desc)) / 4u);
    }
};

// Up to OI_WIDE_MESHES meshes in the kernel arguments, for a refit's launches: one
// pair for 16 trees instead of four (16 moving bodies 253 -> 216 us a frame, five 127
// -> 117). A table of its own, so that four trees and fewer pass a quarter of the
// bytes.
#define OI_WIDE_MESHES 16
struct WideTab {
    uint32_t n;
    uint32_t boff[OI_WIDE_MESHES + 1];
    oi_build_desc inl[OI_WIDE_MESHES];
    __device__ __forceinline__ uint2 item() const { return item_at(blockIdx.x, gridDim.x); }
    __device__ __forceinline__ uint2 item_at(uint32_t v, uint32_t total) const
    {
        const uint32_t w = oi_xcd_remap(v, total);
        uint32_t m = 0, first = 0;
#pragma unroll
        for (uint32_t k = 1; k < OI_WIDE_MESHES; k++)
            if (k < n && w >= boff[k]) {
                m = k;
                first = boff[k];
            }
        return make_uint2(m, w - first);
    }
    __device__ __forceinline__ oi_build_desc mesh(uint32_t m) const
    {
        m = (uint32_t)__builtin_amdgcn_readfirstlane((int)m);
        return uniform_desc((args_t)__builtin_amdgcn_kernarg_segment_ptr() +
                            (offsetof(WideTab, inl) + m * sizeof(oi_build_desc)) / 4u);
    }
};

// a mesh's model matrix, held in registers
struct Xf {
    float m[16];
    bool on;
    __device__ __forceinline__ void load(const float* xf)
    {
        on = xf != nullptr;
#pragma unroll
        for (int k = 0; k < 16; k++) m[k] = on ? oi_g(xf)[k] : 0.0f;
    }
    // a loaded position through the matrix (or as is)
    __device__ __forceinline__ void apply(const float* p, float* o) const
    {
        if (on) {
            oi_xform(m, p[0], p[1], p[2], o);
        } else {
            o[0] = p[0];
            o[1] = p[1];
            o[2] = p[2];
        }
    }
    __device__ __forceinline__ void vertex(const float* pos, uint32_t v, float* o) const
    {
        float p[3];
        oi_ld3(pos, v, p);
        apply(p, o);
    }
};

// ---------------------------------------------------------------------------
// k_mesh_box: vertex AABB with the sequential fold's exact result.
// The fold acc = glm::min(v, acc) keeps the later value on ties, so partial
// results combine as lo(L, R) = L < R ? L : R and hi(L, R) = R < L ? L : R in
// index order; +-inf are the identities, the default box (+-FLT_MAX) is folded
// in first, as aabb_box_t's initial value (utils.h:17-18).
// Work item (m, c): vertices [c * vchunk, (c + 1) * vchunk) of mesh m, partial
// box c of the mesh (at partials + 6 (pbase + c), or with partials null in the
// mesh's own box buffer at box + 6 + 6 c).
// ---------------------------------------------------------------------------
__device__ __forceinline__ float lo_c(float l, float r) { return (l < r) ? l : r; }
__device__ __forceinline__ float hi_c(float l, float r) { return (r < l) ? l : r; }

// A wave's lo_c / hi_c in lane order (lane 63 holds it), neighbours first, then
// pairs of pairs, through the data-parallel primitives of oi_wave_scan_incl; a
// lane without a left neighbour folds the identity.
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_left(float identity, float x)
{
    return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp((int)__float_as_uint(identity),
                                                                 (int)__float_as_uint(x), CTRL, ROWS, 0xf, false));
}
__device__ __forceinline__ float wave_lo(float x)
{
    const float id = __builtin_inff();
    x = lo_c(dpp_left<0x111, 0xf>(id, x), x);
    x = lo_c(dpp_left<0x112, 0xf>(id, x), x);
    x = lo_c(dpp_left<0x114, 0xf>(id, x), x);
    x = lo_c(dpp_left<0x118, 0xf>(id, x), x);
    x = lo_c(dpp_left<0x142, 0xa>(id, x), x);
    return lo_c(dpp_left<0x143, 0xc>(id, x), x);
}
__device__ __forceinline__ float wave_hi(float x)
{
    const float id = -__builtin_inff();
    x = hi_c(dpp_left<0x111, 0xf>(id, x), x);
    x = hi_c(dpp_left<0x112, 0xf>(id, x), x);
    x = hi_c(dpp_left<0x114, 0xf>(id, x), x);
    x = hi_c(dpp_left<0x118, 0xf>(id, x), x);
    x = hi_c(dpp_left<0x142, 0xa>(id, x), x);
    return hi_c(dpp_left<0x143, 0xc>(id, x), x);
}

// The ordered fold of OI_BLOCK threads' boxes (threads from OI_BLOCK on have
// none); every thread gets the result.
__device__ __forceinline__ void fold_box(float (*s_v)[6], float* mn, float* mx)
{
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    if (wave < OI_BLOCK / 64) {
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const float lo = wave_lo(mn[k]), hi = wave_hi(mx[k]);
            if (lane == 63u) {
                s_v[wave][k] = lo;
                s_v[wave][3 + k] = hi;
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 3; k++) {
        mn[k] = lo_c(lo_c(s_v[0][k], s_v[1][k]), lo_c(s_v[2][k], s_v[3][k]));
        mx[k] = hi_c(hi_c(s_v[0][3 + k], s_v[1][3 + k]), hi_c(s_v[2][3 + k], s_v[3][3 + k]));
    }
}

__global__ void __launch_bounds__(OI_BLOCK)
k_mesh_box(BuildTab T, float* __restrict__ partials, uint32_t* __restrict__ clear_u32, uint32_t clear_n)
{
    const uint32_t tid = threadIdx.x;
    for (uint32_t i = blockIdx.x * OI_BLOCK + tid; i < clear_n; i += gridDim.x * OI_BLOCK) clear_u32[i] = 0u;

    __shared__ float s_v[OI_BLOCK / 64][6];
    const uint2 it = T.item();
    const oi_build_desc D = T.mesh(it.x);
    Xf X;
    X.load(D.xf);
    const float INF = __builtin_inff();
    float mn[3] = {INF, INF, INF}, mx[3] = {-INF, -INF, -INF};
    const uint32_t chunk = D.vchunk;
    const uint32_t b0 = it.y * chunk;
    const uint32_t b1 = min(D.V, b0 + chunk);
    const uint32_t sub = (chunk + OI_BLOCK - 1) / OI_BLOCK;
    const uint32_t s0 = b0 + tid * sub;
    const uint32_t s1 = min(b1, s0 + sub);
    // the thread's run in index order, eight vertices loaded per round trip
    // (positions past the run load vertex s0 and are not folded). Through the matrix
    // only after the last load: whether there is one is a scalar branch, and the loads
    // waited for each other across it (21M vertices with matrices 392 -> 112 us)
    for (uint32_t v0 = s0; v0 < s1; v0 += 8u) {
        float p[8][3];
#pragma unroll
        for (int j = 0; j < 8; j++) oi_ld3(D.pos, v0 + j < s1 ? v0 + j : s0, p[j]);
#pragma unroll
        for (int j = 0; j < 8; j++) {
            if (v0 + j >= s1) continue;
            float o[3];
            X.apply(p[j], o);
#pragma unroll
            for (int k = 0; k < 3; k++) {
                mn[k] = lo_c(mn[k], o[k]);
                mx[k] = hi_c(mx[k], o[k]);
            }
        }
    }
    fold_box(s_v, mn, mx);
    float* P = partials ? partials + 6u * D.pbase : D.box + 6;
    if (tid < 6) {
        float r = 0.0f;
#pragma unroll
        for (int k = 0; k < 6; k++)
            if ((int)tid == k) r = k < 3 ? mn[k] : mx[k - 3];
        oi_gw(P)[6u * it.y + tid] = r;
    }
}

// ---------------------------------------------------------------------------
// k_morton: Morton30 of each face's leaf-box centroid (oibvh.cu:6-22, 42-70)
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t spread10(uint32_t x)
{
    x &= 0x3ffu;
    x = (x | (x << 16)) & 0x30000ffu;
    x = (x | (x << 8)) & 0x300f00fu;
    x = (x | (x << 4)) & 0x30c30c3u;
    x = (x | (x << 2)) & 0x9249249u;
    return x;
}

// thrust::min(thrust::max(p * 1024, 0), 1023) -> unsigned; NaN -> 0
__device__ __forceinline__ uint32_t quantise10(float p)
{
    float q = p * 1024.0f;
    q = (q < 0.0f) ? 0.0f : q;
    q = (1023.0f < q) ? 1023.0f : q;
    return (q != q) ? 0u : (uint32_t)q;
}

// Work item (m, c): faces [c * chunk, (c + 1) * chunk) of mesh m, chunk = 1024 NJ. Keys go to keys[fbase + face]; the 8-bit digit histograms of the
// keys accumulate in ghist + m * hstride (hstride 0: one set for all keys of
// the launch); fmesh (if not null) receives the mesh id of each face
// (fmesh[fbase + face] = m). The mesh-box partials are read from partials +
// 6 pbase, or with partials null from the mesh's own box buffer (box + 6).
// 63-bit form (no reference counterpart): 21 bits per axis, quantised as
// min(max(p * 2^21, 0), 2^21 - 1), NaN -> 0
__device__ __forceinline__ uint64_t spread21(uint64_t x)
{
    x &= 0x1fffffull;
    x = (x | (x << 32)) & 0x1f00000000ffffull;
    x = (x | (x << 16)) & 0x1f0000ff0000ffull;
    x = (x | (x << 8)) & 0x100f00f00f00f00full;
    x = (x | (x << 4)) & 0x10c30c30c30c30c3ull;
    x = (x | (x << 2)) & 0x1249249249249249ull;
    return x;
}

__device__ __forceinline__ uint32_t quantise21(float p)
{
    float q = p * 2097152.0f;
    q = (q < 0.0f) ? 0.0f : q;
    q = (2097151.0f < q) ? 2097151.0f : q;
    return (q != q) ? 0u : (uint32_t)q;
}

// h[bin] += 1 for every active lane, one LDS atomic per run of consecutive
// active lanes with the same bin: consecutive faces lie close together, so
// the high digits of neighbouring lanes mostly agree, and atomics of a wave
// to one address would serialise.
__device__ __forceinline__ void hist_add(uint32_t* h, uint32_t bin, bool active)
{
    const uint32_t lane = threadIdx.x & 63u;
    // the bin of the lane below (wave_shr:1; lane 0 reads its own and is always a head)
    const uint32_t below = (uint32_t)__builtin_amdgcn_update_dpp((int)bin, (int)bin, 0x138, 0xf, 0xf, false);
    const unsigned long long act = __ballot(active);
    const bool below_active = lane > 0 && ((act >> (lane - 1u)) & 1ull);
    const bool head = active && (!below_active || below != bin);
    const unsigned long long heads = __ballot(head);
    if (head) {
        // the run ends at the next head or the next inactive lane
        const unsigned long long above = (lane == 63u) ? 0ull : ~0ull << (lane + 1u);
        const unsigned long long stop = (heads | ~act) & above;
        const uint32_t end = stop ? (uint32_t)__builtin_ctzll(stop) : 64u;
        atomicAdd(&h[bin], end - lane);
    }
}

// keys_hi == null: 30-bit keys and the histograms of 4 8-bit digits (hbits 8)
// or of 3 10-bit digits (hbits 10); else 63-bit keys split into keys (low
// word) and keys_hi (high word) and 8 8-bit digit histograms. Digit d's
// histogram is ghist[d << hbits .. (d + 1) << hbits), in `hreps` copies OI_HIST_WORDS
// apart (a workgroup adds to copy blockIdx.x mod hreps; a reader sums them).
// Bound by its chain of waits (faces, vertices, box, LDS histograms, additions to the
// shared ones): with 256 threads of 8 faces each, the box folded before the first
// load and one shared histogram, 13K faces took 14 us and 1M 24; 16 waves of 1 to 4
// faces a lane take 5.8 and 13.
template <int NJ>
__global__ void __launch_bounds__(OI_MORTON_T)
k_morton(BuildTab T, const float* __restrict__ partials, uint32_t* __restrict__ keys, uint32_t* __restrict__ keys_hi,
         uint32_t* __restrict__ ghist, uint32_t hstride, uint32_t hreps, uint32_t* __restrict__ fmesh, uint32_t hbits)
{
    __shared__ uint32_t s_h[OI_HIST_WORDS];
    __shared__ float s_v[OI_BLOCK / 64][6];
    const uint32_t tid = threadIdx.x;
    const uint2 it = T.item();
    const oi_build_desc D = T.mesh(it.x);
    Xf X;
    X.load(D.xf);
    const bool h10 = hbits == 10u;
    const uint32_t nd = keys_hi ? 8u : h10 ? 3u : 4u;
    const uint32_t f0 = it.y * (OI_MORTON_T * NJ);
    const uint32_t f1 = min(D.F, f0 + OI_MORTON_T * NJ);  // f0 < f1: a work item holds a face
    // a thread's faces i = f0 + tid + 1024 j: every face load is issued, then
    // every vertex load, and while these are on their way the mesh's box is
    // folded; then the keys are formed. Faces past f1 load face f0 and are dropped
    uint32_t fv[NJ][3];
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        const uint32_t i = f0 + tid + (uint32_t)j * OI_MORTON_T;
        oi_ld3(D.faces, i < f1 ? i : f0, fv[j]);
    }
    // the mesh's partial boxes (at most OI_BLOCK of them), folded in order and
    // then with the default box (+-FLT_MAX) in front
    const float* part = partials ? partials + 6u * D.pbase : D.box + 6;
    float bmn[3], bmx[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        bmn[k] = (tid < D.nparts) ? oi_g(part)[6u * tid + k] : __builtin_inff();
        bmx[k] = (tid < D.nparts) ? oi_g(part)[6u * tid + 3 + k] : -__builtin_inff();
    }
    for (uint32_t i = tid; i < OI_HIST_WORDS; i += OI_MORTON_T) s_h[i] = 0u;
    float p[NJ][9];
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        oi_ld3(D.pos, fv[j][0], &p[j][0]);
        oi_ld3(D.pos, fv[j][1], &p[j][3]);
        oi_ld3(D.pos, fv[j][2], &p[j][6]);
    }
    fold_box(s_v, bmn, bmx);  // (its barrier also orders the cleared histograms)
#pragma unroll
    for (int k = 0; k < 3; k++) {
        bmn[k] = lo_c(__FLT_MAX__, bmn[k]);
        bmx[k] = hi_c(-__FLT_MAX__, bmx[k]);
    }
    ghist += it.x * hstride + (blockIdx.x % hreps) * OI_HIST_WORDS;
    if (it.y == 0 && tid == 0) {
#pragma unroll
        for (int k = 0; k < 3; k++) {
            oi_gw(D.box)[k] = bmn[k];
            oi_gw(D.box)[3 + k] = bmx[k];
        }
    }
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        const uint32_t i = f0 + tid + (uint32_t)j * OI_MORTON_T;
        const bool live = i < f1;
        float a[3], b[3], c[3];
        X.apply(&p[j][0], a);
        X.apply(&p[j][3], b);
        X.apply(&p[j][6], c);
        float u[3];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const float lo = gmin(gmin(a[k], b[k]), c[k]);
            const float hi = gmax(gmax(a[k], b[k]), c[k]);
            const float cen = (lo + hi) * 0.5f;
            const float off = cen - bmn[k];
            const float len = bmx[k] - bmn[k];
            u[k] = off / len;
        }
        uint32_t key, khi = 0;
        if (keys_hi) {
            const uint64_t k64 = (spread21(quantise21(u[0])) << 2) | (spread21(quantise21(u[1])) << 1) |
                                 spread21(quantise21(u[2]));
            key = (uint32_t)k64;
            khi = (uint32_t)(k64 >> 32);
            if (live) oi_gw(keys_hi)[D.fbase + i] = khi;
        } else {
            key = (spread10(quantise10(u[0])) << 2) | (spread10(quantise10(u[1])) << 1) | spread10(quantise10(u[2]));
        }
        if (live) {
            oi_gw(keys)[D.fbase + i] = key;
            if (fmesh) oi_gw(fmesh)[D.fbase + i] = it.x;
        }
        // every lane of the wave takes part (ballots), dead lanes add nothing
        if (h10) {
            // (the low digits of neighbours mostly differ: no runs to join)
            if (live) {
                atomicAdd(&s_h[key & 0x3ffu], 1u);
                atomicAdd(&s_h[1024u + ((key >> 10) & 0x3ffu)], 1u);
            }
            hist_add(s_h + 2048, key >> 20, live);
        } else {
#pragma unroll
            for (int d = 0; d < 4; d++) hist_add(s_h + 256 * d, (key >> (8 * d)) & 0xffu, live);
        }
        if (keys_hi) {
#pragma unroll
            for (int d = 0; d < 4; d++) hist_add(s_h + 256 * (4 + d), (khi >> (8 * d)) & 0xffu, live);
        }
    }
    __syncthreads();
    const uint32_t words = nd << hbits;
    for (uint32_t i = tid; i < words; i += OI_MORTON_T) {
        const uint32_t c = s_h[i];
        if (c) atomicAdd(&ghist[i], c);
    }
}

// ---------------------------------------------------------------------------
// k_sort_pass<DB, ITEMS>: one stable LSD pass over a DB-bit digit (8 or 10),
// onesweep style, over up to OI_SORT_SEGS independent segments of the
// concatenated key arrays (one per tree when several trees are built in one launch).
// A tile is 16 waves x ITEMS rounds x 64 lanes (1,024 to 8,192 keys) of one segment
// in input order (wave w owns keys [64 ITEMS w, 64 ITEMS (w + 1)) of the tile,
// round j lane l holds the 64j + l-th of them). Keys are ranked per wave with DB
// ballots per round (stable: earlier rounds and lower lanes come first), staged
// through LDS in tile-local sorted order and written out in runs. Segment s
// owns the workgroups and tile ids [tile0[s], tile0[s + 1]); a workgroup takes
// its tile from its segment's atomic counter (tile_counter[s]), so every tile
// a look-back waits on is already running, and the look-back ends at the
// segment's own first tile.
// Look-back status word: bits 31:30 = 1 aggregate / 2 inclusive prefix,
// bits 29:0 = count. A tile's word counts from the start of its group of LB_GROUP
// tiles; the group's last tile publishes the group's word (row tiles + group, from
// the start of the segment), so that a tile reads the words of its group before it,
// and then group words. A digit that no key of the segment has (its histogram
// entry is 0) is neither published nor looked back on. Values default to the
// key's index in the concatenated arrays. With key_of_val the key of a value v
// is key_of_val[v] (a batch's mesh-id passes: a stable partition of the
// Morton-sorted faces of all meshes back into their meshes).
// A pass is a chain of waits: of 25 us on 1M keys (123 tiles of 8,192, one window of
// look-back after the other over all tiles) the ranking took 5, the look-back 9, the
// keys' and counts' loads 3.5. Now 19 (245 tiles of 4,096), and 7.9 instead of 14 on
// 13K keys (13 tiles, before 2). The statuses cross XCDs and their traffic counts: with
// 16 instead of 8 per round trip a build of 1M triangles took 111 instead of 105 us,
// and with groups of 16 and 8 tiles 99.
// ---------------------------------------------------------------------------
#define RS_WAVES 16
#define RS_THREADS (64 * RS_WAVES)
#define RS_ITEMS_MAX 8
#define LB_AGG (1u << 30)
#define LB_PRE (2u << 30)
#define LB_CNT 0x3fffffffu
#define LB_WIN 8  // look-back statuses loaded per round trip
#define LB_GROUP OI_SORT_GROUP  // tiles of a look-back group
#define OI_SORT_SEGS 4

struct SortSegs {
    uint32_t ns;                        // segments, 1..OI_SORT_SEGS
    uint32_t hstride;                   // words between the segments' digit histograms
    uint32_t tile0[OI_SORT_SEGS + 1];   // segment s owns tiles [tile0[s], tile0[s + 1])
    uint32_t base[OI_SORT_SEGS];        // its first key in the concatenated arrays
    uint32_t n[OI_SORT_SEGS];           // its keys
};

// exclusive prefixes over the workgroup of two counts per thread
__device__ __forceinline__ uint2 block_excl_scan2(uint2 v, uint2* s_wsum)
{
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint2 x = make_uint2(oi_wave_scan_incl(v.x), oi_wave_scan_incl(v.y));
    if (lane == 63) s_wsum[wave] = x;
    __syncthreads();
    uint2 before = make_uint2(x.x - v.x, x.y - v.y);
#pragma unroll
    for (int w = 0; w < RS_WAVES; w++) {
        const uint2 t = s_wsum[w];
        before.x += (w < (int)wave) ? t.x : 0u;
        before.y += (w < (int)wave) ? t.y : 0u;
    }
    return before;
}

// Sum of digit `d` over the `n` entries (tiles of a group, or groups) before entry
// `at`. The statuses of LB_WIN entries at - 1, at - 2, ... are loaded in one round trip
// (the loads cross XCDs) and consumed in order, summing counts until an inclusive
// prefix or the n-th; an entry not yet published ends the window, which is loaded
// again from there.
template <int DB>
__device__ __forceinline__ uint32_t look_back(const uint32_t* lookback, uint32_t at, uint32_t n, uint32_t d)
{
    uint32_t sum = 0;
    while (n) {
        uint32_t st[LB_WIN];
#pragma unroll
        for (uint32_t w = 0; w < LB_WIN; w++)
            st[w] = w < n ? ld_acq_relaxed(lookback + ((at - 1u - w) << DB) + d) : 0u;
        uint32_t used = 0;
#pragma unroll
        for (uint32_t w = 0; w < LB_WIN; w++) {
            if (used != w || w >= n) continue;
            const uint32_t fl = st[w] & ~LB_CNT;
            if (fl == 0u) continue;
            sum += st[w] & LB_CNT;
            used = w + 1u;
            if (fl == LB_PRE) n = w + 1u;  // none before it is wanted
        }
        at -= used;
        n -= used;
        if (n && used != LB_WIN) __builtin_amdgcn_s_sleep(1);
    }
    return sum;
}

template <int DB, int ITEMS>
__global__ void __launch_bounds__(RS_THREADS)
k_sort_pass(const uint32_t* __restrict__ keys_in, const uint32_t* __restrict__ vals_in,
            uint32_t* __restrict__ keys_out, uint32_t* __restrict__ vals_out, SortSegs S, uint32_t shift,
            const uint32_t* __restrict__ ghist, uint32_t hreps, uint32_t* lookback, uint32_t* lookback_next,
            uint32_t* tile_counter, const uint32_t* __restrict__ key_of_val)
{
    constexpr uint32_t NB = 1u << DB;  // bins; at most RS_THREADS
    constexpr uint32_t TILE = RS_THREADS * ITEMS;
    static_assert(NB <= RS_THREADS, "one digit per thread");
    __shared__ uint32_t s_tile;
    __shared__ uint32_t s_whist[RS_WAVES][NB];
    __shared__ uint32_t s_lstart[NB];
    __shared__ uint32_t s_gbase[NB];
    __shared__ uint2 s_wsum[RS_WAVES];
    __shared__ uint32_t s_keys[TILE];
    __shared__ uint32_t s_vals[TILE];

    // threads tid < NB also own digit tid
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const bool dig = tid < NB;
    // the workgroup's segment (constant indices keep the argument block out
    // of scratch memory)
    uint32_t seg = 0, seg0 = S.tile0[0], sbase = S.base[0], n = S.n[0];
#pragma unroll
    for (int k = 1; k < OI_SORT_SEGS; k++) {
        if (k < (int)S.ns && blockIdx.x >= S.tile0[k]) {
            seg = k;
            seg0 = S.tile0[k];
            sbase = S.base[k];
            n = S.n[k];
        }
    }
    if (tid == 0)
        s_tile = __hip_atomic_fetch_add(tile_counter + seg, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (uint32_t i = tid; i < RS_WAVES * NB; i += RS_THREADS) (&s_whist[0][0])[i] = 0u;
    __syncthreads();
    const uint32_t tile = s_tile;
    const uint32_t gt = seg0 + tile;  // tile id over all segments
    const uint32_t base = tile * TILE;

    uint32_t k[ITEMS], v[ITEMS], rk[ITEMS];
    const uint32_t wbase = base + wave * (64u * ITEMS);
#pragma unroll
    for (int j = 0; j < ITEMS; j++) {
        const uint32_t idx = wbase + 64u * j + lane;
        const bool ok = idx < n;
        const uint32_t gi = sbase + idx;
        v[j] = ok ? (vals_in ? vals_in[gi] : gi) : 0u;
        k[j] = ok ? (key_of_val ? key_of_val[v[j]] : keys_in[gi]) : 0u;
    }
    // (the digit's count over the segment is on its way with the keys)
    uint32_t hcnt = 0;
    if (dig) {
        const uint32_t* h = ghist + seg * S.hstride + tid;
        if (hreps == OI_HIST_REPS) {
            uint32_t c[OI_HIST_REPS];
#pragma unroll
            for (uint32_t r = 0; r < OI_HIST_REPS; r++) c[r] = h[r * OI_HIST_WORDS];
#pragma unroll
            for (uint32_t r = 0; r < OI_HIST_REPS; r++) hcnt += c[r];
        } else {
            hcnt = h[0];
        }
        if (lookback_next) {
            lookback_next[gt * NB + tid] = 0u;
            if (tile % LB_GROUP == 0u)
                lookback_next[(S.tile0[S.ns] + seg0 / LB_GROUP + seg + tile / LB_GROUP) * NB + tid] = 0u;
        }
    }
    const unsigned long long lt = (1ull << lane) - 1ull;
#pragma unroll
    for (int j = 0; j < ITEMS; j++) {
        const uint32_t idx = wbase + 64u * j + lane;
        const bool ok = idx < n;
        const uint32_t d = (k[j] >> shift) & (NB - 1u);
        const unsigned long long live = __ballot(ok);
        uint32_t p0 = (uint32_t)live, p1 = (uint32_t)(live >> 32);
#pragma unroll
        for (int b = 0; b < DB; b++) {
            // lanes whose bit b equals this lane's
            const uint32_t bit = (uint32_t)((int32_t)(d << (31 - b)) >> 31);
            const unsigned long long m = __ballot(bit != 0u);
            p0 &= ~((uint32_t)m ^ bit);
            p1 &= ~((uint32_t)(m >> 32) ^ bit);
        }
        const unsigned long long peers = ((unsigned long long)p1 << 32) | p0;
        const uint32_t prev = s_whist[wave][d];
        const uint32_t cnt = (uint32_t)__popcll(peers);
        rk[j] = prev + (uint32_t)__popcll(peers & lt);
        const bool leader = ok && ((peers & lt) == 0ull);
        if (leader) s_whist[wave][d] = prev + cnt;
    }
    __syncthreads();
    // per-wave exclusive offsets and tile totals (thread tid owns digit tid)
    uint32_t tot = 0;
    if (dig) {
#pragma unroll
        for (int w = 0; w < RS_WAVES; w++) {
            const uint32_t c = s_whist[w][tid];
            s_whist[w][tid] = tot;
            tot += c;
        }
    }
    // publish this tile's count (a group's first tile has none before it)
    const bool live = dig && hcnt != 0u;
    if (live) st_relaxed(lookback + gt * NB + tid, (tile % LB_GROUP == 0 ? LB_PRE : LB_AGG) | tot);
    // exclusive prefixes of the tile's and of the segment's digit counts
    const uint2 ex = block_excl_scan2(make_uint2(tot, hcnt), s_wsum);
    if (dig) s_lstart[tid] = ex.x;
    // look-back for digit tid: the group's tiles before this one, then, in the
    // group's last tile, publishing the group's count, the groups before it
    uint32_t excl = 0;
    if (live) {
        const uint32_t in_group = tile % LB_GROUP;
        excl = look_back<DB>(lookback, gt, in_group, tid);
        const uint32_t g0 = seg0 / LB_GROUP + seg, grp = tile / LB_GROUP;
        uint32_t* const groups = lookback + (uint64_t)S.tile0[S.ns] * NB;
        uint32_t* const mine = groups + (g0 + grp) * NB + tid;
        const bool last = in_group == LB_GROUP - 1u;
        if (last) st_relaxed(mine, (grp == 0 ? LB_PRE : LB_AGG) | (excl + tot));
        if (grp > 0) {
            const uint32_t before = look_back<DB>(groups, g0 + grp, grp, tid);
            excl += before;
            if (last) st_relaxed(mine, LB_PRE | (excl + tot));
        }
    }
    if (dig) s_gbase[tid] = sbase + ex.y + excl;
    __syncthreads();
    // stage in tile-local sorted order
#pragma unroll
    for (int j = 0; j < ITEMS; j++) {
        const uint32_t idx = wbase + 64u * j + lane;
        if (idx < n) {
            const uint32_t d = (k[j] >> shift) & (NB - 1u);
            const uint32_t lp = s_lstart[d] + s_whist[wave][d] + rk[j];
            s_keys[lp] = k[j];
            s_vals[lp] = v[j];
        }
    }
    __syncthreads();
    const uint32_t cnt_tile = (n - base < TILE) ? (n - base) : TILE;
    for (uint32_t i = tid; i < cnt_tile; i += RS_THREADS) {
        const uint32_t key = s_keys[i];
        const uint32_t d = (key >> shift) & (NB - 1u);
        const uint32_t g = s_gbase[d] + (i - s_lstart[d]);
        if (keys_out) keys_out[g] = key;
        vals_out[g] = s_vals[i];
    }
}

// ---------------------------------------------------------------------------
// k_reduce: leaves + bottom-up reduce.
// Stage 1: work item (m, w) owns the subtree of mesh m of height
// h = min(L, 8 + log2 M) rooted at level L - h, position w (its 2^h leaves).
// Each thread computes M consecutive leaves and folds them log2(M) levels in
// registers; the 256 results climb the remaining levels through LDS. Every
// level of the subtree is a contiguous run of real nodes: it is staged in LDS
// and written out as whole cache lines from consecutive lanes (one thread
// writing its own 24-byte nodes would leave lines partially written). Every
// real node is written once, at its real index.
// Stage 2 (k_reduce_apex, a second launch): one workgroup per mesh reads the
// stage-1 roots and climbs to the root in chunks of up to 2^11 nodes.
// A parent is real iff its left child is; with no real right child the
// parent equals the left child (oibvh.cu:139-146).
// ---------------------------------------------------------------------------
struct Box6 {
    float v[6];
};

__device__ __forceinline__ void box_merge_into(Box6& a, const Box6& r)
{
#pragma unroll
    for (int k = 0; k < 3; k++) {
        a.v[k] = gmin(a.v[k], r.v[k]);
        a.v[3 + k] = gmax(a.v[3 + k], r.v[3 + k]);
    }
}

__device__ __forceinline__ Box6 load_node(const float* nodes, uint32_t r)
{
    const OI_GLOBAL float* p = oi_g(nodes) + 6ull * r;
    Box6 o;
#pragma unroll
    for (int k = 0; k < 6; k++) o.v[k] = p[k];
    return o;
}

template <class Tab>
struct ReduceArgs {
    Tab T;  // first (WideTab)
    const uint32_t* vals;  // build: Morton-sorted face ids (fbase + face); null: refit over sfaces
    uint32_t write_perm;   // build: also write perm (faces local to the mesh)
    uint32_t nwork;        // k_reduce_w: work items (0: one per workgroup)
};

struct LeafLoad {
    const oi_build_desc& D;
    const Xf& X;
    const uint32_t* vals;
    uint32_t write_perm;
    __device__ __forceinline__ Box6 operator()(uint32_t p) const
    {
        uint32_t f[3];
        if (vals) {
            const uint32_t fi = oi_g(vals)[D.fbase + p] - D.fbase;
            oi_ld3(D.faces, fi, f);
            OI_GLOBAL uint32_t* q = oi_gw(D.sfaces) + 3ull * p;
            q[0] = f[0];
            q[1] = f[1];
            q[2] = f[2];
            if (write_perm) oi_gw(D.perm)[p] = fi;
        } else {
            oi_ld3(D.sfaces, p, f);
        }
        float a[3], b[3], c[3];
        X.vertex(D.pos, f[0], a);
        X.vertex(D.pos, f[1], b);
        X.vertex(D.pos, f[2], c);
        Box6 r;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            r.v[k] = gmin(gmin(a[k], b[k]), c[k]);
            r.v[3 + k] = gmax(gmax(a[k], b[k]), c[k]);
        }
        return r;
    }
};

struct NodeLoad {
    const float* nodes;
    uint32_t lvl_start;
    __device__ __forceinline__ Box6 operator()(uint32_t p) const { return load_node(nodes, lvl_start + p); }
};

// LDS staging of one level's nodes in node layout (6 floats per node)
__device__ __forceinline__ void put_box(float* stage, uint32_t i, const Box6& b)
{
    float2* d = reinterpret_cast<float2*>(stage + 6u * i);
    d[0] = make_float2(b.v[0], b.v[1]);
    d[1] = make_float2(b.v[2], b.v[3]);
    d[2] = make_float2(b.v[4], b.v[5]);
}
__device__ __forceinline__ Box6 get_box(const float* stage, uint32_t i)
{
    const float2* d = reinterpret_cast<const float2*>(stage + 6u * i);
    const float2 a = d[0], b = d[1], c = d[2];
    Box6 o;
    o.v[0] = a.x;
    o.v[1] = a.y;
    o.v[2] = b.x;
    o.v[3] = b.y;
    o.v[4] = c.x;
    o.v[5] = c.y;
    return o;
}

// Write `count` staged nodes to real index `first` onwards as one contiguous
// run of float2 (whole cache lines from consecutive lanes); the block's
// threads share the copy.
__device__ __forceinline__ void copy_out(float* nodes, uint32_t first, uint32_t count, const float* stage)
{
    OI_GLOBAL float* dst = oi_gw(nodes) + 6ull * first;
    const float2* src = reinterpret_cast<const float2*>(stage);
    for (uint32_t i = threadIdx.x; i < 3u * count; i += OI_BLOCK) {
        const float2 v = src[i];
        dst[2u * i] = v.x;
        dst[2u * i + 1u] = v.y;
    }
}

// LDS for one subtree reduce with M leaves per thread: two staging buffers
// used in turn, 256 M and max(128 M, 256) nodes
template <int M>
struct StageSize {
    static constexpr uint32_t n0 = 256u * M;
    static constexpr uint32_t n1 = (128u * M > 256u) ? 128u * M : 256u;
    static constexpr uint32_t floats = 6u * (n0 + n1);
};

// Reduce the subtree whose bottom level is lc, h levels up, root position w
// at level lc - h. Requires 2^h <= 256 * M and stage >= StageSize<M>::floats.
// Each level is staged in LDS and written out contiguously; consecutive
// levels use the two buffers in turn, so one barrier per level orders both
// the next level's reads and the previous buffer's reuse.
// Returns with every node of the subtree written; ends with a barrier.
template <int M, class Load>
__device__ void reduce_subtree(const Load& load, float* nodes, uint32_t L, uint32_t vl, uint32_t lc, uint32_t h,
                               uint32_t w, float* stage)
{
    constexpr uint32_t LGM = (M == 1) ? 0 : (M == 2) ? 1 : (M == 4) ? 2 : 3;
    float* const s0 = stage;
    float* const s1 = stage + 6u * StageSize<M>::n0;
    const uint32_t tid = threadIdx.x;
    const bool act = (tid * M) < (1u << h);
    const uint32_t c0 = (w << h) + tid * M;
    uint32_t ncnt = oi_lvl_cnt(lc, L, vl);
    Box6 b[M];
#pragma unroll
    for (int j = 0; j < M; j++)
        if (act && c0 + j < ncnt) {
            b[j] = load(c0 + j);
            put_box(s0, tid * M + j, b[j]);
        }
    __syncthreads();
    copy_out(nodes, oi_lvl_start(lc, L, vl) + (w << h), min(1u << h, ncnt - (w << h)), s0);
    uint32_t cur = 0;  // buffer holding the last level
    const uint32_t hl = (h < LGM) ? h : LGM;
    uint32_t l = lc;
#pragma unroll
    for (uint32_t s = 1; s <= LGM; s++) {
        if (s <= hl) {
            const uint32_t cc = ncnt;  // real count of the child level
            l -= 1;
            ncnt = oi_lvl_cnt(l, L, vl);
            cur ^= 1u;
#pragma unroll
            for (uint32_t j = 0; j < (uint32_t)(M >> s); j++) {
                const uint32_t q = (c0 >> s) + j;
                if (act && 2u * q < cc) {
                    Box6 x = b[2 * j];
                    if (2u * q + 1u < cc) box_merge_into(x, b[2 * j + 1]);
                    b[j] = x;
                    put_box(cur ? s1 : s0, tid * (uint32_t)(M >> s) + j, x);
                }
            }
            __syncthreads();
            const uint32_t f = w << (h - s);
            copy_out(nodes, oi_lvl_start(l, L, vl) + f, min(1u << (h - s), ncnt - f), cur ? s1 : s0);
        }
    }
    const uint32_t hs = h - hl;
    // LDS climb: slot t of the current buffer holds node (w << hs) + t of level l
    for (uint32_t s = 1; s <= hs; s++) {
        const uint32_t cc = ncnt;
        l -= 1;
        ncnt = oi_lvl_cnt(l, L, vl);
        const uint32_t width = 1u << (hs - s);
        const uint32_t f = w << (hs - s);
        const uint32_t q = f + tid;
        const float* src = cur ? s1 : s0;
        float* dst = cur ? s0 : s1;
        if (tid < width && 2u * q < cc) {
            Box6 x = get_box(src, 2u * tid);
            if (2u * q + 1u < cc) box_merge_into(x, get_box(src, 2u * tid + 1u));
            put_box(dst, tid, x);
        }
        cur ^= 1u;
        __syncthreads();
        copy_out(nodes, oi_lvl_start(l, L, vl) + f, min(width, ncnt - f), dst);
    }
    __syncthreads();
}

template <int M, class Tab>
__global__ void __launch_bounds__(OI_BLOCK) k_reduce(ReduceArgs<Tab> a)
{
    __shared__ float stage[StageSize<M>::floats];
    constexpr uint32_t LGM = (M == 1) ? 0 : (M == 2) ? 1 : (M == 4) ? 2 : 3;
    const uint2 it = a.T.item();
    const oi_build_desc D = a.T.mesh(it.x);
    Xf X;
    X.load(D.xf);
    const uint32_t L = D.L, vl = D.vl;
    const uint32_t h = (L < 8 + LGM) ? L : 8 + LGM;
    LeafLoad ll{D, X, a.vals, a.write_perm};
    reduce_subtree<M>(ll, D.nodes, L, vl, L, h, it.y, stage);
}

// ---------------------------------------------------------------------------
// k_reduce_w: stage 1 with one subtree per wave (the alternative to
// k_reduce's one subtree per workgroup). Wave ws owns the 2^hw leaves
// [ws 2^hw, (ws + 1) 2^hw) of the leaf level, hw = min(L, 8); lane l holds
// leaves 64k + l (k < 4), so every face, vertex and node access of one
// instruction covers consecutive leaves. Each level is staged in the wave's
// own LDS and written out as a contiguous run; the wave climbs hw levels
// with no workgroup barrier. The workgroup's waves then meet once, and
// thread 0 merges their roots hb = min(L - hw, 2) levels further, so stage 1
// ends at level L - hw - hb as k_reduce with M = 4 does (apex lgm = 2).
// ---------------------------------------------------------------------------
#define RW_LG 8
#define RW_W (1u << RW_LG)

// Write `count` staged nodes (at most CMAX) to real index `first` onwards as
// one contiguous run of float2 per lane; all LDS reads are issued before the
// first store.
template <uint32_t CMAX>
__device__ __forceinline__ void wave_copy_out(float* nodes, uint32_t first, uint32_t count, const float* stage,
                                              uint32_t lane)
{
    constexpr uint32_t IT = (3u * CMAX + 63u) / 64u;
    OI_GLOBAL float* dst = oi_gw(nodes) + 6ull * first;
    const float2* src = reinterpret_cast<const float2*>(stage);
    const uint32_t n = 3u * count;
    float2 v[IT];
#pragma unroll
    for (uint32_t it = 0; it < IT; it++) {
        const uint32_t i = lane + 64u * it;
        if (i < n) v[it] = src[i];
    }
#pragma unroll
    for (uint32_t it = 0; it < IT; it++) {
        const uint32_t i = lane + 64u * it;
        if (i < n) {
            dst[2u * i] = v[it].x;
            dst[2u * i + 1u] = v[it].y;
        }
    }
}

// One level of a wave climb in place: slots 2t, 2t + 1 of stage (the child
// level, first node 2f, cc real) -> slot t (first node f). Every read of the
// level precedes every write.
template <uint32_t WMAX>
__device__ __forceinline__ void wave_level(float* stage, uint32_t width, uint32_t f, uint32_t cc, uint32_t lane)
{
    constexpr uint32_t IT = (WMAX + 63u) / 64u;
    Box6 x[IT], y[IT];
    bool has[IT], two[IT];
#pragma unroll
    for (uint32_t it = 0; it < IT; it++) {
        const uint32_t t = lane + 64u * it;
        const uint32_t q = f + t;
        has[it] = t < width && 2u * q < cc;
        two[it] = has[it] && 2u * q + 1u < cc;
        if (has[it]) x[it] = get_box(stage, 2u * t);
        if (two[it]) y[it] = get_box(stage, 2u * t + 1u);
    }
    oi_wave_fence();
#pragma unroll
    for (uint32_t it = 0; it < IT; it++) {
        if (two[it]) box_merge_into(x[it], y[it]);
        if (has[it]) put_box(stage, lane + 64u * it, x[it]);
    }
    oi_wave_fence();
}

// the refit's sorted faces of the leaves a wave owns
__device__ __forceinline__ void wave_sfaces(const oi_build_desc& D, uint32_t f0, uint32_t hw, uint32_t nleaf,
                                            uint32_t lane, uint32_t (&f)[RW_W / 64][3])
{
#pragma unroll
    for (int k = 0; k < RW_W / 64; k++) {
        const uint32_t off = 64u * k + lane;
        const uint32_t p = f0 + off;
        const bool ok = off < (1u << hw) && p < nleaf;
        oi_ld3(D.sfaces, ok ? p : f0, f[k]);  // in range; only ok results are kept
    }
}

// the leaf boxes of a wave's faces f (vertex gathers, model matrix if XF),
// staged at their leaf slots
template <bool XF>
__device__ __forceinline__ void wave_boxes(const oi_build_desc& D, uint32_t f0, uint32_t hw, uint32_t nleaf,
                                           uint32_t lane, float* stage, const uint32_t (&f)[RW_W / 64][3])
{
    constexpr int K = RW_W / 64;
    float m[16];
    if constexpr (XF) {
#pragma unroll
        for (int k = 0; k < 16; k++) m[k] = oi_g(D.xf)[k];
    }
    float v[K][3][3];
#pragma unroll
    for (int k = 0; k < K; k++)
#pragma unroll
        for (int j = 0; j < 3; j++) {
            if constexpr (XF) {
                float q[3];
                oi_ld3(D.pos, f[k][j], q);
                oi_xform(m, q[0], q[1], q[2], v[k][j]);
            } else {
                oi_ld3(D.pos, f[k][j], v[k][j]);
            }
        }
#pragma unroll
    for (int k = 0; k < K; k++) {
        Box6 r;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            r.v[c] = gmin(gmin(v[k][0][c], v[k][1][c]), v[k][2][c]);
            r.v[3 + c] = gmax(gmax(v[k][0][c], v[k][1][c]), v[k][2][c]);
        }
        const uint32_t off = 64u * k + lane;
        if (off < (1u << hw) && f0 + off < nleaf) put_box(stage, off, r);
    }
}

// The leaf level of one wave subtree into stage (node layout): every load is
// issued before any box is formed. BUILD reads the sorted face ids and writes
// sfaces and perm; XF applies the model matrix. Both are compile-time, so the
// loads form one straight run.
template <bool BUILD, bool XF, class Tab>
__device__ __forceinline__ void wave_leaves(const ReduceArgs<Tab>& A, const oi_build_desc& D, uint32_t f0, uint32_t hw,
                                            uint32_t nleaf, uint32_t lane, float* stage)
{
    constexpr int K = RW_W / 64;
    uint32_t f[K][3], fid[K];
    if constexpr (BUILD) {
#pragma unroll
        for (int k = 0; k < K; k++) {
            const uint32_t off = 64u * k + lane;
            const uint32_t p = f0 + off;
            const uint32_t pc = (off < (1u << hw) && p < nleaf) ? p : f0;  // only in-range results are kept
            fid[k] = oi_g(A.vals)[D.fbase + pc] - D.fbase;
            oi_ld3(D.faces, fid[k], f[k]);
        }
    } else {
        wave_sfaces(D, f0, hw, nleaf, lane, f);
    }
    wave_boxes<XF>(D, f0, hw, nleaf, lane, stage, f);
    if constexpr (BUILD) {
#pragma unroll
        for (int k = 0; k < K; k++) {
            const uint32_t off = 64u * k + lane;
            const uint32_t p = f0 + off;
            if (off < (1u << hw) && p < nleaf) {
                OI_GLOBAL uint32_t* q = oi_gw(D.sfaces) + 3ull * p;
                q[0] = f[k][0];
                q[1] = f[k][1];
                q[2] = f[k][2];
                if (A.write_perm) oi_gw(D.perm)[p] = fid[k];
            }
        }
    }
}

// climb levels S..8 of a full-height (hw = 8) wave subtree; level s has
// 256 >> s nodes
template <uint32_t S>
__device__ __forceinline__ void wave_climb8(float* stage, float* nodes, uint32_t L, uint32_t vl, uint32_t f0,
                                            uint32_t cc, uint32_t lane)
{
    if constexpr (S <= RW_LG) {
        constexpr uint32_t WIDTH = RW_W >> S;
        const uint32_t l = L - S;
        const uint32_t ncnt = oi_lvl_cnt(l, L, vl);
        const uint32_t f = f0 >> S;
        wave_level<WIDTH>(stage, WIDTH, f, cc, lane);
        wave_copy_out<WIDTH>(nodes, oi_lvl_start(l, L, vl) + f, min(WIDTH, ncnt - f), stage, lane);
        wave_climb8<S + 1>(stage, nodes, L, vl, f0, ncnt, lane);
    }
}

// a wave's part of one work item once its leaf boxes are staged: write the
// leaves, climb hw levels (wave 0 .. 2^hb - 1 of the workgroup)
__device__ __forceinline__ void wave_climb_all(const oi_build_desc& D, uint32_t f0, uint32_t hw, uint32_t nleaf,
                                               uint32_t lane, float* W)
{
    const uint32_t L = D.L, vl = D.vl;
    oi_wave_fence();
    wave_copy_out<RW_W>(D.nodes, oi_lvl_start(L, L, vl) + f0, min(1u << hw, nleaf - f0), W, lane);
    if (hw == RW_LG) {
        wave_climb8<1>(W, D.nodes, L, vl, f0, nleaf, lane);
    } else {
        // short trees: the same climb with run-time widths
        uint32_t ncnt = nleaf;
        for (uint32_t s = 1; s <= hw; s++) {
            const uint32_t l = L - s;
            const uint32_t cc = ncnt;
            ncnt = oi_lvl_cnt(l, L, vl);
            const uint32_t width = 1u << (hw - s);
            const uint32_t f = f0 >> s;
            wave_level<RW_W / 2>(W, width, f, cc, lane);
            wave_copy_out<RW_W / 2>(D.nodes, oi_lvl_start(l, L, vl) + f, min(width, ncnt - f), W, lane);
        }
    }
}

// thread 0 merges the wave roots of work item `it` (slot 0 of each wave's
// stage) hb levels further; called by every thread after a barrier
__device__ __forceinline__ void item_top(const oi_build_desc& D, uint2 it, uint32_t hw, uint32_t hb,
                                         float (*S)[6 * RW_W])
{
    if (threadIdx.x != 0) return;
    const uint32_t L = D.L, vl = D.vl;
    const uint32_t lw = L - hw;
    uint32_t cc = oi_lvl_cnt(lw, L, vl);
    Box6 m[2];
    const uint32_t n1 = 1u << (hb - 1u);  // nodes of the first merged level
#pragma unroll
    for (uint32_t t = 0; t < 2u; t++) {
        const uint32_t q = (it.y << (hb - 1u)) + t;
        if (t < n1 && 2u * q < cc) {
            Box6 x = get_box(S[2u * t], 0);
            if (2u * q + 1u < cc) box_merge_into(x, get_box(S[2u * t + 1u], 0));
            m[t] = x;
            OI_GLOBAL float* o = oi_gw(D.nodes) + 6ull * (oi_lvl_start(lw - 1u, L, vl) + q);
#pragma unroll
            for (int c = 0; c < 6; c++) o[c] = x.v[c];
        }
    }
    if (hb == 2) {
        cc = oi_lvl_cnt(lw - 1u, L, vl);
        const uint32_t q = it.y;
        if (2u * q < cc) {
            Box6 x = m[0];
            if (2u * q + 1u < cc) box_merge_into(x, m[1]);
            OI_GLOBAL float* o = oi_gw(D.nodes) + 6ull * (oi_lvl_start(lw - 2u, L, vl) + q);
#pragma unroll
            for (int c = 0; c < 6; c++) o[c] = x.v[c];
        }
    }
}

// what one wave of a workgroup does for work item `it` (1024 leaves: a
// subtree per wave, then up to two levels above them)
struct WaveItem {
    oi_build_desc D;
    uint32_t hw, hb, f0, nleaf;
    bool on;  // this wave owns leaves of the item
};
template <class Tab>
__device__ __forceinline__ WaveItem wave_item(const ReduceArgs<Tab>& A, uint2 it, uint32_t wave)
{
    WaveItem w;
    w.D = A.T.mesh(it.x);
    const uint32_t L = w.D.L;
    w.hw = (L < RW_LG) ? L : RW_LG;
    w.hb = (L - w.hw < 2u) ? L - w.hw : 2u;
    w.f0 = ((it.y << w.hb) + wave) << w.hw;
    w.nleaf = oi_lvl_cnt(L, L, w.D.vl);
    w.on = wave < (1u << w.hb) && w.f0 < w.nleaf;
    return w;
}

// one work item; S is the workgroup's staging, free again on return
template <class Tab>
__device__ __forceinline__ void reduce_w_item(const ReduceArgs<Tab>& A, uint2 it, float (*S)[6 * RW_W])
{
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const WaveItem w = wave_item(A, it, wave);
    const oi_build_desc& D = w.D;
    float* W = S[wave];
    if (w.on) {
        if (A.vals) {
            if (D.xf)
                wave_leaves<true, true>(A, D, w.f0, w.hw, w.nleaf, lane, W);
            else
                wave_leaves<true, false>(A, D, w.f0, w.hw, w.nleaf, lane, W);
        } else {
            if (D.xf)
                wave_leaves<false, true>(A, D, w.f0, w.hw, w.nleaf, lane, W);
            else
                wave_leaves<false, false>(A, D, w.f0, w.hw, w.nleaf, lane, W);
        }
        wave_climb_all(D, w.f0, w.hw, w.nleaf, lane, W);
    }
    if (w.hb == 0) return;
    __syncthreads();
    item_top(D, it, w.hw, w.hb, S);
}

template <class Tab>
__global__ void __launch_bounds__(OI_BLOCK) k_reduce_w(ReduceArgs<Tab> A)
{
    __shared__ float S[OI_BLOCK / 64][6 * RW_W];
    reduce_w_item(A, A.T.item(), S);
}

// k_reduce_w for a refit with fewer workgroups than work items (A.nwork):
// each takes items b, b + gridDim.x, ...; the barrier keeps a workgroup's
// next item off S until thread 0 has read the wave roots of this one (hb is
// uniform over the workgroup). A kernel of its own: the loop costs
// registers. (Loading the next item's faces before the current item's
// vertices was measured: the refit was no faster beside a detect, and the
// detect slower.)
template <class Tab>
__global__ void __launch_bounds__(OI_BLOCK) k_reduce_wl(ReduceArgs<Tab> A)
{
    __shared__ float S[OI_BLOCK / 64][6 * RW_W];
    for (uint32_t v = blockIdx.x; v < A.nwork; v += gridDim.x) {
        reduce_w_item(A, A.T.item_at(v, A.nwork), S);
        if (v + gridDim.x < A.nwork) __syncthreads();
    }
}

// Stage 2, one workgroup per mesh: the levels above the stage-1 subtree roots
// (level lc = L - h), in chunks of up to 2^11 nodes per climb, with as many
// nodes per thread as keep all 256 threads busy. A separate launch, so the
// roots written by every stage-1 workgroup are visible without device-scope
// fences.
template <int M>
__device__ __forceinline__ void apex_chunks(const oi_build_desc& D, uint32_t lc, uint32_t h2, float* stage)
{
    const uint32_t nchunk = oi_lvl_cnt(lc - h2, D.L, D.vl);
    NodeLoad nl{D.nodes, oi_lvl_start(lc, D.L, D.vl)};
    for (uint32_t c = 0; c < nchunk; c++) reduce_subtree<M>(nl, D.nodes, D.L, D.vl, lc, h2, c, stage);
}

// Stage 1 leaves more than 2^11 roots of a tree above 2M faces (APEX_MID): one
// workgroup would climb them a chunk after the other, 9 us each. k_reduce_mid climbs
// 8 levels in a workgroup per 256 roots first, and k_reduce_apex starts above them:
// a frame of the folded cloth of 8.4M faces 1,695 -> 1,675 us.
#define APEX_MID 11u
template <class Tab>
__global__ void __launch_bounds__(OI_BLOCK) k_reduce_mid(ReduceArgs<Tab> a, uint32_t lgm)
{
    __shared__ float stage[StageSize<1>::floats];
    const uint2 it = a.T.item();
    const oi_build_desc D = a.T.mesh(it.x);
    const uint32_t lc = D.L - (8u + lgm);  // (launched for meshes with lc > APEX_MID)
    NodeLoad nl{D.nodes, oi_lvl_start(lc, D.L, D.vl)};
    reduce_subtree<1>(nl, D.nodes, D.L, D.vl, lc, 8u, it.y, stage);
}

// zeroed level counts and result counters for the detect that follows
// (the work of the collide side's k_seed, one workgroup)
__device__ __forceinline__ void seed_counters(const oi_seed_args& s)
{
    const uint32_t i = threadIdx.x;
    if (i < s.n_counts) s.counts[i] = (i == 0) ? s.n0 : 0u;
    oi_reset_ctl(s.ctl, i, s.reset_sticky);
}

// with seed.counts set, the launch has one more workgroup, which resets the
// counters of the detect that follows instead of climbing a mesh. Work items
// are numbered through the XCD remap (BuildTab::item), so the extra workgroup
// is the one whose remapped index is the last: the others then cover exactly
// the items 0 .. n - 1 of the work list.
template <class Tab>
__global__ void __launch_bounds__(OI_BLOCK) k_reduce_apex(ReduceArgs<Tab> a, uint32_t lgm, uint32_t mid, oi_seed_args seed)
{
    __shared__ float stage[StageSize<8>::floats];
    if (seed.counts && oi_xcd_remap(blockIdx.x, gridDim.x) == gridDim.x - 1) {
        seed_counters(seed);
        return;
    }
    const uint2 it = a.T.item();
    const oi_build_desc D = a.T.mesh(it.x);
    const uint32_t L = D.L;
    const uint32_t h = (L < 8 + lgm) ? L : 8 + lgm;
    uint32_t lc = L - h;
    if (mid && lc > APEX_MID) lc -= 8u;  // k_reduce_mid has climbed them
    while (lc > 0) {
        const uint32_t h2 = (lc < 11u) ? lc : 11u;
        if (h2 <= 8)
            apex_chunks<1>(D, lc, h2, stage);
        else if (h2 == 9)
            apex_chunks<2>(D, lc, h2, stage);
        else if (h2 == 10)
            apex_chunks<4>(D, lc, h2, stage);
        else
            apex_chunks<8>(D, lc, h2, stage);
        lc -= h2;
        __threadfence_block();
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// host-side launchers (called from oibvh_host.cpp)
// ---------------------------------------------------------------------------
// a tree's model matrix, written in stream order (the host copy may go away)
struct Mat16 {
    float m[16];
};
__global__ void k_set_xf(float* dst, Mat16 m)
{
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < 16; k++) dst[k] = m.m[k];
    }
}

// point mesh m of a batch at other vertex memory, in stream order (so that a
// captured frame replays against it without capturing again)
__global__ void k_set_mesh_pos(oi_build_desc* bd, oi_mesh_desc* md, uint32_t m, const float* pos)
{
    if (threadIdx.x == 0) {
        bd[m].pos = pos;
        md[m].pos = pos;
    }
}

static BuildTab make_btab(const oi_build_desc* d, const uint2* work, const oi_build_desc* one)
{
    BuildTab t{};
    t.d = d;
    t.work = work;
    t.n_inl = 1;
    if (one) t.inl[0] = *one;
    return t;
}

// n (<= OI_INLINE_MESHES) meshes in the kernel arguments; mesh m owns
// workgroups [boff[m], boff[m + 1])
static BuildTab make_btab_inline(const oi_build_desc* meshes, uint32_t n, const uint32_t* boff)
{
    BuildTab t{};
    t.n_inl = n;
    for (uint32_t m = 0; m < n && m < OI_INLINE_MESHES; m++) {
        t.inl[m] = meshes[m];
        t.boff[m] = boff[m];
    }
    t.boff[n < OI_INLINE_MESHES ? n : OI_INLINE_MESHES] = boff[n];
    return t;
}

// n (<= OI_WIDE_MESHES) meshes, as make_btab_inline
static WideTab make_wide(const oi_build_desc* meshes, uint32_t n, const uint32_t* boff)
{
    WideTab t{};
    t.n = n;
    for (uint32_t m = 0; m < n && m < OI_WIDE_MESHES; m++) {
        t.inl[m] = meshes[m];
        t.boff[m] = boff[m];
    }
    t.boff[n < OI_WIDE_MESHES ? n : OI_WIDE_MESHES] = boff[n];
    return t;
}

// a launch that records t0 as it starts and t1 as it completes (when set)
template <class K, class... Args>
static void launch_timed(K kernel, dim3 g, dim3 b, hipStream_t st, hipEvent_t t0, hipEvent_t t1, Args... args)
{
    if (t1)
        hipExtLaunchKernelGGL(kernel, g, b, 0, st, t0, t1, 0, args...);
    else
        hipLaunchKernelGGL(kernel, g, b, 0, st, args...);
}

extern "C" {

// Every launcher takes the mesh table as (d, work, one): a device descriptor
// table and work list, or d = work = null and `one` for a single mesh whose
// workgroup b takes chunk b.
hipError_t oi_launch_mesh_box(hipStream_t st, const oi_build_desc* d, const uint2* work, const oi_build_desc* one,
                              uint32_t nblocks, float* partials, uint32_t* clear_u32, uint32_t clear_n)
{
    hipLaunchKernelGGL(k_mesh_box, dim3(nblocks), dim3(OI_BLOCK), 0, st, make_btab(d, work, one), partials,
                       clear_u32, clear_n);
    return hipGetLastError();
}

// Faces a workgroup of k_morton takes in a launch over F faces: 1, 2 or 4 a thread.
// About one workgroup per CU, so that small launches spread and large ones add fewer
// histograms to the shared ones: 1M faces 15 us with 2 a thread, 13 with 4. Where
// they cannot all run at once, 2 a thread, of which two workgroups fit on a CU (50
// VGPRs; one with 4 a thread, 74): 42M faces 599 -> 436 us, builds of 1.06M to 7.8M
// faces 3 to 5 % less.
uint32_t oi_morton_chunk(uint64_t F)
{
    if (F <= 256ull * OI_MORTON_T) return OI_MORTON_T;
    return F <= 512ull * OI_MORTON_T || F > 1024ull * OI_MORTON_T ? 2u * OI_MORTON_T : 4u * OI_MORTON_T;
}

static hipError_t launch_morton(hipStream_t st, uint32_t chunk, uint32_t nblocks, const BuildTab& t,
                                const float* partials, uint32_t* keys, uint32_t* keys_hi, uint32_t* ghist,
                                uint32_t hstride, uint32_t hreps, uint32_t* fmesh, uint32_t hbits)
{
    if ((hbits != 8 && hbits != 10) || (keys_hi && hbits != 8) || hreps == 0) return hipErrorInvalidValue;
    switch (chunk) {
    case OI_MORTON_T:
        hipLaunchKernelGGL(k_morton<1>, dim3(nblocks), dim3(OI_MORTON_T), 0, st, t, partials, keys, keys_hi, ghist,
                           hstride, hreps, fmesh, hbits);
        break;
    case 2 * OI_MORTON_T:
        hipLaunchKernelGGL(k_morton<2>, dim3(nblocks), dim3(OI_MORTON_T), 0, st, t, partials, keys, keys_hi, ghist,
                           hstride, hreps, fmesh, hbits);
        break;
    case 4 * OI_MORTON_T:
        hipLaunchKernelGGL(k_morton<4>, dim3(nblocks), dim3(OI_MORTON_T), 0, st, t, partials, keys, keys_hi, ghist,
                           hstride, hreps, fmesh, hbits);
        break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t oi_launch_set_xf(hipStream_t st, float* dst, const float* mat4)
{
    Mat16 m;
    for (int k = 0; k < 16; k++) m.m[k] = mat4[k];
    hipLaunchKernelGGL(k_set_xf, dim3(1), dim3(64), 0, st, dst, m);
    return hipGetLastError();
}

// keys_hi: null for 30-bit keys, else the high words of 63-bit keys; chunk: the
// work items' (oi_morton_chunk)
hipError_t oi_launch_morton(hipStream_t st, const oi_build_desc* d, const uint2* work, const oi_build_desc* one,
                            uint32_t nblocks, uint32_t chunk, const float* partials, uint32_t* keys,
                            uint32_t* keys_hi, uint32_t* ghist, uint32_t hreps, uint32_t* fmesh, uint32_t hbits)
{
    return launch_morton(st, chunk, nblocks, make_btab(d, work, one), partials, keys, keys_hi, ghist, 0u, hreps,
                         fmesh, hbits);
}

// n (<= OI_INLINE_MESHES) meshes in the kernel arguments, mesh m owning the
// workgroups [boff[m], boff[m + 1]): the mesh boxes (partials in each mesh's
// own box buffer), and the Morton keys with mesh m's digit histograms at
// ghist + m * hstride
hipError_t oi_launch_mesh_box_inline(hipStream_t st, const oi_build_desc* meshes, uint32_t n, const uint32_t* boff,
                                     uint32_t* clear_u32, uint32_t clear_n)
{
    if (n == 0 || n > OI_INLINE_MESHES) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_mesh_box, dim3(boff[n]), dim3(OI_BLOCK), 0, st, make_btab_inline(meshes, n, boff), nullptr,
                       clear_u32, clear_n);
    return hipGetLastError();
}

hipError_t oi_launch_morton_inline(hipStream_t st, const oi_build_desc* meshes, uint32_t n, const uint32_t* boff,
                                   uint32_t chunk, uint32_t* keys, uint32_t* keys_hi, uint32_t* ghist,
                                   uint32_t hstride, uint32_t hreps, uint32_t hbits)
{
    if (n == 0 || n > OI_INLINE_MESHES) return hipErrorInvalidValue;
    return launch_morton(st, chunk, boff[n], make_btab_inline(meshes, n, boff), nullptr, keys, keys_hi, ghist,
                         hstride, hreps, nullptr, hbits);
}

hipError_t oi_launch_set_mesh_pos(hipStream_t st, oi_build_desc* bd, oi_mesh_desc* md, uint32_t m, const float* pos)
{
    hipLaunchKernelGGL(k_set_mesh_pos, dim3(1), dim3(64), 0, st, bd, md, m, pos);
    return hipGetLastError();
}

// Keys a thread of k_sort_pass takes, over ns segments of n[] keys: 1, 2, 4 or 8, the
// fewest that leave at most 128 tiles (256 with 4). More tiles rank fewer keys each
// but read more look-back statuses: builds of 122K, 250K and 518K triangles take 55.1,
// 63.5 and 77.1 us, and up to 256 tiles of fewer keys 55.3, 68.3 and 79.7; of 1M 99.2
// with 4 keys a thread, 103.9 with 8.
static uint32_t sort_items(uint32_t ns, const uint32_t* n)
{
    for (uint32_t it = 1; it < RS_ITEMS_MAX; it *= 2) {
        uint64_t tiles = 0;
        for (uint32_t k = 0; k < ns; k++) tiles += ((uint64_t)n[k] + RS_THREADS * it - 1) / (RS_THREADS * it);
        if (tiles <= (it < 4 ? OI_SORT_WGS / 2 : OI_SORT_WGS)) return it;
    }
    return RS_ITEMS_MAX;
}

uint32_t oi_sort_tiles(uint32_t ns, const uint32_t* n)
{
    const uint32_t tile = RS_THREADS * sort_items(ns, n);
    uint32_t tiles = 0;
    for (uint32_t k = 0; k < ns; k++) tiles += (uint32_t)(((uint64_t)n[k] + tile - 1) / tile);
    return tiles;
}

// rows of a look-back buffer: one per tile, then one per group
uint64_t oi_sort_rows(uint32_t ns, uint64_t tiles) { return tiles + tiles / LB_GROUP + ns; }

uint64_t oi_sort_tiles_max(uint64_t cap)
{
    const uint64_t fine = (cap + RS_THREADS - 1) / RS_THREADS;
    const uint64_t coarse = (cap + RS_THREADS * RS_ITEMS_MAX - 1) / (RS_THREADS * RS_ITEMS_MAX);
    return fine < OI_SORT_WGS ? fine : coarse > OI_SORT_WGS ? coarse : OI_SORT_WGS;
}

hipError_t oi_launch_sort_pass_segs(hipStream_t st, const uint32_t* keys_in, const uint32_t* vals_in,
                                    uint32_t* keys_out, uint32_t* vals_out, uint32_t ns, const uint32_t* base,
                                    const uint32_t* n, uint32_t shift, const uint32_t* ghist, uint32_t hstride,
                                    uint32_t hreps, uint32_t* lookback, uint32_t* lookback_next,
                                    uint32_t* tile_counter, const uint32_t* key_of_val, uint32_t bits);

hipError_t oi_launch_sort_pass(hipStream_t st, const uint32_t* keys_in, const uint32_t* vals_in, uint32_t* keys_out,
                               uint32_t* vals_out, uint32_t n, uint32_t shift, const uint32_t* ghist, uint32_t hreps,
                               uint32_t* lookback, uint32_t* lookback_next, uint32_t* tile_counter,
                               const uint32_t* key_of_val, uint32_t bits)
{
    const uint32_t base = 0;
    return oi_launch_sort_pass_segs(st, keys_in, vals_in, keys_out, vals_out, 1, &base, &n, shift, ghist, 0, hreps,
                                    lookback, lookback_next, tile_counter, key_of_val, bits);
}

uint32_t oi_sort_segs_max() { return OI_SORT_SEGS; }

// ns segments: segment s is keys [base[s], base[s] + n[s]) of the arrays, its
// digit histogram at ghist + s * hstride (hreps copies, 1 or OI_HIST_REPS), its tile
// counter tile_counter[s]; look-back statuses are indexed by the tile id over all
// segments (oi_sort_tiles of them)
hipError_t oi_launch_sort_pass_segs(hipStream_t st, const uint32_t* keys_in, const uint32_t* vals_in,
                                    uint32_t* keys_out, uint32_t* vals_out, uint32_t ns, const uint32_t* base,
                                    const uint32_t* n, uint32_t shift, const uint32_t* ghist, uint32_t hstride,
                                    uint32_t hreps, uint32_t* lookback, uint32_t* lookback_next,
                                    uint32_t* tile_counter, const uint32_t* key_of_val, uint32_t bits)
{
    if (ns == 0 || ns > OI_SORT_SEGS || (bits != 8 && bits != 10) || (hreps != 1 && hreps != OI_HIST_REPS))
        return hipErrorInvalidValue;
    const uint32_t items = sort_items(ns, n), tile = RS_THREADS * items;
    SortSegs S{};
    S.ns = ns;
    S.hstride = hstride;
    uint32_t tiles = 0;
    for (uint32_t k = 0; k < ns; k++) {
        if (n[k] == 0) return hipErrorInvalidValue;
        S.tile0[k] = tiles;
        S.base[k] = base[k];
        S.n[k] = n[k];
        tiles += (uint32_t)(((uint64_t)n[k] + tile - 1) / tile);
    }
    S.tile0[ns] = tiles;
#define PASS(DB, IT)                                                                                              \
    hipLaunchKernelGGL((k_sort_pass<DB, IT>), dim3(tiles), dim3(RS_THREADS), 0, st, keys_in, vals_in, keys_out,   \
                       vals_out, S, shift, ghist, hreps, lookback, lookback_next, tile_counter, key_of_val)
    switch (items) {
    case 1:
        if (bits == 10) PASS(10, 1); else PASS(8, 1);
        break;
    case 2:
        if (bits == 10) PASS(10, 2); else PASS(8, 2);
        break;
    case 4:
        if (bits == 10) PASS(10, 4); else PASS(8, 4);
        break;
    default:
        if (bits == 10) PASS(10, 8); else PASS(8, 8);
        break;
    }
#undef PASS
    return hipGetLastError();
}

// subtree height of stage 1 for M leaves per thread
// M = 16 selects k_reduce_w, whose stage 1 climbs as high as k_reduce<4>
static uint32_t lgm_of(int M) { return (M == 1) ? 0 : (M == 2) ? 1 : (M == 4 || M == 16) ? 2 : 3; }

uint32_t oi_reduce_height(int M, uint32_t L)
{
    const uint32_t lgm = lgm_of(M);
    return (L < 8 + lgm) ? L : 8 + lgm;
}

}  // extern "C"

template <class Tab>
static hipError_t launch_reduce(hipStream_t st, int M, ReduceArgs<Tab> a, uint32_t nblocks, hipEvent_t t0,
                                hipEvent_t t1, uint32_t max_blocks)
{
    if (!t0 != !t1) return hipErrorInvalidValue;
    dim3 g(nblocks);
    const dim3 b(OI_BLOCK);
    if (M == 16 && !a.vals && max_blocks && max_blocks < nblocks) {
        const uint32_t cap = (max_blocks + 7u) & ~7u;
        if (cap < nblocks) {
            a.nwork = nblocks;
            g = dim3(cap);
        }
    }
    switch (M) {
    case 1: launch_timed((k_reduce<1, Tab>), g, b, st, t0, t1, a); break;
    case 2: launch_timed((k_reduce<2, Tab>), g, b, st, t0, t1, a); break;
    case 4: launch_timed((k_reduce<4, Tab>), g, b, st, t0, t1, a); break;
    case 16:
        if (a.nwork)
            launch_timed((k_reduce_wl<Tab>), g, b, st, t0, t1, a);
        else
            launch_timed((k_reduce_w<Tab>), g, b, st, t0, t1, a);
        break;
    default: launch_timed((k_reduce<8, Tab>), g, b, st, t0, t1, a); break;
    }
    return hipGetLastError();
}

// mid: k_reduce_mid has run for the meshes that need it
template <class Tab>
static hipError_t launch_apex(hipStream_t st, int M, const Tab& t, uint32_t n, uint32_t mid, const oi_seed_args* seed,
                              hipEvent_t done)
{
    if (seed && seed->n_counts > OI_BLOCK) return hipErrorInvalidValue;
    const ReduceArgs<Tab> a{t, nullptr, 0, 0};
    const oi_seed_args sd = seed ? *seed : oi_seed_args{};
    const dim3 g(n + (seed ? 1u : 0u)), b(OI_BLOCK);
    // with done the launch records it on completion (no separate event call)
    if (done)
        hipExtLaunchKernelGGL((k_reduce_apex<Tab>), g, b, 0, st, nullptr, done, 0, a, lgm_of(M), mid, sd);
    else
        hipLaunchKernelGGL((k_reduce_apex<Tab>), g, b, 0, st, a, lgm_of(M), mid, sd);
    return hipGetLastError();
}

// k_reduce_mid over those of n (<= OI_WIDE_MESHES) meshes that need it
static hipError_t launch_mid(hipStream_t st, int M, const oi_build_desc* meshes, uint32_t n)
{
    const uint32_t lgm = lgm_of(M);
    oi_build_desc d[OI_WIDE_MESHES];
    uint32_t boff[OI_WIDE_MESHES + 1] = {0}, k = 0;
    for (uint32_t m = 0; m < n; m++) {
        if (meshes[m].L <= 8u + lgm + APEX_MID) continue;
        d[k] = meshes[m];
        boff[k + 1] = boff[k] + oi_lvl_cnt(d[k].L - (8u + lgm) - 8u, d[k].L, d[k].vl);
        k++;
    }
    if (k == 0) return hipSuccess;
    const dim3 g(boff[k]), b(OI_BLOCK);
    if (k <= OI_INLINE_MESHES)
        hipLaunchKernelGGL((k_reduce_mid<BuildTab>), g, b, 0, st,
                           (ReduceArgs<BuildTab>{make_btab_inline(d, k, boff), nullptr, 0, 0}), lgm);
    else
        hipLaunchKernelGGL((k_reduce_mid<WideTab>), g, b, 0, st,
                           (ReduceArgs<WideTab>{make_wide(d, k, boff), nullptr, 0, 0}), lgm);
    return hipGetLastError();
}

extern "C" {

// stage 1 (M = leaves per thread: 1, 2, 4 or 8; 16: wave subtrees); vals:
// build, null: refit. With t0 and t1 (both or neither) the launch records
// them as it starts and completes. max_blocks > 0 (refits with M = 16 only):
// at most that many workgroups (rounded up to a multiple of 8), each looping
// over work items, as in oi_launch_reduce_inline
hipError_t oi_launch_reduce(hipStream_t st, int M, const oi_build_desc* d, const uint2* work,
                            const oi_build_desc* one, uint32_t nblocks, const uint32_t* vals, uint32_t write_perm,
                            hipEvent_t t0, hipEvent_t t1, uint32_t max_blocks)
{
    return launch_reduce(st, M, ReduceArgs<BuildTab>{make_btab(d, work, one), vals, write_perm, 0}, nblocks, t0, t1,
                         max_blocks);
}

uint32_t oi_inline_meshes() { return OI_INLINE_MESHES; }
uint32_t oi_wide_meshes() { return OI_WIDE_MESHES; }

// stage 1 over up to OI_WIDE_MESHES meshes passed by value; boff[n + 1]
// gives each mesh's first workgroup
// with t0 and t1 (both or neither) the launch itself records them as it
// starts and completes: their elapsed time is the kernel's own duration.
// max_blocks > 0 (refits with k_reduce_w only): at most that many workgroups (rounded up
// to a multiple of 8), each looping over work items, which leaves the rest
// of the GPU to work running beside the launch
hipError_t oi_launch_reduce_inline(hipStream_t st, int M, const oi_build_desc* meshes, uint32_t n,
                                   const uint32_t* boff, const uint32_t* vals, uint32_t write_perm, hipEvent_t t0,
                                   hipEvent_t t1, uint32_t max_blocks)
{
    if (n == 0 || n > OI_WIDE_MESHES) return hipErrorInvalidValue;
    if (n <= OI_INLINE_MESHES)
        return launch_reduce(st, M, ReduceArgs<BuildTab>{make_btab_inline(meshes, n, boff), vals, write_perm, 0},
                             boff[n], t0, t1, max_blocks);
    return launch_reduce(st, M, ReduceArgs<WideTab>{make_wide(meshes, n, boff), vals, write_perm, 0}, boff[n], t0, t1,
                         max_blocks);
}

// stage 2 for n inline meshes, one workgroup each; with seed (may be null)
// one more workgroup resets the following detect's counters
hipError_t oi_launch_reduce_apex_inline(hipStream_t st, int M, const oi_build_desc* meshes, uint32_t n,
                                        const oi_seed_args* seed, hipEvent_t done)
{
    if (n == 0 || n > OI_WIDE_MESHES) return hipErrorInvalidValue;
    uint32_t boff[OI_WIDE_MESHES + 1];
    for (uint32_t m = 0; m <= n; m++) boff[m] = m;
    const hipError_t e = launch_mid(st, M, meshes, n);
    if (e != hipSuccess) return e;
    if (n <= OI_INLINE_MESHES) return launch_apex(st, M, make_btab_inline(meshes, n, boff), n, 1, seed, done);
    return launch_apex(st, M, make_wide(meshes, n, boff), n, 1, seed, done);
}

// stage 2, one workgroup per work item (mesh, 0) whose L exceeds the stage-1 height
hipError_t oi_launch_reduce_apex(hipStream_t st, int M, const oi_build_desc* d, const uint2* work,
                                 const oi_build_desc* one, uint32_t nblocks, const oi_seed_args* seed)
{
    if (one) {
        const hipError_t e = launch_mid(st, M, one, 1);
        if (e != hipSuccess) return e;
    }
    return launch_apex(st, M, make_btab(d, work, one), nblocks, one ? 1u : 0u, seed, nullptr);
}

}  // extern "C"
