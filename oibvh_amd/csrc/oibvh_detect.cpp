// oibvh_detect.cpp -- the BVTT detector shared by scenes and batches: buffer
// management, the launch sequence of one query and the overflow re-run loop
// (Scene::detectCollisionOnGPU, scene.cu:225-446, which instead copies the
// front size to the host after every level and uses fixed 10M-entry buffers).
#include <chrono>

#include "oibvh_internal.h"

// before a buffer an overlapped frame's detect may still use is freed or
// rewritten
static oibvh_status idle(oibvh_ctx* c)
{
    if (c->side[0]) HIPCHK(c, oi_ctx_quiesce(c));
    return OIBVH_OK;
}

template <class T>
static oibvh_status grow(oibvh_ctx* c, T*& p, uint32_t& cap, uint64_t need, uint64_t& gen)
{
    if (cap >= need) return OIBVH_OK;
    if (need > 0x7fffffffull) return oi_set_err(c, OIBVH_ERR_OVERFLOW, "detect buffer would exceed 2^31 entries");
    oibvh_status r = idle(c);
    if (r != OIBVH_OK) return r;
    dfree(p);
    cap = 0;
    gen++;
    HIPCHK(c, dalloc(&p, need));
    cap = (uint32_t)need;
    return OIBVH_OK;
}

oibvh_status oi_det_init(oi_detector* d, oibvh_ctx* c)
{
    d->ctx = c;
    hipError_t e = dalloc(&d->ctl_base, OI_FRAME_DEPTH);
    if (e == hipSuccess) e = hipMemsetAsync(d->ctl_base, 0, OI_FRAME_DEPTH * sizeof(oi_detect_ctl), c->stream);
    if (e == hipSuccess)
        e = hipHostMalloc((void**)&d->h_pub, sizeof(oi_published), hipHostMallocCoherent | hipHostMallocMapped);
    if (e != hipSuccess) {
        oi_det_free(d);
        return oi_set_err(c, OIBVH_ERR_HIP, "detector alloc: %s", hipGetErrorString(e));
    }
    std::memset(d->h_pub, 0, sizeof(oi_published));
    d->ctl = d->ctl_base;
    return OIBVH_OK;
}

// the current set's working buffers to / from their per-set slots
static void save_view(oi_detector* d)
{
    const uint32_t k = d->set;
    d->set_front[k][0] = d->front[0];
    d->set_front[k][1] = d->front[1];
    d->set_front_cap[k] = d->front_cap;
    d->set_cands[k] = d->cands;
    d->set_cand_cap[k] = d->cand_cap;
    d->set_hits[k] = d->hits;
    d->set_hits_cap[k] = d->hits_cap;
}

static void load_view(oi_detector* d)
{
    const uint32_t k = d->set;
    d->front[0] = d->set_front[k][0];
    d->front[1] = d->set_front[k][1];
    d->front_cap = d->set_front_cap[k];
    d->cands = d->set_cands[k];
    d->cand_cap = d->set_cand_cap[k];
    d->hits = d->set_hits[k];
    d->hits_cap = d->set_hits_cap[k];
}

void oi_det_use_set(oi_detector* d, uint32_t k)
{
    if (k == d->set) return;
    save_view(d);
    // the set left behind keeps an unchecked result until a check reads it;
    // the set taken holds none any more: an asynchronous seed folds its
    // errors into its sticky bits, and a synchronous frame checks first
    if (d->unchecked) d->set_unchecked[d->set] = true;
    d->set = k % OI_FRAME_DEPTH;
    load_view(d);
    d->set_unchecked[d->set] = false;
    d->ctl = d->ctl_base + d->set;
    d->counts = d->counts_base ? d->counts_base + 256u * d->set : nullptr;
}

void oi_det_flip_set(oi_detector* d) { oi_det_use_set(d, (d->set + 1u) % OI_FRAME_DEPTH); }

void oi_det_free(oi_detector* d)
{
    dfree(d->d_init);
    save_view(d);
    for (uint32_t k = 0; k < OI_FRAME_DEPTH; k++) {
        dfree(d->set_front[k][0]);
        dfree(d->set_front[k][1]);
        dfree(d->set_cands[k]);
        dfree(d->set_hits[k]);
        d->set_front_cap[k] = d->set_cand_cap[k] = d->set_hits_cap[k] = 0;
    }
    load_view(d);
    dfree(d->counts_base);
    d->counts = nullptr;
    dfree(d->d_sorted);
    dfree(d->sort_words);
    dfree(d->sort_vals);
    dfree(d->sort_scratch);
    dfree(d->sort_mem);
    dfree(d->d_stage);
    dfree(d->ctl_base);
    d->ctl = nullptr;
    if (d->h_pairs) (void)hipHostFree(d->h_pairs);
    d->h_pairs = nullptr;
    if (d->h_pub) (void)hipHostFree(d->h_pub);
    d->h_pub = nullptr;
}

oibvh_status oi_det_set_front(oi_detector* d, const std::vector<uint2>& front)
{
    oibvh_ctx* c = d->ctx;
    oibvh_status r = idle(c);
    if (r != OIBVH_OK) return r;
    d->n_front = (uint32_t)front.size();
    r = grow(c, d->d_init, d->init_cap, std::max(1u, d->n_front), d->generation);
    if (r != OIBVH_OK) return r;
    if (d->n_front)
        HIPCHK(c, hipMemcpyAsync(d->d_init, front.data(), d->n_front * sizeof(uint2), hipMemcpyHostToDevice,
                                 c->stream));
    return OIBVH_OK;
}

// Steps over short fronts as k_bvtt_walk launches, two steps each where the
// second's tests are few as well. The host does not know the fronts' lengths: it
// takes them to grow by e + 1 per step of e levels (measured: 2.0-2.9 for two
// levels and 2.8-4.2 for three, two bodies), in self mode by 2^e + 3 (4-8 and
// 9-15, folded cloth), or, after a query that met far longer ones, as that query met
// them (judge_walk). A wrong guess costs speed only.
// Where the lines lie: one k_bvtt_step of three levels takes 15 us on any front up
// to 10,000 pairs and 18-25 us at 50,000, a walk of two such steps 11 us at 100
// pairs, 19 us at 2,800 and of one step 14 us at 10,000; a step of two levels
// takes 8 us up to 10,000 pairs, a walk of two 11 us at 36 and 19 us at 2,400.
#define OI_WALK_MAX3 65536u
#define OI_WALK_MAX 2048u
#define OI_WALK_TESTS (1u << 21)
// lengths from here on get workgroups for a long front (beside the next frame's
// refit they would take its room)
#define OI_WALK_LONG 16384u
static uint64_t walk_max(uint32_t e) { return e == 3 ? OI_WALK_MAX3 : OI_WALK_MAX; }

// walk[k] for n steps of e[k] levels over fronts of len[k] pairs
static void walk_steps(uint32_t n, const uint8_t* e, const uint32_t* len, uint8_t* walk)
{
    std::memset(walk, 0, n);
    for (uint32_t k = 0; k < n && len[k] <= walk_max(e[k]); k++) {
        walk[k] = len[k] >= OI_WALK_LONG ? 5 : 1;
        if (k + 1 < n && (uint64_t)len[k + 1] << (2u * e[k + 1]) <= OI_WALK_TESTS) walk[k++]++;
    }
}

// whether a walk of that plan meets a front too long for it, with `far` much too long.
// (The lines of `far`. First steps: a walk of two levels over 60K pairs of one dense
// spot takes 98 us where the step takes 124, one of three over 948K, leaf pairs mostly,
// no more than the step, and 140K pairs with their 500K children 64 against 74; but
// over 741K others 105 against 69. Second steps: 12K pairs with their 108K children of
// three levels 62-82 us against 45 by a walk and a step, 39K with 260K 165 against 52.)
static bool walk_too_long(uint32_t n, const uint8_t* e, const uint8_t* walk, const uint32_t* len, bool far)
{
    for (uint32_t k = 0; k < n && walk[k]; k++) {
        if (len[k] > (far ? 4u : 2u) * OI_WALK_MAX3) return true;
        if ((walk[k] & 3u) != 2u) continue;
        k++;
        if ((uint64_t)len[k] << (2u * e[k]) > (far ? OI_WALK_TESTS * 3u / 2u : OI_WALK_TESTS)) return true;
    }
    return false;
}

static void guess_lengths(const oi_detector* d, uint32_t* len)
{
    const bool self = (d->flags & OIBVH_DETECT_SELF) != 0;
    uint64_t est = d->n_front;
    for (uint32_t k = 0; k < d->n_levels; k++) {
        len[k] = (uint32_t)std::min<uint64_t>(est, 1u << 31);
        est = len[k] * (uint64_t)(self ? (1u << d->step_e[k]) + 3u : d->step_e[k] + 1u);
    }
}

static void plan_walk(oi_detector* d)
{
    std::memset(d->step_walk, 0, sizeof d->step_walk);
    // lengths that another query met
    if (d->n_seen && (d->n_seen != d->n_levels || d->seen[0] != d->n_front ||
                      d->seen_self != ((d->flags & OIBVH_DETECT_SELF) != 0) ||
                      std::memcmp(d->seen_e, d->step_e, d->n_levels) != 0)) {
        d->n_seen = 0;
        d->generation++;
    }
    if (d->local_chunk || d->tail_chunk || d->n_front == 0) return;
    uint32_t guess[256];
    if (!d->n_seen) guess_lengths(d, guess);
    walk_steps(d->n_levels, d->step_e, d->n_seen ? d->seen : guess, d->step_walk);
}

// After a query whose front lengths have been read: where a walk met a front far past
// its limit, the next queries are planned by these lengths, until one fits the guess's
// plan. (Overlapping triangle clouds grow by 9 to 19 a step of three levels. Two of
// 400,000 triangles: 305 and, denser, 535 us a query as guessed, 158 and 274 from the
// second query on; 218 and 340 by the steps alone that were there before the walks.)
static void judge_walk(oi_detector* d)
{
    if (d->local_chunk || d->tail_chunk || d->n_front == 0) return;
    const uint32_t n = d->n_levels, *len = d->h_counts.data();
    if (walk_too_long(n, d->step_e, d->step_walk, len, true)) {
        d->n_seen = n;
        std::copy(len, len + n, d->seen);
        std::copy(d->step_e, d->step_e + n, d->seen_e);
        d->seen_self = (d->flags & OIBVH_DETECT_SELF) != 0;
        d->generation++;
    } else if (d->n_seen) {
        uint32_t guess[256];
        uint8_t walk[256];
        guess_lengths(d, guess);
        walk_steps(n, d->step_e, guess, walk);
        if (walk_too_long(n, d->step_e, walk, len, false)) return;
        d->n_seen = 0;
        d->generation++;
    }
}

oibvh_status oi_det_prepare(oi_detector* d)
{
    oibvh_ctx* c = d->ctx;
    // every BVTT step takes each non-leaf side up to `expand` levels down and
    // tests the pairs it reaches: the walk ends at the leaves after
    // ceil(depth / expand) steps (one step tests entry-level leaf pairs)
    // the schedule's leading steps, then `expand` per step, until the deepest
    // tree's leaves are reached (at least one step)
    uint32_t k = 0, done = 0, sch = d->schedule;
    bool lead = true;
    while (k == 0 || done < d->depth) {
        uint32_t e = lead ? (sch & 3u) : 0u;
        if (e == 0) {
            lead = false;
            e = d->expand;
        }
        sch >>= 2;
        if (k + 1 >= 256) return oi_set_err(c, OIBVH_ERR_INVALID, "detect: more than 255 BVTT steps");
        d->step_e[k++] = (uint8_t)e;
        done += e;
    }
    d->n_levels = k;
    const uint32_t past = d->depth && done > d->depth ? done - d->depth : 0u;
    // the first steps as one local walk when asked for, unless it overflowed
    // recently; its steps all descend `expand` levels
    const uint32_t mode = c->trav_local;
    d->local_chunk = 0;
    d->local_levels = 0;
    // a walk that overflowed stays off until the tuning is set again: an
    // asynchronous detect cannot re-run, so one that overflowed again
    // would leave its frame incomplete
    if (mode && d->local_off != c->tuning_gen + 1 && d->n_front) {
        d->local_chunk = mode;
        k = 0;
        done = 0;
        while (k == 0 || done < d->depth) {
            d->step_e[k++] = (uint8_t)d->expand;
            done += d->expand;
        }
        d->n_levels = k;
        d->local_levels = c->trav_local_levels ? std::min(c->trav_local_levels, k) : k;
    }
    // the last steps as a tail walk when asked for (unless it overflowed
    // recently): it starts after the head walk and after every step whose
    // depth the schedule set, since it descends `expand` levels per step
    d->tail_chunk = 0;
    d->tail_from = 0;
    if (c->trav_tail && d->tail_off != c->tuning_gen + 1 && d->n_front) {
        const uint32_t S = c->trav_tail_steps;
        uint32_t T = (S && S < d->n_levels) ? d->n_levels - S : 0u;
        T = std::max(T, d->local_chunk ? d->local_levels : 0u);
        for (uint32_t j = T; j < d->n_levels; j++)
            if (d->step_e[j] != d->expand) T = j + 1;
        if (T < d->n_levels) {
            d->tail_chunk = c->trav_tail;
            d->tail_from = T;
        }
    }
    // no side has more levels left than the deepest tree: levels of the last step
    // past its leaves would only repeat tests
    if (!d->local_chunk && !d->tail_chunk) d->step_e[d->n_levels - 1] -= (uint8_t)past;
    plan_walk(d);
    const uint32_t fcap = std::max(std::max(c->queue_cap, d->want_front), oi_np2(std::max(1u, d->n_front)));
    if (d->front_cap < fcap) {
        oibvh_status ri = idle(c);
        if (ri != OIBVH_OK) return ri;
        dfree(d->front[0]);
        dfree(d->front[1]);
        d->front_cap = 0;
        d->generation++;
        HIPCHK(c, dalloc(&d->front[0], fcap));
        HIPCHK(c, dalloc(&d->front[1], fcap));
        d->front_cap = fcap;
    }
    oibvh_status r;
    if ((r = grow(c, d->counts_base, d->counts_cap, 256u * OI_FRAME_DEPTH, d->generation)) != OIBVH_OK) return r;
    d->counts = d->counts_base + 256u * d->set;
    if ((r = grow(c, d->cands, d->cand_cap, std::max(c->cand_cap, d->want_cands), d->generation)) != OIBVH_OK)
        return r;
    if ((r = grow(c, d->hits, d->hits_cap, std::max(c->hits_cap, d->want_hits), d->generation)) != OIBVH_OK)
        return r;
    return OIBVH_OK;
}

oi_seed_args oi_det_seed_args(const oi_detector* d, bool reset_sticky)
{
    oi_seed_args s{};
    s.counts = d->counts;
    s.ctl = d->ctl;
    s.n0 = d->n_front;
    s.n_counts = d->n_levels + 1;
    s.reset_sticky = reset_sticky ? 1u : 0u;
    return s;
}

oibvh_status oi_det_enqueue(oi_detector* d, bool reset_sticky, bool seeded, hipEvent_t done)
{
    oibvh_ctx* c = d->ctx;
    hipStream_t st = d->stream ? d->stream : c->stream;
    if (!seeded)
        HIPCHK(c, oi_launch_seed(st, d->n_front, d->counts, d->n_levels + 1, d->ctl, reset_sticky ? 1u : 0u));
    const bool fp64 = (d->flags & OIBVH_DETECT_FP64_FALLBACK) != 0;
    const uint32_t J = d->local_chunk ? d->local_levels : 0u;
    const uint32_t T = d->tail_chunk ? d->tail_from : d->n_levels;
    // Leaf pairs are tested inside the BVTT launches that find them (unless
    // narrow_separate): FP32 queries with the SAT; FP64-fallback queries with
    // the FP32 filter in the steps (not in local walks), the pairs it leaves
    // undecided collected in the candidate buffer for one FP64 pass
    d->fused = !c->narrow_separate && (!fp64 || (J == 0 && T >= d->n_levels));
    const int fuse = d->fused ? (fp64 ? 2 : 1) : 0;
    // Workgroups per step. A step of up to two levels fits six workgroups on a CU;
    // with six instead of four the folded cloth of 8.4M triangles takes 1,743
    // instead of 1,849 us a frame, one of 522K 264 instead of 279. With the FP32
    // filter in the step four are faster (331 against 339 us on coplanar scenes),
    // and beside the next frame's refit they leave it room (overlapped batches, with
    // six a CU, and four in long walks, against four and two: 32 cloths of 32K
    // triangles 361 against 323 us a frame, one of 522K 170 against 160, 16 scenes of
    // rigid bodies 281 against 262; two cloths of 2.1M, one of 8.4M and 128 scenes the
    // same within 2 %).
    const uint32_t cus = (uint32_t)std::max(1, c->cus), grid = oi_grid_for(c);
    const uint32_t grid2 = c->trav_blocks || fuse != 1 || d->beside_refit ? grid : 6u * cus;
    // and per walk, over a short and over a long front; a setting is the most they launch
    const uint32_t most = c->trav_blocks ? c->trav_blocks : ~0u;
    const uint32_t walk_wgs = std::min(most, 2u * cus), walk_long = std::min(most, 4u * cus);
    // `done` rides on the last launch: k_narrow, else the tail walk, else
    // the last step, else the head walk
    const bool narrow = !d->fused || fp64, tail = T < d->n_levels, steps = T > J;
    hipEvent_t done_head = (!narrow && !tail && !steps) ? done : nullptr;
    hipEvent_t done_tail = (!narrow && tail) ? done : nullptr;
    if (J) {
        // steps 0 .. J-1 in one launch; its front goes where step J - 1's would
        oi_local_args w{};
        w.front_in = d->d_init;
        w.n_in = d->n_front;
        w.chunk = d->local_chunk;
        w.levels = J;
        w.test_entries = 1;
        w.overflow_bit = OI_ERR_LOCAL_OVERFLOW;
        w.front_out = d->front[(J - 1) & 1];
        w.count_out = d->counts + J;
        w.cap_out = d->front_cap;
        w.done = done_head;
        HIPCHK(c, oi_launch_bvtt_local(st, &d->tab, &w, d->cands, &d->ctl->cands, d->cand_cap, d->hits, d->hits_cap,
                                       d->ctl, d->expand, d->implicit_end, d->fused ? 1 : 0));
        done_head = nullptr;
    }
    // the buffer that holds the current front (step 0 reads the initial front
    // in place); every launch writes the other one
    uint32_t rd = J ? (J - 1) & 1u : 1u;
    for (uint32_t k = J; k < T; k++) {
        const uint2* in = k ? d->front[rd] : d->d_init;
        rd ^= 1u;
        if (d->step_walk[k]) {
            // this step, or this and the next one, over a short front
            const bool two = (d->step_walk[k] & 3u) == 2;
            const uint32_t o = two ? k + 1 : k;
            oi_walk_args w{};
            w.front_in = in;
            w.count_in = k ? d->counts + k : nullptr;
            w.n_in = d->n_front;
            w.cap_in = k ? d->front_cap : d->n_front;
            w.e1 = d->step_e[k];
            w.e2 = two ? d->step_e[k + 1] : 0u;
            w.test_entries = k == 0 ? 1u : 0u;
            w.front_out = d->front[rd];
            w.count_mid = two ? d->counts + k + 1 : nullptr;
            w.count_out = d->counts + o + 1;
            w.cap_out = d->front_cap;
            w.wgs_long = (d->step_walk[k] & 4u) && !d->beside_refit ? walk_long : 0u;
            w.done = (!narrow && !tail && o + 1 == T) ? done : nullptr;
            HIPCHK(c, oi_launch_bvtt_walk(st, walk_wgs, &d->tab, &w, d->cands, &d->ctl->cands, d->cand_cap, d->hits,
                                          d->hits_cap, d->ctl, d->implicit_end, fuse));
            k = o;
            continue;
        }
        HIPCHK(c, oi_launch_bvtt_step(st, d->step_e[k] < 3 ? grid2 : grid, &d->tab, k == 0, in, k ? d->counts + k : nullptr, d->n_front,
                                      k ? d->front_cap : d->n_front, d->front[rd], d->counts + k + 1,
                                      d->front_cap, d->cands, &d->ctl->cands, d->cand_cap, d->hits, d->hits_cap,
                                      d->ctl, d->step_e[k], d->implicit_end, fuse,
                                      (!narrow && !tail && k + 1 == T) ? done : nullptr));
    }
    if (tail) {
        // steps T .. n_levels - 1 in one launch over the front step T - 1
        // left: every pair ends at the leaves, so the last level writes no
        // front (its count, checked below, stays 0); front_out is the buffer
        // not being read
        oi_local_args w{};
        w.front_in = T ? d->front[rd] : d->d_init;
        w.count_in = T ? d->counts + T : nullptr;
        w.n_in = d->n_front;
        w.cap_in = T ? d->front_cap : d->n_front;
        w.chunk = d->tail_chunk;
        w.levels = d->n_levels - T;
        w.grid = 4u * (uint32_t)std::max(1, c->cus);
        w.test_entries = T == 0 ? 1u : 0u;
        w.overflow_bit = OI_ERR_TAIL_OVERFLOW;
        w.front_out = d->front[rd ^ 1u];
        w.count_out = d->counts + d->n_levels;
        w.cap_out = d->front_cap;
        w.done = done_tail;
        HIPCHK(c, oi_launch_bvtt_local(st, &d->tab, &w, d->cands, &d->ctl->cands, d->cand_cap, d->hits, d->hits_cap,
                                       d->ctl, d->expand, d->implicit_end, d->fused ? 1 : 0));
    }
    if (narrow && !fp64)
        HIPCHK(c, oi_launch_narrow(st, grid, &d->tab, d->cands, &d->ctl->cands, d->cand_cap, d->hits,
                                   &d->ctl->n_hits, d->hits_cap, d->ctl, 0, nullptr, 0, done));
    if (fp64 && d->fused) {
        // the FP64 SAT over the pairs the steps' filter left undecided
        HIPCHK(c, oi_launch_narrow(st, grid, &d->tab, d->cands, &d->ctl->deferred, d->cand_cap, d->hits,
                                   &d->ctl->n_hits, d->hits_cap, d->ctl, 2, nullptr, 0, done));
    } else if (narrow && fp64) {
        // the FP32 filter over the candidates, then the FP64 SAT over the
        // pairs it left undecided; the BVTT fronts are idle by now, and the
        // first holds that list (an overflow grows them like a front's)
        HIPCHK(c, oi_launch_narrow(st, grid, &d->tab, d->cands, &d->ctl->cands, d->cand_cap, d->hits,
                                   &d->ctl->n_hits, d->hits_cap, d->ctl, 1, d->front[0], d->front_cap, nullptr));
        HIPCHK(c, oi_launch_narrow(st, grid, &d->tab, d->front[0], &d->ctl->deferred, d->front_cap, d->hits,
                                   &d->ctl->n_hits, d->hits_cap, d->ctl, 2, nullptr, 0, done));
    }
    else if (done_head)  // a query with no BVTT launch
        HIPCHK(c, hipEventRecord(done, st));
    d->unchecked = true;
    d->have_result = true;
    d->sorted_ok = false;
    return OIBVH_OK;
}

// Wait for the sequence number that the last launch on the context's stream
// writes: a short wait on the memory itself (a stream wait costs about 10 us
// more than the launch it waits for), then the stream's, which also reports a
// failed launch. A program that chose to block or yield in its waits wants its core
// back: there the stream's wait only.
static hipError_t wait_published(oi_detector* d)
{
    unsigned flags = 0;
    if (hipGetDeviceFlags(&flags) == hipSuccess && (flags & (hipDeviceScheduleYield | hipDeviceScheduleBlockingSync)))
        return hipStreamSynchronize(d->ctx->stream);
    const auto t0 = std::chrono::steady_clock::now();
    while (__atomic_load_n(&d->h_pub->seq, __ATOMIC_ACQUIRE) != d->pub_seq)
        if (std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(20))
            return hipStreamSynchronize(d->ctx->stream);
    return hipSuccess;
}

// wait until everything queued on the context's stream so far has completed,
// through the published sequence number
static oibvh_status finish(oi_detector* d)
{
    oi_publish_args pa{};
    pa.out = d->h_pub;
    pa.seq = ++d->pub_seq;
    HIPCHK(d->ctx, oi_launch_publish(d->ctx->stream, &pa));
    HIPCHK(d->ctx, wait_published(d));
    return OIBVH_OK;
}

oibvh_status oi_det_check(oi_detector* d)
{
    oibvh_ctx* c = d->ctx;
    if (!d->unchecked) return OIBVH_OK;
    HIPCHK(c, oi_ctx_join(c));  // an overlapped frame's detect ran on a side stream
    uint32_t retries = 0, earlier = 0;
    for (;;) {
        // this query's counters and front lengths, and those of the other sets
        // still holding unchecked overlapped frames' results
        uint32_t others[OI_FRAME_DEPTH], n_others = 0;
        oi_publish_args pa{};
        pa.ctl[pa.n_sets++] = d->ctl;
        for (uint32_t s = 0; s < OI_FRAME_DEPTH; s++)
            if (s != d->set && d->set_unchecked[s]) {
                others[n_others++] = s;
                pa.ctl[pa.n_sets++] = d->ctl_base + s;
            }
        pa.counts = d->counts;
        pa.n_counts = d->n_levels + 1;
        pa.out = d->h_pub;
        pa.seq = ++d->pub_seq;
        HIPCHK(c, oi_launch_publish(c->stream, &pa));
        HIPCHK(c, wait_published(d));
        d->h_counts.assign(d->h_pub->counts, d->h_pub->counts + d->n_levels + 1);
        const oi_published& k = *d->h_pub;
        earlier |= k.sticky | k.earlier;  // errors of unchecked asynchronous detects before this one
        for (uint32_t j = 0; j < n_others; j++) {
            // earlier overlapped frames' detects and the unchecked ones before them
            d->set_unchecked[others[j]] = false;
        }
        if (d->h_counts[d->n_levels] != 0) {
            // the last step reaches the leaves on every side: it writes no front
            d->unchecked = false;
            d->have_result = false;
            return oi_set_err(c, OIBVH_ERR_HIP, "detect: %u BVTT pairs left after the last step",
                              d->h_counts[d->n_levels]);
        }
        if (k.error & OI_ERR_CORRUPT) {
            d->unchecked = false;
            d->have_result = false;
            return oi_set_err(c, OIBVH_ERR_HIP, "detect: corrupt BVTT entry (error bits 0x%x)", k.error);
        }
        bool rerun = false;
        oibvh_status r = OIBVH_OK;
        if (k.error & OI_ERR_LOCAL_OVERFLOW) {
            // a workgroup's front outgrew LDS: steps for the next queries
            d->local_off = c->tuning_gen + 1;
            rerun = true;
        }
        if (k.error & OI_ERR_TAIL_OVERFLOW) {
            d->tail_off = c->tuning_gen + 1;
            rerun = true;
        }
        uint32_t maxfront = 0;
        for (uint32_t v : d->h_counts) maxfront = std::max(maxfront, v);
        if (k.error & OI_ERR_QUEUE_OVERFLOW) {
            uint64_t need = 1;
            while (need < std::max<uint64_t>(maxfront, 4ull * d->front_cap)) need <<= 1;
            if (need > (1u << 30)) {
                d->unchecked = false;
                d->have_result = false;
                return oi_set_err(c, OIBVH_ERR_OVERFLOW, "BVTT front exceeds %u entries", 1u << 30);
            }
            dfree(d->front[0]);
            dfree(d->front[1]);
            d->front_cap = 0;
            d->generation++;
            HIPCHK(c, dalloc(&d->front[0], need));
            HIPCHK(c, dalloc(&d->front[1], need));
            d->front_cap = (uint32_t)need;
            d->want_front = d->front_cap;
            rerun = true;
        }
        if ((k.error & OI_ERR_CAND_OVERFLOW) || (!d->fused && k.cands > d->cand_cap)) {
            r = grow(c, d->cands, d->cand_cap, std::max<uint64_t>(k.cands, 2ull * d->cand_cap), d->generation);
            if (r != OIBVH_OK) return r;
            d->want_cands = d->cand_cap;
            rerun = true;
        }
        if ((k.error & OI_ERR_HITS_OVERFLOW) || k.n_hits > d->hits_cap) {
            const uint64_t need = std::max<uint64_t>((uint64_t)k.n_hits + (k.n_hits >> 3), 2ull * d->hits_cap);
            if ((r = grow(c, d->hits, d->hits_cap, need, d->generation)) != OIBVH_OK) return r;
            d->want_hits = d->hits_cap;
            rerun = true;
        }
        if (!rerun) {
            d->n_pairs = k.n_hits;
            d->stats.bvtt_tests = k.tests;
            d->stats.candidates = k.cands;
            d->stats.fp64_rechecks = k.fp64;
            d->stats.fp64_candidates = k.deferred;
            d->stats.adjacent = k.adj;
            d->stats.pairs = k.n_hits;
            d->stats.retries = retries;
            d->stats.async_errors = earlier;
            d->unchecked = false;
            d->sorted_ok = false;  // a new result: sorted again on demand
            judge_walk(d);
            return OIBVH_OK;
        }
        retries++;
        if (retries > 16) return oi_set_err(c, OIBVH_ERR_OVERFLOW, "detect: too many retries");
        if ((r = oi_det_prepare(d)) != OIBVH_OK) return r;
        if ((r = oi_det_enqueue(d, true)) != OIBVH_OK) return r;
    }
}

static uint32_t bits_for(uint32_t max_value)
{
    return max_value ? 32u - (uint32_t)__builtin_clz(max_value) : 0u;
}

// Lists up to this length are ranked in one launch (k_pairs_rank, n^2
// compares: 11 us at 5,100 pairs), longer ones sample sorted in five (27 us at
// 15,800); the two meet at about 9,000 pairs.
#define OI_PAIRS_RANK_MAX 9216u
// The sample sort's buckets hold about n / 1024 keys at this length, a quarter
// of what a workgroup sorts in LDS.
#define OI_PAIRS_SORT_MAX (1u << 20)

// The checked hits sorted on the device into d_sorted, in get_pairs order
// (meshA, meshB, triA, triB), once per query. Mesh ids are below the table's
// mesh count and face ids below its largest face count; where two of each fit
// into a 64-bit key, or the list is short, oibvh_pairs.hip sorts it, else LSD
// radix passes over the bytes that can be non-zero sort hit indices with keys
// looked up by index, then one gather.
// host (null, or room for OI_PAIRS_RANK_MAX pairs in pinned memory) receives a list
// of at most that length too, once the stream has run.
static oibvh_status sort_hits(oi_detector* d, uint4* host = nullptr)
{
    oibvh_ctx* c = d->ctx;
    const uint32_t n = d->n_pairs;
    if (d->sorted_ok || n == 0) return OIBVH_OK;
    if (n >= (1u << 30)) return oi_set_err(c, OIBVH_ERR_OVERFLOW, "pair sort: more than 2^30 pairs");
    uint32_t max_f = 1;
    for (uint32_t m = 0; m < d->tab.n_meshes; m++) max_f = std::max(max_f, d->tab.h_meshes[m].F);
    const uint32_t mbits = bits_for(d->tab.n_meshes ? d->tab.n_meshes - 1 : 0), tbits = bits_for(max_f - 1);
    uint64_t gen = 0;
    oibvh_status r;
    const bool wide = 2u * (mbits + tbits) > 64u;
    if (n <= OI_PAIRS_RANK_MAX || (n <= OI_PAIRS_SORT_MAX && !wide)) {
        const oi_pair_bits bits{mbits, tbits};
        if ((r = grow(c, d->d_sorted, d->d_sorted_cap, n, gen)) != OIBVH_OK) return r;
        if (n <= OI_PAIRS_RANK_MAX) {
            HIPCHK(c, oi_launch_pairs_rank(c->stream, d->hits, n, bits, wide, d->d_sorted, host));
        } else {
            if (d->sort_mem_cap < oi_pairs_sort_bytes(n)) {
                // sized with headroom, so that the next queries rarely grow it
                const uint64_t cap = oi_pairs_sort_bytes(std::min(OI_PAIRS_SORT_MAX, n + (n >> 2)));
                dfree(d->sort_mem);
                d->sort_mem_cap = 0;
                HIPCHK(c, dalloc(&d->sort_mem, cap));
                d->sort_mem_cap = cap;
            }
            HIPCHK(c, oi_launch_pairs_sort(c->stream, d->hits, n, bits, d->sort_mem, d->d_sorted));
        }
        d->sorted_ok = true;
        return OIBVH_OK;
    }
    oi_hit_digits dg{};
    for (uint32_t w : {3u, 2u, 1u, 0u}) {
        const uint32_t nb = ((w >= 2 ? tbits : mbits) + 7u) / 8u;
        for (uint32_t k = 0; k < nb; k++) {
            dg.word[dg.nd] = (uint8_t)w;
            dg.shift[dg.nd] = (uint8_t)(8u * k);
            dg.nd++;
        }
    }
    const uint32_t rows = (uint32_t)oi_sort_rows(1, oi_sort_tiles(1, &n));
    if (d->sort_cap < n) {
        // sized with headroom, so that the next queries rarely grow them
        const uint64_t cap = std::min<uint64_t>((1ull << 30) - 1, (uint64_t)n + (n >> 2));
        const uint64_t crows = oi_sort_rows(1, oi_sort_tiles_max(cap));
        dfree(d->sort_words);
        dfree(d->sort_vals);
        dfree(d->sort_scratch);
        d->sort_cap = 0;
        HIPCHK(c, dalloc(&d->sort_words, 4 * cap));
        HIPCHK(c, dalloc(&d->sort_vals, 2 * cap));
        HIPCHK(c, dalloc(&d->sort_scratch, 256ull * OI_HIT_DIGITS + OI_HIT_DIGITS + 512ull * crows));
        d->sort_cap = (uint32_t)cap;
    }
    if ((r = grow(c, d->d_sorted, d->d_sorted_cap, n, gen)) != OIBVH_OK) return r;
    uint32_t* hist = d->sort_scratch;
    uint32_t* tctr = hist + 256u * OI_HIT_DIGITS;
    uint32_t* lb[2] = {tctr + OI_HIT_DIGITS, tctr + OI_HIT_DIGITS + 256ull * rows};
    uint32_t* vals[2] = {d->sort_vals, d->sort_vals + d->sort_cap};
    hipStream_t st = c->stream;
    // histograms, tile counters and the first look-back buffer start at zero
    HIPCHK(c, oi_launch_zero_u32(st, hist, 256u * OI_HIT_DIGITS + OI_HIT_DIGITS + 256u * rows));
    HIPCHK(c, oi_launch_hits_digits(st, d->hits, n, d->sort_words, hist, &dg));
    const uint32_t* order = nullptr;  // identity
    for (uint32_t p = 0; p < dg.nd; p++) {
        HIPCHK(c, oi_launch_sort_pass(st, nullptr, order, nullptr, vals[p & 1], n, dg.shift[p], hist + 256u * p, 1u,
                                      lb[p & 1], p + 1 < dg.nd ? lb[(p + 1) & 1] : nullptr, tctr + p,
                                      d->sort_words + (uint64_t)n * dg.word[p]));
        order = vals[p & 1];
    }
    if (order) {
        HIPCHK(c, oi_launch_hits_gather(st, d->hits, order, n, d->d_sorted));
    } else {
        // one mesh of one face: at most one distinct pair
        HIPCHK(c, hipMemcpyAsync(d->d_sorted, d->hits, n * sizeof(uint4), hipMemcpyDeviceToDevice, st));
    }
    d->sorted_ok = true;
    return OIBVH_OK;
}

oibvh_status oi_det_get_pairs(oi_detector* d, uint32_t* out, uint64_t cap, uint32_t* n)
{
    oibvh_ctx* c = d->ctx;
    oibvh_status r = oi_det_check(d);
    if (r != OIBVH_OK) return r;
    if (n) *n = d->n_pairs;
    if (d->n_pairs == 0) return OIBVH_OK;
    if (!out || cap < d->n_pairs) return oi_set_err(c, OIBVH_ERR_CAPACITY, "need %u pairs", d->n_pairs);
    if (!d->sorted_ok && d->n_pairs <= OI_PAIRS_RANK_MAX) {
        // a short list is written to pinned memory by the launch that ranks it; a copy
        // and the wait for it took 10 us more with 107 pairs, 40 with 1,500 (16 KB and
        // more are staged)
        if (!d->h_pairs)
            HIPCHK(c, hipHostMalloc((void**)&d->h_pairs, OI_PAIRS_RANK_MAX * sizeof(uint4),
                                    hipHostMallocCoherent | hipHostMallocMapped));
        if ((r = sort_hits(d, d->h_pairs)) != OIBVH_OK) return r;
        if ((r = finish(d)) != OIBVH_OK) return r;
        std::memcpy(out, d->h_pairs, d->n_pairs * sizeof(uint4));
        return OIBVH_OK;
    }
    if ((r = sort_hits(d)) != OIBVH_OK) return r;
    HIPCHK(c, hipMemcpyAsync(out, d->d_sorted, d->n_pairs * sizeof(uint4), hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return OIBVH_OK;
}

oibvh_status oi_det_sorted_device(oi_detector* d, const uint4** dptr, uint32_t* n)
{
    oibvh_status r = oi_det_check(d);
    if (r != OIBVH_OK) return r;
    if ((r = sort_hits(d)) != OIBVH_OK) return r;
    // the sort runs on the context's stream: complete it before the pointer
    // is handed to a consumer on any stream or the host
    if ((r = finish(d)) != OIBVH_OK) return r;
    *dptr = d->d_sorted;
    *n = d->n_pairs;
    return OIBVH_OK;
}

oibvh_status oi_det_pair_vertices(oi_detector* d, const oi_build_desc* geom, float* out, uint64_t cap,
                                  uint32_t ptr_kind, uint32_t* n)
{
    oibvh_ctx* c = d->ctx;
    if (ptr_kind != OIBVH_PTR_HOST && ptr_kind != OIBVH_PTR_DEVICE)
        return oi_set_err(c, OIBVH_ERR_INVALID, "pair vertices: ptr_kind must be HOST or DEVICE");
    oibvh_status r = oi_det_check(d);
    if (r != OIBVH_OK) return r;
    if (n) *n = d->n_pairs;
    if (d->n_pairs == 0) return OIBVH_OK;
    const uint64_t need = 18ull * d->n_pairs;
    if (!out || cap < need) return oi_set_err(c, OIBVH_ERR_CAPACITY, "need %llu floats", (unsigned long long)need);
    if ((r = sort_hits(d)) != OIBVH_OK) return r;
    float* dst = out;
    if (ptr_kind == OIBVH_PTR_HOST) {
        if (d->stage_cap < need) {
            dfree(d->d_stage);
            d->stage_cap = 0;
            HIPCHK(c, dalloc(&d->d_stage, need));
            d->stage_cap = need;
        }
        dst = d->d_stage;
    }
    HIPCHK(c, oi_launch_pair_vertices(c->stream, geom, d->d_sorted, d->n_pairs, dst));
    if (ptr_kind == OIBVH_PTR_HOST) {
        HIPCHK(c, hipMemcpyAsync(out, d->d_stage, need * sizeof(float), hipMemcpyDeviceToHost, c->stream));
        HIPCHK(c, hipStreamSynchronize(c->stream));
        return OIBVH_OK;
    }
    return finish(d);  // device output is complete when this returns
}

oibvh_status oi_det_level_counts(oi_detector* d, uint32_t* out, uint64_t cap, uint32_t* n)
{
    oibvh_status r = oi_det_check(d);
    if (r != OIBVH_OK) return r;
    *n = d->have_result ? d->n_levels : 0;
    if (*n == 0) return OIBVH_OK;
    if (!out || cap < *n) return oi_set_err(d->ctx, OIBVH_ERR_CAPACITY, "need %u entries", *n);
    std::memcpy(out, d->h_counts.data(), *n * sizeof(uint32_t));
    return OIBVH_OK;
}
