// The plan of a query's walks before and after a check has read the front lengths:
// walks that were guessed far too short become steps, and those guessed right stay.
#include <cstdio>
#include <string>

#include "oibvh_detect.cpp"

static std::vector<uint32_t> lengths;  // what the next check reads
static oi_published published;

hipError_t oi_ctx_join(oibvh_ctx*) { return hipSuccess; }
extern "C" hipError_t hipGetDeviceFlags(unsigned* flags) { return *flags = 0, hipSuccess; }
extern "C" hipError_t oi_launch_publish(hipStream_t, const oi_publish_args* a)
{
    std::copy(lengths.begin(), lengths.end(), a->out->counts);
    a->out->seq = a->seq;
    return hipSuccess;
}

struct Query {
    oibvh_ctx c;
    oi_detector d;
    oi_detect_ctl ctl;
    uint2 pairs;
    Query(uint32_t n_front, uint32_t depth, uint32_t expand, uint32_t flags = 0)
    {
        c.cus = 256;
        d.ctx = &c;
        d.ctl_base = d.ctl = &ctl;
        d.h_pub = &published;
        d.n_front = n_front;
        d.depth = depth;
        d.expand = expand;
        d.flags = flags;
        d.front[0] = d.front[1] = &pairs;
        d.front_cap = d.counts_cap = d.cand_cap = d.hits_cap = 1u << 30;
    }
    // one letter per step: 1 a walk of one step, 2 and . one of two, s a step
    std::string plan()
    {
        std::string p;
        if (oi_det_prepare(&d) != OIBVH_OK) return "?";
        for (uint32_t k = 0; k < d.n_levels; k++) {
            const uint32_t w = d.step_walk[k] & 3u;
            p += w == 0 ? "s" : w == 1 ? "1" : "2.";
            k += w == 2;
        }
        return p;
    }
    // a query of this plan that met fronts of these lengths
    bool run(std::vector<uint32_t> fronts)
    {
        d.unchecked = true;
        lengths = fronts;
        lengths.push_back(0);
        return oi_det_check(&d) == OIBVH_OK;
    }
};

static int bad = 0;
static void expect(const char* what, const std::string& got, const std::string& want)
{
    if (got != want) std::printf("%s: %s, not %s\n", what, got.c_str(), want.c_str()), bad = 1;
}

int main()
{
    // two overlapping clouds of 200,000 triangles each: the guess merges steps two
    // and three, which met 41,160 and 368,543 pairs
    const std::vector<uint32_t> dense = {169, 3266, 41160, 368543, 1546835};
    Query q(169, 14, 3);
    expect("guess", q.plan(), "2.2.s");
    uint64_t gen = q.d.generation;
    if (!q.run(dense)) return 1;
    expect("after a dense query", q.plan(), "2.1ss");
    if (q.d.generation == gen) std::printf("a captured query would keep its plan\n"), bad = 1;
    gen = q.d.generation;
    if (!q.run(dense)) return 1;
    expect("after another", q.plan(), "2.1ss");
    if (q.d.generation != gen) std::printf("the same lengths again changed the plan\n"), bad = 1;
    // lengths between the guess's limits and the far ones: the plan stays
    if (!q.run({169, 1200, 7000, 50000, 200000})) return 1;
    expect("after a query in between", q.plan(), "2.1ss");
    // as the guess takes them to grow
    if (!q.run({169, 600, 2000, 9000, 30000})) return 1;
    expect("after a sparse one", q.plan(), "2.2.s");
    if (!q.run({169, 1200, 7000, 45000, 100000})) return 1;
    expect("a little longer than guessed", q.plan(), "2.2.s");

    // a walk of one step, over fewer and over more than 2^18 pairs
    Query w(4000, 12, 3);
    expect("one step", w.plan(), "2.1s");
    if (!w.run({4000, 20000, 200000, 500000})) return 1;
    expect("longer, not far", w.plan(), "2.1s");
    if (!w.run({4000, 20000, 300000, 500000})) return 1;
    expect("far longer", w.plan(), "2.ss");

    // another query of the same detector starts from the guess
    if (!q.run(dense)) return 1;
    q.d.expand = 2;
    expect("two levels a step", q.plan(), Query(169, 14, 2).plan());
    q.d.expand = 3;
    expect("and three again", q.plan(), "2.2.s");

    // settings without walks are not judged
    Query t(169, 14, 3);
    t.c.trav_tail = 64;
    t.plan();
    gen = t.d.generation;
    if (!t.run(dense)) return 1;
    if (t.d.generation != gen) std::printf("a tail walk was judged\n"), bad = 1;
    t.c.trav_tail = 0;
    expect("without the tail walk", t.plan(), "2.2.s");
    return bad;
}
