// Workgroups of a query's launches for the traverse_blocks settings: the launch
// functions are replaced by ones that write down their grids.
#include <cstdio>

#include "oibvh_detect.cpp"

struct Launch {
    bool walk;
    uint32_t grid, grid_long;
};
static std::vector<Launch> launches;

extern "C" {
hipError_t oi_launch_seed(hipStream_t, uint32_t, uint32_t*, uint32_t, oi_detect_ctl*, uint32_t) { return hipSuccess; }
hipError_t oi_launch_bvtt_step(hipStream_t, uint32_t grid, const oi_tab_args*, int, const uint2*, const uint32_t*,
                               uint32_t, uint32_t, uint2*, uint32_t*, uint32_t, uint2*, uint32_t*, uint32_t, uint4*,
                               uint32_t, oi_detect_ctl*, uint32_t, uint32_t, int, hipEvent_t)
{
    launches.push_back({false, grid, 0});
    return hipSuccess;
}
hipError_t oi_launch_bvtt_walk(hipStream_t, uint32_t grid, const oi_tab_args*, const oi_walk_args* w, uint2*, uint32_t*,
                               uint32_t, uint4*, uint32_t, oi_detect_ctl*, uint32_t, int)
{
    launches.push_back({true, grid, w->wgs_long});
    return hipSuccess;
}
}

// the launches of a query of two bodies (16 x 16 initial pairs, 16 levels)
static void query(oibvh_ctx* c, uint32_t blocks, uint32_t expand)
{
    c->trav_blocks = blocks;
    static uint2 pairs[1];
    static oi_detect_ctl ctl;
    oi_detector d;
    d.ctx = c;
    d.n_front = 256;
    d.depth = 16;
    d.expand = expand;
    d.front[0] = d.front[1] = pairs;
    d.ctl = &ctl;
    d.front_cap = d.counts_cap = d.cand_cap = d.hits_cap = 1u << 30;
    launches.clear();
    if (oi_det_prepare(&d) != OIBVH_OK || oi_det_enqueue(&d, true) != OIBVH_OK) std::printf("the query failed\n");
}

int main()
{
    static oibvh_ctx c;
    c.cus = 256;
    int bad = 0;
    for (uint32_t expand : {1u, 2u, 3u}) {
        query(&c, 0, expand);
        const std::vector<Launch> by_default = launches;
        bool walks = false;
        for (const Launch& l : by_default) walks |= l.walk;
        if (!walks) std::printf("expand %u: nothing walked\n", expand), bad = 1;
        for (uint32_t blocks : {1u, 64u, 700u, 4096u}) {
            query(&c, blocks, expand);
            if (launches.size() != by_default.size()) std::printf("expand %u: another plan\n", expand), bad = 1;
            for (size_t k = 0; k < launches.size(); k++) {
                const Launch &l = launches[k], &d = by_default[k];
                // a step takes the setting, a walk at most that many workgroups
                const bool ok = l.walk ? l.grid == std::min(blocks, d.grid) &&
                                             l.grid_long == (d.grid_long ? std::min(blocks, d.grid_long) : 0u)
                                       : l.grid == blocks;
                if (!ok)
                    std::printf("expand %u, traverse_blocks %u, launch %zu: %u / %u workgroups\n", expand, blocks, k,
                                l.grid, l.grid_long), bad = 1;
            }
        }
    }
    return bad;
}
