// Workgroups of a batch frame's collision query, alone and overlapped: beside the
// next frame's refit a query launches fewer. HIP calls and launches are replaced by
// ones that do nothing or write down their grids.
#include <cstdio>

#include "oibvh_batch.cpp"
#include "oibvh_detect.cpp"

static uint32_t most_step, most_walk;

extern "C" {
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { return *g = (hipGraph_t)1, hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t)
{
    return *e = (hipGraphExec_t)1, hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned int) { return hipSuccess; }
hipError_t oi_launch_reduce(hipStream_t, int, const oi_build_desc*, const uint2*, const oi_build_desc*, uint32_t,
                            const uint32_t*, uint32_t, hipEvent_t, hipEvent_t, uint32_t)
{
    return hipSuccess;
}
hipError_t oi_launch_seed(hipStream_t, uint32_t, uint32_t*, uint32_t, oi_detect_ctl*, uint32_t) { return hipSuccess; }
hipError_t oi_launch_bvtt_step(hipStream_t, uint32_t grid, const oi_tab_args*, int, const uint2*, const uint32_t*,
                               uint32_t, uint32_t, uint2*, uint32_t*, uint32_t, uint2*, uint32_t*, uint32_t, uint4*,
                               uint32_t, oi_detect_ctl*, uint32_t, uint32_t, int, hipEvent_t)
{
    most_step = std::max(most_step, grid);
    return hipSuccess;
}
hipError_t oi_launch_bvtt_walk(hipStream_t, uint32_t grid, const oi_tab_args*, const oi_walk_args* w, uint2*, uint32_t*,
                               uint32_t, uint4*, uint32_t, oi_detect_ctl*, uint32_t, int)
{
    most_walk = std::max(most_walk, std::max(grid, w->wgs_long));
    return hipSuccess;
}
}
hipError_t oi_ctx_join(oibvh_ctx*) { return hipSuccess; }
hipError_t oi_ctx_quiesce(oibvh_ctx*) { return hipSuccess; }
hipError_t oi_ctx_wait_tickets(oibvh_ctx*, const uint64_t*, uint32_t) { return hipSuccess; }
hipError_t oi_ctx_host_wait_tickets(oibvh_ctx*, const uint64_t*, uint32_t) { return hipSuccess; }
oibvh_status oi_ctx_side_init(oibvh_ctx*) { return OIBVH_OK; }

// one frame of a batch of two meshes of 2^20 leaves, 16 x 16 initial pairs
static bool frame(uint32_t expand, uint32_t flags)
{
    static uint2 pairs[1];
    static uint32_t counts[256 * OI_FRAME_DEPTH];
    static oi_detect_ctl ctl[OI_FRAME_DEPTH];
    static oi_build_desc desc[2];
    oibvh_ctx c;
    c.cus = 256;
    c.leaves_per_thread = 16;
    oibvh_batch b;
    b.ctx = &c;
    b.det.ctx = &c;
    b.built = true;
    b.n_scenes = 1;
    b.meshes.resize(2);
    for (oibvh_batch::Mesh& m : b.meshes) m.L = 20, m.F = 1u << 20;
    b.front_key[0] = 4;
    b.front_key[1] = 0;
    for (int k = 0; k < 2; k++) {
        b.slot[k].d_bdesc = desc + k;
        b.slot[k].h_mdesc.resize(2);
        b.slot[k].h_bdesc.resize(2);
    }
    b.reduce_M = 16;
    oi_detector& d = b.det;
    d.n_front = 256;
    d.counts_base = counts;
    d.ctl_base = d.ctl = ctl;
    d.front[0] = d.front[1] = pairs;
    d.front_cap = d.counts_cap = d.cand_cap = d.hits_cap = 1u << 30;
    most_step = most_walk = 0;
    const oibvh_status r = oibvh_batch_frame(&b, 4, expand, flags | OIBVH_DETECT_ASYNC);
    if (r != OIBVH_OK) std::printf("frame: status %d %s\n", (int)r, c.err.c_str());
    return r == OIBVH_OK;
}

int main()
{
    int bad = 0;
    for (uint32_t overlap : {0u, (uint32_t)OIBVH_FRAME_OVERLAP}) {
        // FP32 steps of two levels
        if (!frame(2, overlap)) return 1;
        if (most_step != (overlap ? 4u : 6u) * 256u)
            std::printf("overlap %u: %u workgroups a step\n", overlap, most_step), bad = 1;
        // walks of three levels over long fronts
        if (!frame(3, overlap)) return 1;
        if (most_walk != (overlap ? 2u : 4u) * 256u)
            std::printf("overlap %u: %u workgroups a walk\n", overlap, most_walk), bad = 1;
    }
    return bad;
}
