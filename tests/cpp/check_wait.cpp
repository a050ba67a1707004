// How a check waits for the GPU: on the published number, or, in a program that chose
// to block or yield in its waits, in the stream's own wait.
#include <cstdio>
#include <ctime>

#include "oibvh_detect.cpp"

static unsigned device_flags;
static bool gpu_done;  // the published number lands at once
static int syncs;
static oi_published published;
static uint32_t last_seq;

hipError_t oi_ctx_join(oibvh_ctx*) { return hipSuccess; }
extern "C" {
hipError_t hipGetDeviceFlags(unsigned* flags) { return *flags = device_flags, hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t)
{
    syncs++;
    published.seq = last_seq;
    return hipSuccess;
}
hipError_t oi_launch_publish(hipStream_t, const oi_publish_args* a)
{
    last_seq = a->seq;
    if (gpu_done) published.seq = last_seq;
    return hipSuccess;
}
}

int main()
{
    int bad = 0;
    for (unsigned flags : {(unsigned)hipDeviceScheduleAuto, (unsigned)hipDeviceScheduleSpin,
                           (unsigned)hipDeviceScheduleYield, (unsigned)hipDeviceScheduleBlockingSync,
                           (unsigned)(hipDeviceScheduleBlockingSync | hipDeviceMapHost)})
        for (bool done : {true, false}) {
            const bool blocks = flags & (hipDeviceScheduleYield | hipDeviceScheduleBlockingSync);
            device_flags = flags;
            gpu_done = done;
            syncs = 0;
            published.seq = 0;
            oibvh_ctx c;
            oi_detect_ctl ctl;
            oi_detector d;
            d.ctx = &c;
            d.ctl_base = d.ctl = &ctl;
            d.h_pub = &published;
            d.n_levels = 1;
            d.unchecked = true;
            const clock_t t0 = clock();
            if (oi_det_check(&d) != OIBVH_OK) return 1;
            const double ms = 1e3 * (double)(clock() - t0) / CLOCKS_PER_SEC;
            if (syncs != (blocks || !done ? 1 : 0) || (blocks && ms > 10.0))
                std::printf("flags %u, done %d: %d waits in the stream, %.1f ms of the CPU\n", flags, done, syncs, ms), bad = 1;
        }
    return bad;
}
