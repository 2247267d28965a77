// pg_hostcheck.cpp -- host code of the library run on the CPU, for its tests:
// the frame reader (pg_frame.h) over a stand-in for the HIP calls it makes, and
// the choice of the 3D radial sweep's tile.
// Part of libpg_adjcheck.so; the product library does not contain it.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <set>
#include <thread>
#include <utility>
#include <vector>

namespace fake {

// One stream.  A copy happens when it is asked for (late = 0) or only when the
// host waits for it (late = 1): between the two lies every moment a device
// could choose.
struct Copy {
    void* dst;
    const void* src;
    size_t n;
};
struct Device {
    int late = 0, refuse_pinned = 0, fail_copy = -1;
    std::vector<Copy> queue;
    size_t done = 0;                          // copies of the queue that have happened
    std::vector<size_t> mark = std::vector<size_t>(64, 0);   // per event: the queue's length at its record
    int nevent = 0, ncopy = 0, nalloc = 0;
    long pinned = 0, most = 0, block = 0;     // bytes allocated now, ever at once, and in one block
    std::vector<std::pair<void*, size_t>> live;
} dev;

void run_to(size_t n) {
    for (; dev.done < n; ++dev.done) std::memcpy(dev.queue[dev.done].dst, dev.queue[dev.done].src, dev.queue[dev.done].n);
}
hipError_t host_malloc(void** p, size_t n, unsigned) {
    if (dev.refuse_pinned && dev.nalloc >= dev.refuse_pinned - 1) return hipErrorOutOfMemory;
    *p = std::malloc(n);
    ++dev.nalloc;
    dev.live.push_back({*p, n});
    dev.pinned += (long)n;
    dev.most = std::max(dev.most, dev.pinned);
    dev.block = std::max(dev.block, (long)n);
    return hipSuccess;
}
hipError_t host_free(void* p) {
    for (size_t k = 0; k < dev.live.size(); ++k)
        if (dev.live[k].first == p) {
            dev.pinned -= (long)dev.live[k].second;
            dev.live.erase(dev.live.begin() + k);
            std::free(p);
            return hipSuccess;
        }
    std::abort();   // not memory of host_malloc
}
hipError_t copy(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    if (dev.ncopy++ == dev.fail_copy) return hipErrorInvalidValue;
    dev.queue.push_back({d, s, n});
    if (!dev.late) run_to(dev.queue.size());
    return hipSuccess;
}
hipError_t event_create(hipEvent_t* e, unsigned) {
    *e = (hipEvent_t)(size_t)++dev.nevent;
    return hipSuccess;
}
hipError_t event_destroy(hipEvent_t) {
    --dev.nevent;
    return hipSuccess;
}
hipError_t event_record(hipEvent_t e, hipStream_t) {
    dev.mark[(size_t)e] = dev.queue.size();
    return hipSuccess;
}
hipError_t event_wait(hipEvent_t e) {
    run_to(dev.mark[(size_t)e]);
    return hipSuccess;
}
hipError_t stream_wait(hipStream_t) {
    run_to(dev.queue.size());
    return hipSuccess;
}
hipError_t last_error() { return hipSuccess; }

}  // namespace fake

#define hipHostMalloc fake::host_malloc
#define hipHostFree fake::host_free
#define hipMemcpyAsync fake::copy
#define hipEventCreateWithFlags fake::event_create
#define hipEventDestroy fake::event_destroy
#define hipEventRecord fake::event_record
#define hipEventSynchronize fake::event_wait
#define hipStreamSynchronize fake::stream_wait
#define hipGetLastError fake::last_error
#include "pg_frame.h"
#include "pg_sph.h"

extern "C" {

// `reads` reads of nf fields of rows x nx floats at src through one FrameBuf,
// converted to doubles at dst; the last one fails at its fail_copy-th copy if
// that is not negative, and the refuse_pinned-th pinned allocation and all after
// it are refused if that is not zero.  Returns the last read's error.  stats:
// copies of the last read, pinned allocations, most pinned bytes at once, pinned
// bytes and events left after the release, threads that converted rows in the
// last read, threads that it was given, bytes of the largest pinned allocation.
int hostcheck_frame(long rows, long nx, int nf, int reads, int late, int refuse_pinned, int fail_copy,
                    const float* src, double* dst, long* stats) {
    fake::dev = fake::Device();
    fake::dev.late = late;
    fake::dev.refuse_pinned = refuse_pinned;
    pg::FrameBuf fb;
    hipError_t e = hipSuccess;
    const size_t N = (size_t)rows * nx;
    std::mutex mu;
    std::set<std::thread::id> ids;
    for (int k = 0; k < reads && e == hipSuccess; ++k) {
        fake::dev.ncopy = 0;
        fake::dev.fail_copy = k == reads - 1 ? fail_copy : -1;
        ids.clear();
        e = pg::read_frame(fb, (hipStream_t) nullptr, src, N * sizeof(float), nf, (size_t)rows, (size_t)nx, sizeof(float),
                           [&](const char* p, size_t m, size_t r0, size_t r1) {
            {
                std::lock_guard<std::mutex> lk(mu);
                ids.insert(std::this_thread::get_id());
            }
            for (size_t r = r0; r < r1; ++r, p += nx * sizeof(float))
                for (int f = 0; f < nf; ++f)
                    for (long i = 0; i < nx; ++i) dst[f * N + r * nx + i] += (double)((const float*)(p + f * m))[i];
        });
    }
    stats[0] = fake::dev.ncopy;
    stats[1] = fake::dev.nalloc;
    stats[2] = fake::dev.most;
    fb.release();
    stats[3] = fake::dev.pinned;
    stats[4] = fake::dev.nevent;
    stats[5] = (long)ids.size();
    stats[6] = (long)fb.threads;
    stats[7] = fake::dev.block;
    return (int)e;
}

// Cells of a segment, rows of a block and row multiplier of the radial sweep of
// a disk of nx radii in `rows` rows, es bytes a real.
void hostcheck_radial_tile(int nx, long rows, int es, int* out) {
    const pg::RadialTile t = pg::radial_tile(nx, rows, es);
    out[0] = t.tx;
    out[1] = t.xr;
    out[2] = t.xm;
}

}  // extern "C"
