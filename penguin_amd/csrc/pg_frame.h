// pg_frame.h -- reading a state back to the caller's FP64 arrays.
//
// A frame leaves the device in the storage precision and in pieces of a few
// megabytes through pinned buffers, so that the transfer of one piece runs
// beside the conversion of the one before it, and the conversion is shared by
// several host threads: it writes two to four times the bytes that cross the
// bus, into pages that the caller has often just allocated, at a rate that one
// thread is far from (a 1024x3072 gas and dust disk in FP32, 75 MB over the
// bus and 226 MB written: 70 ms by one thread through pageable memory, 4.7 ms
// here; a 384x1536x64 disk, 755 MB and 1.5 GB: 330 -> 29 ms).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <condition_variable>
#include <cstddef>
#include <cstdlib>
#include <mutex>
#include <thread>
#include <vector>

namespace pg {

// The pieces of one handle: at most NBUF of MOST bytes, or of one row of all
// fields where that is more, allocated by the first frame, pinned if it reads enough through them and the system gives pinned
// memory, and freed with the handle.  One frame at a time (a handle is used by
// one host thread).
struct FrameBuf {
    static constexpr int NBUF = 3;
    static constexpr size_t LEAST = (size_t)1 << 20, MOST = (size_t)8 << 20;   // of a piece
    static constexpr size_t PIN_FROM = (size_t)4 << 20;   // bytes read
    char* mem = nullptr;
    bool pinned = false, refused = false;
    size_t read = 0;    // bytes of all frames so far
    size_t piece = 0;   // bytes of one piece
    int nbuf = 0;       // pieces held
    size_t threads = 0; // that converted the last frame
    hipEvent_t ev[NBUF] = {nullptr, nullptr, nullptr};

    void drop() {
        if (mem && pinned) (void)hipHostFree(mem);
        else std::free(mem);
        mem = nullptr;
        piece = 0;
        nbuf = 0;
    }
    void release() {
        drop();
        for (hipEvent_t& e : ev) {
            if (e) (void)hipEventDestroy(e);
            e = nullptr;
        }
    }
    // n buffers of `bytes` for a frame of `frame` bytes; a frame of one piece
    // needs neither more nor an event, nor pinned memory, whose allocation and
    // release cost as much as several such frames (64x128 FP32: first read 30
    // us, 53 pinned, every other 22 either way; 192x384, 0.9 MB: 111 and 127,
    // then 104 and 84).  Pieces are pinned once the handle has read 4 MB, this
    // frame included: three of 1 MB take 0.1-1 ms to allocate and gain 0.05-0.1
    // ms for each MB read (256x512 FP32, 1.6 MB: first read 250 us, pinned
    // 200-1200, then 230 and 165 a frame; 333x777 FP64 gas and dust, 12 MB: 1.9
    // ms, pinned 1.3; 1024x3072 FP32 gas, 38 MB: 4.7 ms, pinned 3.6, then 2.9).
    hipError_t reserve(size_t bytes, int n, size_t frame) {
        for (hipEvent_t& e : ev)
            if (!e && n > 1) {
                const hipError_t r = hipEventCreateWithFlags(&e, hipEventDisableTiming);
                if (r != hipSuccess) {
                    e = nullptr;
                    return r;
                }
            }
        read += frame;
        const bool pin = pinned || (n > 1 && read >= PIN_FROM && !refused);
        if (piece >= bytes && nbuf >= n && pin == pinned) return hipSuccess;
        bytes = std::max(bytes, piece);   // disks of a batch share the buffers
        n = std::max(n, nbuf);
        drop();
        pinned = pin && hipHostMalloc((void**)&mem, n * bytes, hipHostMallocDefault) == hipSuccess;
        if (!pinned) {   // a frame can be read without: the copies are then staged by the runtime
            if (pin) (void)hipGetLastError();
            refused = pin;
            mem = (char*)std::malloc(n * bytes);
            if (!mem) return hipErrorOutOfMemory;
        }
        piece = bytes;
        nbuf = n;
        return hipSuccess;
    }
};

// nf fields of rows x nx values of `es` bytes at dev (field stride fstride
// bytes), as they are on stream s when its earlier work is done.
// convert(src, m, r0, r1) is called, from several threads at once, for runs of
// rows [r0, r1) that cover every row once: src is the host copy of row r0 of
// field 0, field f of it f * m bytes on.
template <typename F>
hipError_t read_frame(FrameBuf& fb, hipStream_t s, const void* dev, size_t fstride, int nf, size_t rows, size_t nx,
                      size_t es, F convert) {
    const size_t row = nx * es;
    // sixteen pieces or pieces of MOST: pinned pages cost the first frame about
    // 0.2 ms a megabyte, and small pieces more waits (the 1.5 GB frame: 29 ms
    // with 8 MB pieces, 45 with 2 MB; the first frame of a 512x1024 FP64 disk
    // 2.5 ms slower with 4 MB pieces than with 1 MB)
    const size_t bytes = std::min(FrameBuf::MOST, std::max(FrameBuf::LEAST, rows * row * nf / 16));
    const size_t per = std::min(rows, std::max<size_t>(1, bytes / (row * nf)));   // rows of a piece
    const size_t npiece = (rows + per - 1) / per;
    hipError_t err = fb.reserve(per * row * nf, npiece > 1 ? FrameBuf::NBUF : 1, rows * row * nf);
    if (err != hipSuccess) return err;
    auto first = [&](size_t c) { return c * per; };
    auto count = [&](size_t c) { return std::min(rows, (c + 1) * per) - c * per; };
    auto buf = [&](size_t c) { return fb.mem + (c % FrameBuf::NBUF) * fb.piece; };
    auto fetch = [&](size_t c) {
        const size_t w = count(c) * row;
        const bool whole = w == fstride;   // one piece of all fields: they adjoin on the device too
        for (int f = 0; f < (whole ? 1 : nf); ++f) {
            const hipError_t e = hipMemcpyAsync(buf(c) + f * w, (const char*)dev + f * fstride + first(c) * row,
                                                whole ? nf * w : w, hipMemcpyDeviceToHost, s);
            if (e != hipSuccess) return e;
        }
        return npiece > 1 ? hipEventRecord(fb.ev[c % FrameBuf::NBUF], s) : hipSuccess;
    };
    // 256k cells a thread: a small frame pays for no thread.  Threads of fewer
    // cells read a frame alone faster, but not beside a caller's own pool that
    // is still spinning: a pass that reads 24 disks of 33k-786k cells and has
    // torch convert each takes 142 ms, with threads of 128k cells 164, of 32k 206.
    const size_t hw = std::max(1u, std::thread::hardware_concurrency());
    // A thread takes whole rows of a piece, so no more threads than those.
    const size_t want = std::min({hw, (size_t)8, per, std::max<size_t>(1, rows * nx / 262144)});
    std::mutex mu;
    std::condition_variable cv;
    size_t ready = 0;                      // pieces that have arrived
    size_t left[FrameBuf::NBUF] = {0, 0, 0};   // threads still reading the piece in each buffer
    bool stop = false;
    size_t nt = 0;
    std::vector<std::thread> th;
    auto slice = [&](size_t c, size_t k) {
        const size_t n = count(c), a = n * k / nt, b = n * (k + 1) / nt;
        if (a < b) convert(buf(c) + a * row, n * row, first(c) + a, first(c) + b);
    };
    auto work = [&](size_t k) {
        for (size_t c = 0; c < npiece; ++c) {
            {
                std::unique_lock<std::mutex> lk(mu);
                cv.wait(lk, [&] { return stop || ready > c; });
                if (stop) return;
            }
            slice(c, k);
            std::lock_guard<std::mutex> lk(mu);
            if (--left[c % FrameBuf::NBUF] == 0) cv.notify_all();
        }
    };
    if (want > 1) {
        // the threads wait for the first piece, so nt is set before any reads it;
        // one that cannot be started is done without
        try {
            th.reserve(want);
            for (size_t k = 0; k < want; ++k) th.emplace_back(work, k);
        } catch (...) {
        }
    }
    fb.threads = nt = std::max<size_t>(1, th.size());
    size_t asked = 0;
    for (size_t c = 0; c < npiece && err == hipSuccess; ++c) {
        // keep the free buffers on their way; piece `asked` takes the buffer of
        // a piece below c, which has been handed out: free once it is read
        while (asked < npiece && asked < c + FrameBuf::NBUF && err == hipSuccess) {
            {
                std::unique_lock<std::mutex> lk(mu);
                const size_t& busy = left[asked % FrameBuf::NBUF];
                if (busy && asked > c) break;   // piece c is on its way already
                cv.wait(lk, [&] { return busy == 0; });
            }
            err = fetch(asked);
            if (err == hipSuccess) ++asked;
        }
        if (err == hipSuccess) err = npiece > 1 ? hipEventSynchronize(fb.ev[c % FrameBuf::NBUF]) : hipStreamSynchronize(s);
        if (err != hipSuccess) break;
        if (th.empty()) {
            slice(c, 0);
        } else {
            std::lock_guard<std::mutex> lk(mu);
            left[c % FrameBuf::NBUF] = nt;
            ready = c + 1;
            cv.notify_all();
        }
    }
    if (err != hipSuccess) {
        std::lock_guard<std::mutex> lk(mu);
        stop = true;
        cv.notify_all();
    }
    for (std::thread& t : th) t.join();
    if (err != hipSuccess) (void)hipStreamSynchronize(s);   // no copy in flight targets the buffers
    return err;
}

}  // namespace pg
