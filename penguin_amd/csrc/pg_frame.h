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
// fields where that is more, allocated by the first frame that needs them and
// freed with the handle.  One frame at a time (a handle is used by one host
// thread).
struct FrameBuf {
    static constexpr int NBUF = 3;
    static constexpr size_t LEAST = (size_t)1 << 20, MOST = (size_t)8 << 20;   // of a piece
    char* mem[NBUF] = {nullptr, nullptr, nullptr};
    bool pinned = false;
    size_t piece = 0;   // bytes of one piece
    int nbuf = 0;       // pieces held
    size_t threads = 0; // that converted the last frame
    hipEvent_t ev[NBUF] = {nullptr, nullptr, nullptr};

    void drop() {
        for (char*& m : mem) {
            if (m && pinned) (void)hipHostFree(m);
            else std::free(m);
            m = nullptr;
        }
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
    bool allocate(size_t bytes, int n, bool pin) {
        pinned = pin;
        for (int k = 0; k < n; ++k) {
            if (pin ? hipHostMalloc((void**)&mem[k], bytes, hipHostMallocDefault) != hipSuccess
                    : !(mem[k] = (char*)std::malloc(bytes))) {
                mem[k] = nullptr;
                if (pin) (void)hipGetLastError();
                drop();
                return false;
            }
        }
        piece = bytes;
        nbuf = n;
        return true;
    }
    // n pieces of `bytes`; a frame of one piece needs neither more nor an event,
    // nor pinned memory, whose allocation and release cost as much as several
    // such frames (64x128 FP32: first read 30 us, 53 pinned, every other 22
    // either way; 192x384, 0.9 MB: 111 and 127, then 104 and 84).  A piece is an
    // allocation of its own: up to 1 MB they take some 35 us each, one of 3 MB
    // takes 0.1 or 1 ms (first read of a 256x512 FP32 disk, 1.6 MB: 210-240 us,
    // with its pieces in one block 200 or 820-1140; of a 256x512 FP64 one 290
    // and 280 or 1410).  Without pinned memory the runtime stages the copies.
    hipError_t reserve(size_t bytes, int n) {
        for (int k = 0; k < n && n > 1; ++k)
            if (!ev[k]) {
                const hipError_t r = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
                if (r != hipSuccess) {
                    ev[k] = nullptr;
                    return r;
                }
            }
        if (piece >= bytes && nbuf >= n) return hipSuccess;
        bytes = std::max(bytes, piece);   // disks of a batch share the pieces
        n = std::max(n, nbuf);
        drop();
        return (n > 1 && allocate(bytes, n, true)) || allocate(bytes, n, false) ? hipSuccess : hipErrorOutOfMemory;
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
    // 2.5 ms slower with 4 MB pieces than with 1 MB; every frame of a 256x512
    // FP32 disk 240 us with pieces of a third of a megabyte, 165 with 1 MB)
    const size_t bytes = std::min(FrameBuf::MOST, std::max(FrameBuf::LEAST, rows * row * nf / 16));
    const size_t per = std::min(rows, std::max<size_t>(1, bytes / (row * nf)));   // rows of a piece
    const size_t npiece = (rows + per - 1) / per;
    hipError_t err = fb.reserve(per * row * nf, (int)std::min<size_t>(npiece, FrameBuf::NBUF));
    if (err != hipSuccess) return err;
    auto first = [&](size_t c) { return c * per; };
    auto count = [&](size_t c) { return std::min(rows, (c + 1) * per) - c * per; };
    auto buf = [&](size_t c) { return fb.mem[c % FrameBuf::NBUF]; };
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
