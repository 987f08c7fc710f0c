// Copies between device arrays and pageable host arrays through pinned chunks.
//
// A plain hipMemcpy to or from pageable memory runs on one host thread: the
// runtime's own staging copy, and for a fresh destination a page fault every
// few KB (150 ms for the 0.6 GB state of 256^2 x 129).  Here up to THREADS host
// threads each move chunks of CHUNK bytes: one thread's host copy overlaps the
// others' transfers, so the device link stays busy.  Writing a state
// of 108 x 96 x 49 as volumes and reading it back took 37.2 ms and takes 9.7; the
// quadratic spectra and physical fields of 96 x 96 x 48 took 29.6 and take 4.8.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <exception>
#include <mutex>
#include <stdexcept>
#include <string>
#include <system_error>
#include <thread>
#include <vector>

namespace coral {

class HostCopy {
  public:
    static constexpr size_t CHUNK = size_t(1) << 20;
    static constexpr int THREADS = 8;

    HostCopy() = default;
    HostCopy(const HostCopy &) = delete;
    HostCopy &operator=(const HostCopy &) = delete;
    ~HostCopy() {
        for (auto &b : bufs_) {
            if (b.ev) (void)hipEventDestroy(b.ev);
            if (b.p) (void)hipHostFree(b.p);
        }
    }

    // nrow rows of row_bytes, contiguous on the device, to host addresses dst(row);
    // after everything queued on st, and complete on return.  fill(part, parts)
    // does a share of further host work (clearing what no row covers).
    template <class Dst, class Fill>
    void to_host(hipStream_t st, int device, const void *dev, size_t nrow, size_t row_bytes, Dst dst, Fill fill) {
        const char *src = static_cast<const char *>(dev);
        run(device, nrow, row_bytes, fill, [&](Buf &b, size_t r0, size_t r1) {
            check(hipMemcpyAsync(b.p, src + r0 * row_bytes, (r1 - r0) * row_bytes, hipMemcpyDeviceToHost, st));
            check(hipEventRecord(b.ev, st));
            check(hipEventSynchronize(b.ev));
            for (size_t r = r0; r < r1; ++r)
                std::memcpy(dst(r), static_cast<char *>(b.p) + (r - r0) * row_bytes, row_bytes);
        });
    }

    // rows from host addresses src(row) to the device, queued on st and complete
    // on return
    template <class Src>
    void to_device(hipStream_t st, int device, void *dev, size_t nrow, size_t row_bytes, Src src) {
        char *d = static_cast<char *>(dev);
        run(device, nrow, row_bytes, [](int, int) {}, [&](Buf &b, size_t r0, size_t r1) {
            for (size_t r = r0; r < r1; ++r)
                std::memcpy(static_cast<char *>(b.p) + (r - r0) * row_bytes, src(r), row_bytes);
            check(hipMemcpyAsync(d + r0 * row_bytes, b.p, (r1 - r0) * row_bytes, hipMemcpyHostToDevice, st));
            check(hipEventRecord(b.ev, st));
            check(hipEventSynchronize(b.ev));
        });
    }

  private:
    struct Buf {
        void *p = nullptr;
        size_t bytes = 0;
        hipEvent_t ev = nullptr;
    };
    std::vector<Buf> bufs_;

    static void check(hipError_t e) {
        if (e != hipSuccess) throw std::runtime_error(std::string("host copy: ") + hipGetErrorString(e));
    }

    template <class Fill, class Move>
    void run(int device, size_t nrow, size_t row_bytes, Fill fill, Move move) {
        if (nrow == 0 || row_bytes == 0) {
            fill(0, 1);
            return;
        }
        const size_t per = std::max<size_t>(1, CHUNK / row_bytes), nchunk = (nrow + per - 1) / per;
        const int nt = int(std::min<size_t>(THREADS, nchunk));
        if (bufs_.size() < size_t(nt)) bufs_.resize(nt);
        for (int t = 0; t < nt; ++t) {
            Buf &b = bufs_[t];
            if (b.bytes < per * row_bytes) {
                if (b.p) check(hipHostFree(b.p));
                b.p = nullptr;
                b.bytes = 0;
                check(hipHostMalloc(&b.p, std::max(CHUNK, per * row_bytes), hipHostMallocDefault));
                b.bytes = std::max(CHUNK, per * row_bytes);
            }
            if (!b.ev) check(hipEventCreateWithFlags(&b.ev, hipEventDisableTiming));
        }
        std::mutex mu;
        std::exception_ptr err;
        auto work = [&](int t) {
            try {
                check(hipSetDevice(device));
                fill(t, nt);
                for (size_t c = t; c < nchunk; c += nt) move(bufs_[t], c * per, std::min(nrow, (c + 1) * per));
            } catch (...) {
                std::lock_guard<std::mutex> g(mu);
                if (!err) err = std::current_exception();
            }
        };
        std::vector<std::thread> team;
        team.reserve(nt);
        int started = 1;   // the calling thread takes share 0
        try {
            for (; started < nt; ++started) team.emplace_back(work, started);
        } catch (const std::system_error &) {
            // no more threads to be had: the shares left over run here
        }
        work(0);
        for (int t = started; t < nt; ++t) work(t);
        for (auto &th : team) th.join();
        if (err) std::rethrow_exception(err);
    }
};

}  // namespace coral
