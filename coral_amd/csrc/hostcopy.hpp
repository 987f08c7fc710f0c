// Copies between device arrays and pageable host arrays through pinned chunks.
//
// A plain hipMemcpy to or from pageable memory runs on one host thread: the
// runtime's own staging copy, and for a fresh destination a page fault every
// few KB (150 ms for the 0.6 GB state of 256^2 x 129).  Here the calling thread
// moves chunks of CHUNK bytes between the device and up to SLOTS pinned slots,
// and up to THREADS more help it to copy them to or from the host array, so
// that the link and the host copies work at the same time.  Writing a state of
// 108 x 96 x 49 as volumes and reading it back took 37.2 ms and takes 10.3; the
// quadratic spectra and physical fields of 96 x 96 x 48 took 29.6 and take 5.0.
// Nothing waits for a helper that has taken no chunk: where a caller's numerical
// library keeps every core spinning for a while, a new thread first runs at the
// scheduler's next tick (a copy of 9 MB took 4 ms instead of 0.4 while it did).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <functional>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <string>
#include <thread>
#include <vector>

namespace coral {

class HostCopy {
  public:
    static constexpr size_t CHUNK = size_t(1) << 20;
    static constexpr size_t SLOTS = 8, THREADS = 8;

    HostCopy() = default;
    HostCopy(const HostCopy &) = delete;
    HostCopy &operator=(const HostCopy &) = delete;
    ~HostCopy() {
        for (auto &h : helpers_) h.thread.join();
        for (auto &e : ev_)
            if (e) (void)hipEventDestroy(e);
        if (slab_) (void)hipHostFree(slab_);
    }

    // nrow rows of row_bytes, contiguous on the device, to host addresses dst(row);
    // after everything queued on st, and complete on return.  fill(part, parts)
    // does a share of further host work (clearing what no row covers).
    template <class Dst, class Fill>
    void to_host(hipStream_t st, const void *dev, size_t nrow, size_t row_bytes, Dst dst, Fill fill) {
        if (nrow == 0 || row_bytes == 0) return fill(0, 1);
        std::lock_guard<std::mutex> one(use_);
        const Plan p = plan(nrow, row_bytes);
        Task task(*this, p.nchunk, 0, fill, [&](size_t c) {
            const char *s = slot(p, c);
            for (size_t r = c * p.per; r < p.end(c); ++r, s += row_bytes) std::memcpy(dst(r), s, row_bytes);
        });
        for (size_t c = 0, issued = 0; c < p.nchunk; ++c) {
            for (; issued < std::min(p.nchunk, c + p.ahead); ++issued) {
                if (issued >= p.nslot) task.wait(issued - p.nslot);
                check(hipMemcpyAsync(slot(p, issued), static_cast<const char *>(dev) + issued * p.per * row_bytes,
                                     (p.end(issued) - issued * p.per) * row_bytes, hipMemcpyDeviceToHost, st));
                check(hipEventRecord(ev_[issued % p.nslot], st));
            }
            check(hipEventSynchronize(ev_[c % p.nslot]));
            task.allow(c + 1);
        }
        task.finish();
    }

    // rows from host addresses src(row) to the device, queued on st and complete
    // on return
    template <class Src>
    void to_device(hipStream_t st, void *dev, size_t nrow, size_t row_bytes, Src src) {
        if (nrow == 0 || row_bytes == 0) return;
        std::lock_guard<std::mutex> one(use_);
        const Plan p = plan(nrow, row_bytes);
        Task task(*this, p.nchunk, p.nslot, nullptr, [&](size_t c) {
            char *s = slot(p, c);
            for (size_t r = c * p.per; r < p.end(c); ++r, s += row_bytes) std::memcpy(s, src(r), row_bytes);
        });
        for (size_t c = 0; c < p.nchunk; ++c) {
            task.wait(c);
            check(hipMemcpyAsync(static_cast<char *>(dev) + c * p.per * row_bytes, slot(p, c),
                                 (p.end(c) - c * p.per) * row_bytes, hipMemcpyHostToDevice, st));
            check(hipEventRecord(ev_[c % p.nslot], st));
            if (c + 1 >= p.ahead) {
                check(hipEventSynchronize(ev_[(c + 1 - p.ahead) % p.nslot]));
                task.allow(c + 2 - p.ahead + p.nslot);
            }
        }
        check(hipEventSynchronize(ev_[(p.nchunk - 1) % p.nslot]));
        task.finish();
    }

  private:
    // chunk c: rows c*per .. end(c)-1, through slot c % nslot; ahead: transfers
    // queued before the caller waits for the oldest
    struct Plan {
        size_t nrow, per, nchunk, nslot, ahead, slot_bytes;
        size_t end(size_t c) const { return std::min(nrow, (c + 1) * per); }
    };

    // The host's share of one copy: parts of the fill, then chunks in order, each
    // taken by the caller (while it waits) or a helper, whoever comes first.
    struct Job {
        std::mutex mu;
        std::condition_variable cv;
        size_t nfill, nchunk, allowed, left, next_fill = 0, next = 0, running = 0;
        std::vector<char> done;
        std::function<void(size_t, size_t)> fill;
        std::function<void(size_t)> copy;

        // one part or chunk, if any may be taken now
        bool run_one(std::unique_lock<std::mutex> &g) {
            const bool f = next_fill < nfill;
            if (!f && next >= std::min(allowed, nchunk)) return false;
            const size_t k = f ? next_fill++ : next++;
            ++running;
            g.unlock();
            f ? fill(k, nfill) : copy(k);
            g.lock();
            --running;
            --left;
            if (!f) done[k] = 1;
            cv.notify_all();
            return true;
        }
        template <class Ready>
        void wait(Ready ready) {
            std::unique_lock<std::mutex> g(mu);
            while (!ready())
                if (!run_one(g)) cv.wait(g);
        }
        void help() {
            std::unique_lock<std::mutex> g(mu);
            while (next_fill < nfill || next < nchunk)
                if (!run_one(g)) cv.wait(g);
        }
    };

    class Task {
      public:
        template <class Fill, class Copy>
        Task(HostCopy &hc, size_t nchunk, size_t allowed, Fill fill, Copy copy) : j_(std::make_shared<Job>()) {
            // up to two chunks: the caller is done before a helper has started
            const size_t nt = nchunk > 2 ? std::min(THREADS, nchunk - 1) : 0;
            j_->fill = fill;
            j_->nfill = j_->fill ? nt + 1 : 0;
            j_->nchunk = nchunk;
            j_->allowed = allowed;
            j_->left = j_->nfill + nchunk;
            j_->done.assign(nchunk, 0);
            j_->copy = copy;
            hc.start_helpers(nt, j_);
        }
        // after an exception: what nobody has taken is dropped, and what has been
        // taken is waited for (it refers to the caller's variables)
        ~Task() {
            std::unique_lock<std::mutex> g(j_->mu);
            j_->next_fill = j_->nfill;
            j_->next = j_->nchunk;
            j_->cv.notify_all();
            j_->cv.wait(g, [&] { return j_->running == 0; });
        }
        // chunks below n may be copied
        void allow(size_t n) {
            {
                std::lock_guard<std::mutex> g(j_->mu);
                j_->allowed = n;
            }
            j_->cv.notify_all();
        }
        // until chunk c has been copied
        void wait(size_t c) {
            j_->wait([&] { return j_->done[c] != 0; });
        }
        void finish() {
            j_->wait([&] { return j_->left == 0; });
        }

      private:
        std::shared_ptr<Job> j_;
    };

    // helpers still on their way from earlier copies count: at most THREADS
    struct Helper {
        std::thread thread;
        std::shared_ptr<std::atomic<bool>> ended;
    };
    std::vector<Helper> helpers_;

    void start_helpers(size_t n, const std::shared_ptr<Job> &job) {
        for (size_t k = 0; k < helpers_.size();)
            if (helpers_[k].ended->load()) {
                helpers_[k].thread.join();
                std::swap(helpers_[k], helpers_.back());
                helpers_.pop_back();
            } else {
                ++k;
            }
        helpers_.reserve(THREADS);
        try {
            while (helpers_.size() < n) {
                auto ended = std::make_shared<std::atomic<bool>>(false);
                helpers_.push_back({std::thread([job, ended] {
                                        job->help();
                                        ended->store(true);
                                    }),
                                    ended});
            }
        } catch (const std::exception &) {
            // no more threads to be had: the caller copies what is left
        }
    }

    std::mutex use_;   // one copy at a time: callers on several threads share the slots
    char *slab_ = nullptr;
    size_t bytes_ = 0;
    std::vector<hipEvent_t> ev_;

    static void check(hipError_t e) {
        if (e != hipSuccess) throw std::runtime_error(std::string("host copy: ") + hipGetErrorString(e));
    }

    char *slot(const Plan &p, size_t c) const { return slab_ + (c % p.nslot) * p.slot_bytes; }

    Plan plan(size_t nrow, size_t row_bytes) {
        Plan p;
        p.nrow = nrow;
        p.per = std::max<size_t>(1, CHUNK / row_bytes);
        p.nchunk = (nrow + p.per - 1) / p.per;
        p.nslot = std::min(SLOTS, p.nchunk);
        p.ahead = (p.nslot + 1) / 2;
        p.slot_bytes = std::min(p.per, nrow) * row_bytes;
        if (bytes_ < p.nslot * p.slot_bytes) {
            if (slab_) check(hipHostFree(slab_));
            slab_ = nullptr;
            bytes_ = 0;
            void *q = nullptr;
            check(hipHostMalloc(&q, p.nslot * p.slot_bytes, hipHostMallocDefault));
            slab_ = static_cast<char *>(q);
            bytes_ = p.nslot * p.slot_bytes;
        }
        while (ev_.size() < p.nslot) {
            hipEvent_t e;
            check(hipEventCreateWithFlags(&e, hipEventDisableTiming));
            ev_.push_back(e);
        }
        return p;
    }
};

}  // namespace coral
