// Copies from device memory to pageable host memory by several threads.
//
// The runtime's own copy of such memory goes through its staging buffer one
// megabyte at a time, the host's half (a memcpy into pages that are mostly
// touched for the first time) after the device's: 20 and 65 us per megabyte on
// MI355X, 16 GB/s.  Here a few threads each keep two pieces in flight through
// pinned memory of their own, so the device's half is hidden and the host's
// divided: the 52 MB list of 100k atoms 3.1 -> 1.4 ms, 155 MB of 300k 15.8 -> 4.7
// ms.  Pieces of 1 to 4 MB: each costs the stream about 14 us beside its transfer
// (pieces of a sixteenth of the list, 10k atoms: 458 us against 290).
#pragma once
#include <hip/hip_runtime.h>
#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <cstring>
#include <functional>
#include <memory>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace nlh {

// Used by one thread at a time (see HostCopierPool); its threads come with its
// first copy and its pinned memory grows to what a copy needs.
class HostCopier {
public:
    // Bytes from which a copy goes this way (lists in pageable memory, this way /
    // the runtime's: 3,000 atoms, 2.2 MB, 185 / 188 us; 6,000 237 / 260; 10k 300 /
    // 368; 20k 458 / 668).  Positions on their way to the device, a twentieth of
    // a list's bytes, were no faster so.
    static constexpr size_t kWorthIt = 3 << 20;

    struct Piece {
        char *host;
        char *device;
        size_t bytes;
    };

    explicit HostCopier(int device) : device(device) {}
    HostCopier(const HostCopier &) = delete;
    HostCopier &operator=(const HostCopier &) = delete;

    // Ends the threads and frees the pinned memory and the events (no capture in
    // the process).  In a forked child the threads do not exist: let go.
    ~HostCopier()
    {
        {
            std::lock_guard<std::mutex> lk(m_);
            stop_ = true;
        }
        wake_.notify_all();
        for (std::thread &t : threads_) {
            if (getpid() == pid_) t.join();
            else t.detach();
        }
        trim(0);
        for (hipEvent_t &e : ev_)
            if (e) (void)hipEventDestroy(e);
    }

    // Frees the pinned memory if there is more of it than `bytes`; returns what is left.
    size_t trim(size_t bytes)
    {
        if (ring_bytes_ > bytes) {
            (void)hipHostFree(ring_);
            ring_ = nullptr;
            ring_bytes_ = 0;
        }
        return ring_bytes_;
    }

    const int device;

    // Whether `p` is host memory that the runtime does not know.
    static bool pageable(const void *p)
    {
        hipPointerAttribute_t at{};
        if (hipPointerGetAttributes(&at, p) != hipSuccess) {
            (void)hipGetLastError();
            return true;
        }
        return at.type == hipMemoryTypeUnregistered;
    }

    // What to_host needs for `total` bytes (no capture in the process).
    hipError_t prepare(size_t total)
    {
        hipError_t r = hipSuccess;
        for (hipEvent_t &e : ev_)
            if (!e && r == hipSuccess) r = hipEventCreateWithFlags(&e, hipEventDisableTiming);
        const size_t need = kSlots * step(total);
        if (r != hipSuccess || ring_bytes_ >= need) return r;
        trim(0);
        r = hipHostMalloc(reinterpret_cast<void **>(&ring_), need, hipHostMallocDefault);
        if (r == hipSuccess) ring_bytes_ = need;
        else ring_ = nullptr;
        return r;
    }

    // device -> pageable host, after the work on `st`; complete on return.
    hipError_t to_host(hipStream_t st, const std::vector<Piece> &arrays, int threads = kThreads)
    {
        size_t size;   // of a slot
        const std::vector<Piece> list = cut(arrays, size);
        std::atomic<size_t> next{0};
        std::atomic<int> error{hipSuccess};
        run([&](int w) {
            hipError_t r = hipSetDevice(device);
            size_t c[2];
            for (int k = 0; k < 2 && r == hipSuccess; ++k) r = fetch(st, list, size, c[k] = next++, 2 * w + k);
            for (int k = 0; r == hipSuccess && c[k] < list.size(); k ^= 1) {
                const int slot = 2 * w + k;
                r = hipEventSynchronize(ev_[slot]);
                if (r != hipSuccess) break;
                std::memcpy(list[c[k]].host, ring_ + slot * size, list[c[k]].bytes);
                r = fetch(st, list, size, c[k] = next++, slot);
            }
            if (r != hipSuccess) error = r;
        }, threads);
        // pieces in flight after an error must not outlive their slots
        if (error != hipSuccess) (void)hipStreamSynchronize(st);
        return (hipError_t)error.load();
    }

    static constexpr int kThreads = 4;             // the caller's among them

private:
    static constexpr int kSlots = 2 * kThreads;
    static constexpr size_t kPiece = 4 << 20;      // largest piece

    // Queue piece c into a slot (nothing past the last piece).
    hipError_t fetch(hipStream_t st, const std::vector<Piece> &list, size_t size, size_t c, int slot)
    {
        if (c >= list.size()) return hipSuccess;
        const hipError_t r =
            hipMemcpyAsync(ring_ + slot * size, list[c].device, list[c].bytes, hipMemcpyDeviceToHost, st);
        return r != hipSuccess ? r : hipEventRecord(ev_[slot], st);
    }

    // The size of a piece: about one piece per slot, 1 MB to kPiece.
    static size_t step(size_t total)
    {
        return std::clamp<size_t>(total / kSlots / 4096 * 4096, 1 << 20, kPiece);
    }

    static std::vector<Piece> cut(const std::vector<Piece> &arrays, size_t &size)
    {
        size_t total = 0;
        for (const Piece &a : arrays) total += a.bytes;
        size = step(total);
        std::vector<Piece> list;
        for (const Piece &a : arrays)
            for (size_t o = 0; o < a.bytes; o += size)
                list.push_back({a.host + o, a.device + o, std::min(size, a.bytes - o)});
        return list;
    }

    // job(0) here and job(w) on every thread w < threads that wakes up in time.
    void run(const std::function<void(int)> &job, int threads)
    {
        if (threads_.empty()) {
            pid_ = getpid();
            try {
                for (int w = 1; w < kThreads; ++w) threads_.emplace_back([this, w] { work(w); });
            } catch (const std::system_error &) {   // fewer threads, then
            }
        }
        {
            std::lock_guard<std::mutex> lk(m_);
            job_ = &job;
            limit_ = threads;
            ++turn_;
        }
        wake_.notify_all();
        job(0);
        std::unique_lock<std::mutex> lk(m_);
        job_ = nullptr;
        done_.wait(lk, [this] { return active_ == 0; });
    }

    void work(int w)
    {
        uint64_t seen = 0;
        std::unique_lock<std::mutex> lk(m_);
        for (;;) {
            wake_.wait(lk, [&] { return stop_ || (job_ && turn_ != seen && w < limit_); });
            if (stop_) return;
            seen = turn_;
            const std::function<void(int)> *job = job_;
            ++active_;
            lk.unlock();
            (*job)(w);
            lk.lock();
            if (--active_ == 0) done_.notify_all();
        }
    }

    char *ring_ = nullptr;
    size_t ring_bytes_ = 0;
    hipEvent_t ev_[kSlots] = {};
    std::vector<std::thread> threads_;
    std::mutex m_;
    std::condition_variable wake_, done_;
    const std::function<void(int)> *job_ = nullptr;
    uint64_t turn_ = 0;
    int active_ = 0, limit_ = kThreads;
    bool stop_ = false;
    pid_t pid_ = 0;
};

// The process's copiers.  A copy borrows one (its own, whatever other threads
// do), and those given back are kept for the next copies: as many as were in use
// at once, up to kKept, with the pinned memory they came to need (at most 32 MB
// each), and once no handle is left, with at most 8 MB together.  (Starting one
// costs 60 us, its pinned memory up to 300: more than a list of 10k atoms saves.)
class HostCopierPool {
public:
    static constexpr size_t kKept = 4;

    std::unique_ptr<HostCopier> borrow(int device)
    {
        {
            std::lock_guard<std::mutex> lk(m_);
            ++busy_;
            for (size_t k = idle_.size(); k-- > 0;)   // the last one used first
                if (idle_[k]->device == device) {
                    std::unique_ptr<HostCopier> c = std::move(idle_[k]);
                    idle_.erase(idle_.begin() + (std::ptrdiff_t)k);
                    return c;
                }
        }
        return std::make_unique<HostCopier>(device);
    }

    // Returns a copier that is not kept, if there is one, for the caller to end.
    std::unique_ptr<HostCopier> give_back(std::unique_ptr<HostCopier> c)
    {
        std::lock_guard<std::mutex> lk(m_);
        --busy_;
        std::unique_ptr<HostCopier> out;
        if (idle_.size() == kKept) {
            out = std::move(idle_.front());
            idle_.erase(idle_.begin());
        }
        idle_.push_back(std::move(c));   // room for kKept: reserved
        return out;
    }

    // Threads for a copy beside those in progress: more than two copies at once
    // share the link and the host's memory already (lists of 20k atoms from four
    // threads, four / two threads each: 990 / 870 us; 50k 1,990 / 1,910).
    int threads()
    {
        std::lock_guard<std::mutex> lk(m_);
        return busy_ <= 2 ? HostCopier::kThreads : HostCopier::kThreads / 2;
    }

    void handle_made()
    {
        std::lock_guard<std::mutex> lk(m_);
        ++handles_;
    }
    void handle_gone()
    {
        std::lock_guard<std::mutex> lk(m_);
        if (--handles_ > 0) return;
        size_t left = 8 << 20;
        for (auto &c : idle_) left -= c->trim(left);
    }

    HostCopierPool() { idle_.reserve(kKept); }

private:
    std::mutex m_;
    std::vector<std::unique_ptr<HostCopier>> idle_;   // by time of their last use
    int64_t handles_ = 0;
    int busy_ = 0;
};

// Never destroyed: the runtime may be gone before static objects are.
inline HostCopierPool &host_copiers()
{
    static HostCopierPool *pool = new HostCopierPool;
    return *pool;
}

}  // namespace nlh
