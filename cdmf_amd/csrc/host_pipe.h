// Large copies between the caller's (pageable) memory and the device.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstring>
#include <thread>
#include <vector>

namespace ccd {

// The runtime copies pageable memory through its own staging on one thread:
// 29 GB/s to the device, 17 GB/s back, 10 GB/s into memory the caller has
// just allocated (its page faults), where the link does 57.  This pipe has
// four threads copy pieces of up to 4 MB to or from pinned memory, two pieces
// each in flight: 43 GB/s either way (each piece costs the stream about 15 us
// besides its bytes: 31 GB/s with pieces of 1 MB).  Below the bounds starting
// the threads costs what they save, and the runtime's path is taken.  One
// pipe belongs to one object and is used by one thread at a time, as the
// object is.  From its first large copy until release() it holds eight events
// and eight pinned pieces as large as its largest copy asked for: 4 MB after
// a copy of 2 MB, 32 MB after one of more than 16.
class HostPipe {
public:
    static constexpr size_t BIG_IN = 12u << 20, BIG_OUT = 2u << 20;

    HostPipe() = default;
    HostPipe(const HostPipe&) = delete;
    HostPipe& operator=(const HostPipe&) = delete;
    ~HostPipe() { release(); }

    // After the object's stream is idle.
    void release() {
        for (hipEvent_t& e : ev_) {
            if (e) (void)hipEventDestroy(e);
            e = nullptr;
        }
        if (buf_) (void)hipHostFree(buf_);
        buf_ = nullptr;
        slot_ = 0;
    }

    // dst (device) = src (host), ordered on stream s; src may change once it
    // returns for large copies, and once s has been waited for otherwise.
    hipError_t in(int device, void* dst, const void* src, size_t bytes, hipStream_t s) {
        if (bytes == 0) return hipSuccess;
        const size_t piece = piece_of(bytes);
        if (bytes < BIG_IN || !ready(piece)) return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s);
        return run(device, bytes, [&](int w, std::atomic<size_t>& next) -> hipError_t {
            int n = 0;
            for (size_t c; (c = next.fetch_add(piece)) < bytes; ++n) {
                const int q = w * SLOTS + n % SLOTS;
                const size_t len = bytes - c < piece ? bytes - c : piece;
                char* p = buf_ + (size_t)q * slot_;
                hipError_t e = hipEventSynchronize(ev_[q]);  // the piece last sent from here (none: returns at once)
                if (e != hipSuccess) return e;
                std::memcpy(p, static_cast<const char*>(src) + c, len);
                e = hipMemcpyAsync(static_cast<char*>(dst) + c, p, len, hipMemcpyHostToDevice, s);
                if (e == hipSuccess) e = hipEventRecord(ev_[q], s);
                if (e != hipSuccess) return e;
            }
            return hipSuccess;
        });
    }

    // dst (host) = src (device) after the work on stream s; complete on return.
    hipError_t out(int device, void* dst, const void* src, size_t bytes, hipStream_t s) {
        if (bytes == 0) return hipStreamSynchronize(s);
        const size_t piece = piece_of(bytes);
        if (bytes < BIG_OUT || !ready(piece)) {
            const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s);
            const hipError_t w = hipStreamSynchronize(s);
            return e != hipSuccess ? e : w;
        }
        return run(device, bytes, [&](int w, std::atomic<size_t>& next) -> hipError_t {
            size_t at[SLOTS], len[SLOTS];
            auto fetch = [&](int q, bool& got) -> hipError_t {
                at[q] = next.fetch_add(piece);
                got = at[q] < bytes;
                if (!got) return hipSuccess;
                len[q] = bytes - at[q] < piece ? bytes - at[q] : piece;
                const int x = w * SLOTS + q;
                hipError_t e = hipEventSynchronize(ev_[x]);
                if (e == hipSuccess)
                    e = hipMemcpyAsync(buf_ + (size_t)x * slot_, static_cast<const char*>(src) + at[q], len[q],
                                       hipMemcpyDeviceToHost, s);
                if (e == hipSuccess) e = hipEventRecord(ev_[x], s);
                return e;
            };
            bool got[SLOTS];
            for (int q = 0; q < SLOTS; ++q) {
                const hipError_t e = fetch(q, got[q]);
                if (e != hipSuccess) return e;
            }
            for (int q = 0; got[q]; q = (q + 1) % SLOTS) {
                const int x = w * SLOTS + q;
                hipError_t e = hipEventSynchronize(ev_[x]);
                if (e != hipSuccess) return e;
                std::memcpy(static_cast<char*>(dst) + at[q], buf_ + (size_t)x * slot_, len[q]);
                e = fetch(q, got[q]);
                if (e != hipSuccess) return e;
            }
            return hipSuccess;
        });
    }

private:
    static constexpr int WORKERS = 4, SLOTS = 2;
    static constexpr size_t PIECE = 4u << 20;  // largest
    char* buf_ = nullptr;
    size_t slot_ = 0;  // bytes of a pinned piece
    hipEvent_t ev_[WORKERS * SLOTS] = {};

    // every worker two pieces, within 512 KB and 4 MB
    static size_t piece_of(size_t bytes) {
        const size_t p = (bytes / (WORKERS * SLOTS) + 4095) & ~(size_t)4095;
        return p < (512u << 10) ? 512u << 10 : p < PIECE ? p : PIECE;
    }

    // Pinned pieces of at least `piece` bytes.  false: the runtime's copies
    // are taken instead, and the error that hipGetLastError would report after
    // the next launch is cleared.
    bool ready(size_t piece) {
        if (slot_ >= piece) return true;
        for (hipEvent_t& e : ev_) {
            if (e) {
                if (hipEventSynchronize(e) != hipSuccess) return give_up();  // the smaller pieces are done with
            } else if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
                e = nullptr;
                return give_up();
            }
        }
        if (buf_) (void)hipHostFree(buf_);
        slot_ = 512u << 10;
        while (slot_ < piece) slot_ *= 2;
        if (hipHostMalloc(reinterpret_cast<void**>(&buf_), WORKERS * SLOTS * slot_, hipHostMallocDefault) != hipSuccess) {
            buf_ = nullptr;
            return give_up();
        }
        return true;
    }

    bool give_up() {
        release();
        (void)hipGetLastError();
        return false;
    }

    // The calling thread is worker 0; pieces are taken from a shared counter,
    // so the copy completes with any number of workers.
    template <class F>
    hipError_t run(int device, size_t bytes, const F& work) {
        std::atomic<size_t> next{0};
        std::atomic<int> bad{(int)hipSuccess};
        auto body = [&](int w) {
            hipError_t e = w ? hipSetDevice(device) : hipSuccess;
            if (e == hipSuccess) e = work(w, next);
            int none = (int)hipSuccess;
            if (e != hipSuccess) bad.compare_exchange_strong(none, (int)e);
        };
        std::vector<std::thread> pool;
        try {
            for (int w = 1; w < WORKERS; ++w) pool.emplace_back(body, w);
        } catch (...) {  // no more threads: those there are do it
        }
        body(0);
        for (std::thread& t : pool) t.join();
        return (hipError_t)bad.load();
    }
};

}  // namespace ccd
