// Host check of HostPipe (host_pipe.h) on a restatement of the runtime calls
// it makes: a stream is a queue that nothing moves but a wait for it or for
// an event in it, so a copy reads its source and writes its destination as
// late as the runtime may.  Exits 0 and prints "ok" when every check holds.
#include "host_pipe.h"

#include <cstdio>
#include <cstdlib>
#include <deque>
#include <mutex>

namespace {

std::mutex mtx;
struct Event {
    bool pending = false;
};
struct Op {
    void* dst;
    const void* src;
    size_t bytes;
    Event* ev;
};
std::deque<Op> queue;
thread_local hipError_t last = hipSuccess;
int events = 0, pinned = 0;       // alive
size_t pinned_bytes = 0;          // of the last pinned allocation
int fail_event = -1;              // the n-th event to create from now on fails
bool fail_pinned = false;
int fail_copy = -1;               // the n-th copy from now on fails

hipError_t fail(hipError_t e) { return last = e; }

void run_until(const Event* ev) {  // null: all
    while (!queue.empty() && (!ev || ev->pending)) {
        const Op op = queue.front();
        queue.pop_front();
        if (op.bytes) std::memcpy(op.dst, op.src, op.bytes);
        if (op.ev) op.ev->pending = false;
    }
}

}  // namespace

extern "C" {
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    std::lock_guard<std::mutex> l(mtx);
    if (fail_event == 0) return fail_event = -1, fail(hipErrorOutOfMemory);
    if (fail_event > 0) --fail_event;
    ++events;
    *e = reinterpret_cast<hipEvent_t>(new Event);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    std::lock_guard<std::mutex> l(mtx);
    --events;
    delete reinterpret_cast<Event*>(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
    std::lock_guard<std::mutex> l(mtx);
    Event* ev = reinterpret_cast<Event*>(e);
    ev->pending = true;
    queue.push_back({nullptr, nullptr, 0, ev});
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    std::lock_guard<std::mutex> l(mtx);
    run_until(reinterpret_cast<Event*>(e));
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
    std::lock_guard<std::mutex> l(mtx);
    run_until(nullptr);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind, hipStream_t) {
    std::lock_guard<std::mutex> l(mtx);
    if (fail_copy == 0) return fail_copy = -1, fail(hipErrorInvalidValue);
    if (fail_copy > 0) --fail_copy;
    queue.push_back({dst, src, bytes, nullptr});
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
    if (fail_pinned) return *p = nullptr, fail(hipErrorOutOfMemory);
    ++pinned;
    pinned_bytes = bytes;
    *p = std::malloc(bytes);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    --pinned;
    std::free(p);
    return hipSuccess;
}
}

namespace {

using ccd::HostPipe;
constexpr size_t MB = 1u << 20;

void check(bool ok, const char* what, size_t bytes) {
    if (ok) return;
    std::printf("failed: %s, %zu bytes\n", what, bytes);
    std::exit(1);
}

// n bytes out of a fixed pattern, another part of it for another seed
std::vector<unsigned char> bytes_of(size_t n, unsigned seed) {
    static const std::vector<unsigned char> pattern = [] {
        std::vector<unsigned char> v(48 * MB);
        unsigned x = 1;
        for (unsigned char& c : v) c = (unsigned char)((x = x * 1664525u + 1013904223u) >> 24);
        return v;
    }();
    const unsigned char* from = pattern.data() + 977 * (size_t)seed;
    return std::vector<unsigned char>(from, from + n);
}

// One array in and back through the pipe.
void round_trip(HostPipe& p, size_t n, unsigned seed) {
    const std::vector<unsigned char> want = bytes_of(n, seed);
    std::vector<unsigned char> src = want, dev(n + 64, 0xa5), back(n + 64, 0x5a);
    check(p.in(0, dev.data(), src.data(), n, nullptr) == hipSuccess, "in", n);
    if (n >= HostPipe::BIG_IN && pinned) std::memset(src.data(), 0xff, n);  // the caller's array is free again
    check(hipStreamSynchronize(nullptr) == hipSuccess, "wait", n);
    check(n == 0 || std::memcmp(dev.data(), want.data(), n) == 0, "what arrived", n);
    check(p.out(0, back.data(), dev.data(), n, nullptr) == hipSuccess, "out", n);
    std::memset(dev.data(), 0, n);  // complete on return
    check(n == 0 || std::memcmp(back.data(), want.data(), n) == 0, "what came back", n);
    for (size_t i = n; i < n + 64; ++i) check(dev[i] == 0xa5 && back[i] == 0x5a, "bytes past the end", n);
    check(hipGetLastError() == hipSuccess, "an error left behind", n);
}

}  // namespace

int main() {
    const size_t sizes[] = {0, 1, 4096, HostPipe::BIG_OUT - 1, HostPipe::BIG_OUT, HostPipe::BIG_OUT + 1, 4 * MB + 3,
                            HostPipe::BIG_IN - 1, HostPipe::BIG_IN, HostPipe::BIG_IN + 1, 32 * MB, 32 * MB + 1,
                            41 * MB + 12345};
    unsigned seed = 0;
    {
        HostPipe p;
        for (size_t n : sizes) round_trip(p, n, ++seed);
        round_trip(p, 13 * MB + 1, ++seed);  // pieces and events used before
        check(events == 8 && pinned == 1, "what a pipe holds", 0);
        p.release();
        check(events == 0 && pinned == 0, "what a released pipe holds", 0);
        for (size_t n : {HostPipe::BIG_OUT, 13 * MB}) round_trip(p, n, ++seed);
    }
    check(events == 0 && pinned == 0, "what is left of a pipe", 0);
    {  // as much as the largest copy asks for, grown while copies are still queued
        HostPipe p;
        round_trip(p, HostPipe::BIG_OUT, ++seed);
        check(pinned == 1 && pinned_bytes == 4 * MB, "after a copy of", HostPipe::BIG_OUT);
        const std::vector<unsigned char> a = bytes_of(13 * MB, ++seed), b = bytes_of(20 * MB, ++seed);
        std::vector<unsigned char> src = a, src2 = b, da(a.size()), db(b.size());
        check(p.in(0, da.data(), src.data(), a.size(), nullptr) == hipSuccess, "in", a.size());
        std::memset(src.data(), 0, src.size());
        check(pinned == 1 && pinned_bytes == 16 * MB, "after a copy of", a.size());
        check(p.in(0, db.data(), src2.data(), b.size(), nullptr) == hipSuccess, "in", b.size());
        std::memset(src2.data(), 0, src2.size());
        check(pinned == 1 && pinned_bytes == 32 * MB, "after a copy of", b.size());
        (void)hipStreamSynchronize(nullptr);
        check(da == a && db == b, "copies about a growth", 0);
        round_trip(p, HostPipe::BIG_OUT + 1, ++seed);
        check(pinned == 1 && pinned_bytes == 32 * MB, "what stays", 0);
        fail_pinned = true;
        p.release();
        round_trip(p, HostPipe::BIG_OUT, ++seed);
        fail_pinned = false;
    }
    check(events == 0 && pinned == 0, "what is left of a grown pipe", 0);
    {  // no pinned memory, no events: the runtime's own copies, and no error for the next call to find
        HostPipe p;
        fail_pinned = true;
        for (size_t n : {HostPipe::BIG_OUT, 13 * MB}) round_trip(p, n, ++seed);
        fail_pinned = false;
        for (int e : {0, 3, 7}) {
            for (bool out : {false, true}) {
                fail_event = e;
                if (out) fail_event = -1;
                round_trip(p, out ? HostPipe::BIG_OUT : 13 * MB, ++seed);
                p.release();
            }
        }
        check(events == 0 && pinned == 0, "what failed calls left", 0);
    }
    {  // a copy that fails is reported, and the pipe works after it
        HostPipe p;
        std::vector<unsigned char> a(33 * MB), b(33 * MB);
        for (int nth : {0, 1, 5, 8}) {
            fail_copy = nth;
            check(p.in(0, b.data(), a.data(), a.size(), nullptr) == hipErrorInvalidValue, "a failed copy in", nth);
            (void)hipStreamSynchronize(nullptr);
            fail_copy = nth;
            check(p.out(0, b.data(), a.data(), a.size(), nullptr) == hipErrorInvalidValue, "a failed copy out", nth);
            (void)hipStreamSynchronize(nullptr);
            (void)hipGetLastError();
            round_trip(p, 12 * MB + nth, ++seed);
        }
    }
    std::puts("ok");
    return 0;
}
