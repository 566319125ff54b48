// Staged uploads of host slices (see aq_host_stage.h).
//
// What a call cannot do without is the bytes over PCIe (9.4 MB: 175 us at the 54 GB/s that one copy from pinned memory
// reaches here; the runtime's own copy from pageable memory takes 262 us and each small one 37 us, and the five allocations
// and frees of a call 180 us).  So the arrays of a call go, one behind the other, through a ring of pinned memory:
// worker threads and the caller copy pieces into it, and as soon as a run of pieces is whole a small kernel that
// reads host memory moves it to the device (back to back such kernels keep the link as busy as one long copy; as many
// separate copy commands lose 8 us each), while the next pieces are being filled.  The ring and a device block stay with the
// context between calls, up to the sizes below.
#include "aq_host_stage.h"

#include <atomic>
#include <condition_variable>
#include <cstring>
#include <functional>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace aq {

namespace {

constexpr size_t kPiece = (size_t)128 << 10;     // bytes a thread copies at a time
constexpr int kFirstRun = 3, kLongRun = 32;      // pieces of the first copy kernel, and of a long one
constexpr size_t kRing = (size_t)64 << 20;       // pinned memory at most
constexpr size_t kKeepDevice = (size_t)256 << 20;  // device memory kept between calls at most
constexpr size_t kAlone = (size_t)384 << 10;     // the caller copies this much by itself: waking threads costs about as much
constexpr int kWorkers = 5;

__global__ __launch_bounds__(256) void pull_kernel(const uint4* __restrict__ src, uint4* __restrict__ dst, uint32_t n) {
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < n; i += gridDim.x * 256u) dst[i] = src[i];
}

void narrow(uint16_t* dst, const float* src, size_t n) {
    for (size_t i = 0; i < n; i++) {
        uint32_t u;
        memcpy(&u, src + i, 4);
        const uint32_t rounded = (u + 0x7fffu + ((u >> 16) & 1u)) >> 16, quiet = (u >> 16) | 0x40u;
        dst[i] = (uint16_t)((u & 0x7fffffffu) > 0x7f800000u ? quiet : rounded);
    }
}

void widen_some(float* dst, const uint16_t* src, size_t n) {
    for (size_t i = 0; i < n; i++) {
        const uint32_t u = (uint32_t)src[i] << 16;
        memcpy(dst + i, &u, 4);
    }
}

}  // namespace

// Threads that take the units 0 .. n - 1 of a job in order, together with the caller.
struct HostStage::Pool {
    std::mutex mu;
    std::condition_variable wake;
    std::vector<std::thread> threads;
    uint64_t job = 0;  // under mu
    bool stop = false;
    std::function<void(int)> work;
    std::atomic<int> next{0}, limit{0}, busy{0}, units{0};  // units below `limit` may be taken

    Pool() {
        threads.reserve(kWorkers);
        try {
            for (int i = 0; i < kWorkers; i++) threads.emplace_back([this] { run(); });
        } catch (const std::system_error&) {
            // the process may start no more threads: those there are, or the caller alone, do the work
        }
    }
    ~Pool() {
        {
            std::lock_guard<std::mutex> lk(mu);
            stop = true;
        }
        wake.notify_all();
        for (auto& t : threads) t.join();
    }
    // Takes and does one unit; false when there is none to take.
    bool one() {
        int u = next.load(std::memory_order_relaxed);
        do {
            if (u >= limit.load(std::memory_order_acquire)) return false;
        } while (!next.compare_exchange_weak(u, u + 1, std::memory_order_acq_rel));
        work(u);
        return true;
    }
    void run() {
        uint64_t seen = 0;
        for (;;) {
            {
                std::unique_lock<std::mutex> lk(mu);
                wake.wait(lk, [&] { return stop || job != seen; });
                if (stop) return;
                seen = job;
                busy.fetch_add(1, std::memory_order_acq_rel);  // under mu: end() sees it or the job is over
            }
            while (next.load(std::memory_order_relaxed) < units.load(std::memory_order_acquire))
                if (!one()) std::this_thread::yield();
            busy.fetch_sub(1, std::memory_order_acq_rel);
        }
    }
    void begin(int n, int allowed, std::function<void(int)> fn) {
        {
            std::lock_guard<std::mutex> lk(mu);
            work = std::move(fn);
            next.store(0, std::memory_order_release);
            units.store(n, std::memory_order_release);
            limit.store(allowed < n ? allowed : n, std::memory_order_release);
            job++;
        }
        wake.notify_all();
    }
    // All units have been taken; waits until none is being worked on and no thread can come to this job any more.
    void end() {
        for (;;) {
            {
                std::lock_guard<std::mutex> lk(mu);
                if (busy.load(std::memory_order_acquire) == 0) {
                    // a thread that wakes up late finds nothing to take until begin() has written the next job
                    limit.store(0, std::memory_order_release);
                    units.store(0, std::memory_order_release);
                    return;
                }
            }
            std::this_thread::yield();
        }
    }
};

HostStage::~HostStage() {
    delete pool_;
    if (event_) (void)hipEventDestroy(event_);
    if (pinned_) (void)hipHostFree(pinned_);
    if (out_) (void)hipHostFree(out_);
    if (dev_) (void)hipFree(dev_);
}

hipError_t HostStage::grow(char** p, size_t* have, size_t want, bool host) {
    if (*have >= want) return hipSuccess;
    if (*p) (void)(host ? hipHostFree(*p) : hipFree(*p));
    *p = nullptr;
    *have = 0;
    const hipError_t rc = host ? hipHostMalloc(reinterpret_cast<void**>(p), want, hipHostMallocDefault) : hipMalloc(reinterpret_cast<void**>(p), want);
    if (rc == hipSuccess) *have = want;
    return rc;
}

hipError_t HostStage::upload(const HostPart* parts, int count, size_t total, hipStream_t stream, char** dev) {
    const size_t ring = total < kRing ? (total + kPiece - 1) / kPiece * kPiece : kRing;
    hipError_t rc = grow(&pinned_, &pinned_bytes_, ring, true);
    if (rc == hipSuccess) rc = grow(&dev_, &dev_bytes_, total, false);
    if (rc != hipSuccess) return rc;
    *dev = dev_;
    const int units = (int)((total + kPiece - 1) / kPiece);   // pieces of the device block
    const int places = (int)(pinned_bytes_ / kPiece);         // pieces the ring holds
    auto fill = [&](int unit) {  // bytes [unit * kPiece, + kPiece) of the device block
        const size_t lo = (size_t)unit * kPiece, hi = lo + kPiece;
        char* const slot = pinned_ + (size_t)(unit % places) * kPiece;
        for (int i = 0; i < count; i++) {
            const size_t a = parts[i].at > lo ? parts[i].at : lo, end = parts[i].at + parts[i].bytes, b = end < hi ? end : hi;
            if (a >= b) continue;
            if (parts[i].from_f32)
                narrow(reinterpret_cast<uint16_t*>(slot + (a - lo)), static_cast<const float*>(parts[i].src) + (a - parts[i].at) / 2, (b - a) / 2);
            else
                memcpy(slot + (a - lo), static_cast<const char*>(parts[i].src) + (a - parts[i].at), b - a);
        }
    };
    auto send = [&](int from, int to) {  // pieces [from, to), consecutive in the ring
        const size_t at = (size_t)from * kPiece, end = (size_t)to * kPiece, n = (end < total ? end : total) - at;
        const uint32_t vectors = (uint32_t)(n / 16);
        const unsigned blocks = vectors < 64 * 256 ? (vectors + 255) / 256 : 64;
        hipLaunchKernelGGL(pull_kernel, dim3(blocks), dim3(256), 0, stream, reinterpret_cast<const uint4*>(pinned_ + (size_t)(from % places) * kPiece),
                           reinterpret_cast<uint4*>(dev_ + at), vectors);
        return hipGetLastError();
    };
    if (total <= kAlone) {
        for (int u = 0; u < units; u++) fill(u);
        return send(0, units);
    }
    if (!pool_) pool_ = new Pool();
    std::vector<std::atomic<char>> ready((size_t)units);
    for (auto& r : ready) r.store(0, std::memory_order_relaxed);
    const bool wraps = units > places;
    if (wraps && !event_) {
        rc = hipEventCreateWithFlags(&event_, hipEventDisableTiming);
        if (rc != hipSuccess) return rc;
    }
    pool_->begin(units, places, [&](int u) {
        fill(u);
        ready[(size_t)u].store(1, std::memory_order_release);
    });
    // What is whole goes out in runs that grow with what has gone before: the link starts early and is then kept busy by a
    // few long kernels (host memory fills the ring faster than the link empties it).
    for (int sent = 0, whole = 0, open = places; sent < units;) {
        while (whole < units && whole < open && ready[(size_t)whole].load(std::memory_order_acquire)) whole++;
        int run = whole - sent;
        const int to_end = places - sent % places;  // a run does not wrap
        if (run >= to_end) run = to_end;
        const int want = sent / 2 < kFirstRun ? kFirstRun : sent / 2 > kLongRun ? kLongRun : sent / 2;
        if (run > 0 && (run >= want || run == to_end || whole == units)) {
            if (rc == hipSuccess) rc = send(sent, sent + run);
            sent += run;
            if (wraps && sent % places == 0 && sent < units) {
                // the ring is full and on its way: it may be filled again once its kernels are done
                if (rc == hipSuccess) rc = hipEventRecord(event_, stream);
                if (rc == hipSuccess) rc = hipEventSynchronize(event_);
                open += places;
                pool_->limit.store(open < units ? open : units, std::memory_order_release);
            }
        } else if (!pool_->one()) {
            std::this_thread::yield();
        }
    }
    pool_->end();
    return rc;
}

hipError_t HostStage::results(size_t bytes, void** host) {
    char* p = static_cast<char*>(out_);
    const hipError_t rc = grow(&p, &out_bytes_, bytes, true);
    out_ = p;
    *host = p;
    return rc;
}

void HostStage::widen(float* out, const uint16_t* in, size_t n) {
    constexpr size_t some = (size_t)32 << 10;
    if (n <= 4 * some) return widen_some(out, in, n);
    if (!pool_) pool_ = new Pool();
    const int units = (int)((n + some - 1) / some);
    pool_->begin(units, units, [&](int u) {
        const size_t lo = (size_t)u * some, m = n - lo < some ? n - lo : some;
        widen_some(out + lo, in + lo, m);
    });
    while (pool_->one()) {
    }
    pool_->end();
}

void HostStage::finish() {
    if (dev_bytes_ > kKeepDevice) {
        (void)hipFree(dev_);
        dev_ = nullptr;
        dev_bytes_ = 0;
    }
}

}  // namespace aq
