// The library's entry points against a HIP runtime of this program's own, which launches nothing and writes down what it is
// asked: which call of which thread launched which kernel, and what memory was asked for.  So order and scratch can be checked
// without a GPU.  The definitions here take the place of the runtime's when the program loads libaq_mi355.so.
#include "aq_kernels.h"
#include "aq_mi355.h"
#include "aq_qmm.h"

#include <dlfcn.h>
#include <hip/hip_runtime_api.h>
#include <pthread.h>
#include <unistd.h>

#include <array>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

struct Launch {
    int thread, call;
    std::string kernel;
    aq::TokArgs tok;  // of the token-tile kernels
    aq::TokMultiArgs multi;
    aq::QmmHalfArgs half;  // of the fp16-operand tiles
    bool is(const char* part) const { return kernel.find(part) != std::string::npos; }
};
static std::vector<Launch> log_;
static std::mutex log_mu;
static thread_local int this_thread = 0, this_call = 0;
static std::map<const void*, std::string>& names() {  // (filled while the library is being loaded)
    static std::map<const void*, std::string> m;
    return m;
}
static uintptr_t next_address = 1ull << 32;
static void* address(size_t n) {
    const uintptr_t p = next_address;
    next_address += (n + 511) & ~(size_t)255;
    return reinterpret_cast<void*>(p);
}

// Other threads get their turn wherever a lock is let go.
extern "C" int pthread_mutex_unlock(pthread_mutex_t* m) {
    static int (*const real)(pthread_mutex_t*) = reinterpret_cast<int (*)(pthread_mutex_t*)>(dlsym(RTLD_NEXT, "pthread_mutex_unlock"));
    const int rc = real(m);
    if (this_thread) usleep(20);
    return rc;
}

extern "C" {
void** __hipRegisterFatBinary(const void*) {
    static void* handle = nullptr;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) { names()[host] = name; }
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
static thread_local dim3 grid_, block_;
static thread_local size_t lds_;
static thread_local hipStream_t stream_;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
    grid_ = g, block_ = b, lds_ = lds, stream_ = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
    *g = grid_, *b = block_, *lds = lds_, *s = stream_;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* fn, dim3, dim3, void** args, size_t, hipStream_t) {
    std::lock_guard<std::mutex> lk(log_mu);
    Launch l{this_thread, this_call, names()[fn], {}, {}, {}};
    if (l.is("qmv_tok16_kernel")) l.tok = *static_cast<const aq::TokArgs*>(args[0]);
    if (l.is("qmv_tok16_multi_kernel")) l.multi = *static_cast<const aq::TokMultiArgs*>(args[0]);
    if (l.is("qmmh_kernel")) l.half = *static_cast<const aq::QmmHalfArgs*>(args[0]);
    log_.push_back(l);
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
static int compute_units = 256;
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {  // (the header's name for the versioned symbol)
    memset(p, 0, sizeof *p);
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = compute_units;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) { return *p = address(4 << 20), hipSuccess; }
static size_t allocated = 0;
hipError_t hipMalloc(void** p, size_t n) {
    allocated += n;
    return *p = address(n), hipSuccess;
}
hipError_t hipFree(void*) { return hipSuccess; }
hipError_t hipMemset(void*, int, size_t) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "?"; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = reinterpret_cast<hipStream_t>(16), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
static int drains = 0;
hipError_t hipStreamSynchronize(hipStream_t) { return drains++, hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
static bool capturing = false;
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
    return *s = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone, hipSuccess;
}
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = reinterpret_cast<hipEvent_t>(32), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
}

static int failures = 0;
#define CHECK(what, ...)                   \
    do {                                   \
        if (!(what)) {                     \
            failures++;                    \
            printf("%s: ", #what);         \
            printf(__VA_ARGS__);           \
            puts("");                      \
        }                                  \
    } while (0)

static aq_ctx* ctx;
static void* const X = address(1 << 24);
static void* const W = address((size_t)1 << 32);
static void* const S = address(1 << 28);
static void* const B = address(1 << 28);
static void* const Y = address(1 << 28);
static int qmv(int M, int K, int N, int group, int bits) { return aq_qmv(ctx, X, W, S, B, Y, M, K, N, group, bits, 0); }

// The launches of a call follow each other: with another thread's call between the one that fills scratch and the one that reads
// it, the reader finds what that call left there.
static void test_calls_stay_whole() {
    typedef int (*Call)();
    static const Call calls[] = {
        [] { return aq_qmv_greedy(ctx, X, W, S, B, nullptr, 0, static_cast<uint64_t*>(Y), 4, 1536, 3000, 32, 4); },
        [] { return aq_qmv_scores(ctx, X, W, S, B, nullptr, 0, static_cast<uint64_t*>(Y), 20, 14336, 700, 64, 4); },
        [] { return aq_qmv_gate_up(ctx, X, W, S, B, W, S, B, Y, 3, 768, 500, 64, 6, AQ_ACT_SILU, 0); },
        [] { return aq_qmv_gate_up(ctx, X, W, S, B, W, S, B, Y, 100, 768, 500, 64, 8, AQ_ACT_SILU, 0); },
        [] { return aq_qmv_act(ctx, X, Y, W, S, B, Y, 24, 14336, 640, 64, 4, AQ_ACT_SILU, 0); },
        [] { return aq_gather_qmv_gate_up(ctx, X, W, S, B, nullptr, static_cast<int32_t*>(S), Y, 9, 1, 768, 96, 4, 192, 0, 96, 64, 6, AQ_ACT_SILU, 0); },
        [] { return aq_gather_qmv_act(ctx, X, Y, W, S, B, nullptr, static_cast<int32_t*>(S), Y, 9, 1, 768, 96, 4, 96, 0, 64, 6, AQ_ACT_SILU, 0); },
        [] {
            const void *w[3] = {W, W, W}, *s[3] = {S, S, S}, *b[3] = {B, B, B};
            void* y[3] = {Y, Y, Y};
            const int N[3] = {600, 500, 1000};
            return aq_qmv_multi(ctx, X, 3, w, s, b, y, N, 40, 14336, 64, 4, 0);
        },
        [] {
            const void *w[3] = {W, W, W}, *s[3] = {S, S, S}, *b[3] = {B, B, B};
            void* y[3] = {Y, Y, Y};
            const int N[3] = {600, 500, 1000};
            return aq_qmm_multi(ctx, X, 3, w, s, b, y, N, 3, 768, 32, 4, 0);
        },
    };
    int several = 0;
    auto body = [&](int thread) {
        this_thread = thread;
        for (int round = 0; round < 4; round++)
            for (const Call& c : calls) {
                this_call++;
                const int rc = thread == 1 ? c() : qmv(24, 14336, 4096, 64, 4);
                std::lock_guard<std::mutex> lk(log_mu);
                CHECK(rc == AQ_OK, "thread %d call %d: %d %s", thread, this_call, rc, aq_last_error());
            }
        this_thread = 0;
    };
    log_.clear();
    std::thread one(body, 1), two(body, 2);
    one.join();
    two.join();
    std::map<std::pair<int, int>, size_t> last;
    for (size_t i = 0; i < log_.size(); i++) {
        const std::pair<int, int> call{log_[i].thread, log_[i].call};
        const auto before = last.find(call);
        if (before != last.end()) {
            several++;
            CHECK(before->second + 1 == i, "thread %d call %d: %s, then %s of thread %d, then %s", call.first, call.second,
                  log_[before->second].kernel.c_str(), log_[i - 1].kernel.c_str(), log_[i - 1].thread, log_[i].kernel.c_str());
        }
        last[call] = i;
    }
    CHECK(several >= 4 * 9, "%d launches behind another of their call", several);
}

// A row of x meets the same sums in a call of 9 rows as in one of 32 (and of 33 as of 64), recorded or not: the shares of K do not
// depend on the number of rows, and their partial tiles lie in a block that is there from the start, apart from each other.
static uintptr_t tiles_lo, tiles_hi;
static void tiles_used(const float* tile, size_t bytes) {
    const uintptr_t p = reinterpret_cast<uintptr_t>(tile);
    tiles_lo = p < tiles_lo ? p : tiles_lo;
    tiles_hi = p + bytes > tiles_hi ? p + bytes : tiles_hi;
}
static void test_shares() {
    int shared = 0, calls = 0;
    tiles_lo = UINTPTR_MAX, tiles_hi = 0;
    unsigned seed = 1;
    auto rnd = [&](int n) { return (int)((seed = seed * 1664525u + 1013904223u) >> 8) % n; };
    for (int i = 0; i < 1500; i++) {
        const int bits = i % 3 ? 4 : 8, group = 32 << rnd(3), K = 128 * (1 + rnd(128)), N = 16 + rnd(1 << (4 + rnd(12)));
        const bool pair = i % 4 == 3;
        for (int from : {9, 33}) {
            int ksplit = -1, share = 0;
            for (int M = from; M <= from + (from == 9 ? 23 : 31); M += 1 + rnd(7)) {
                log_.clear();
                capturing = (M + i) % 2;
                const size_t before = allocated;
                const int drained = drains;
                const int rc = pair ? aq_qmv_gate_up(ctx, X, W, S, B, W, S, B, Y, M, K, N, group, bits, AQ_ACT_SILU, 0) : qmv(M, K, N, group, bits);
                if (log_.empty() || !log_[0].is("qmv_tok16_kernel")) continue;  // (other kernels: they may want scratch, and be refused it)
                CHECK(rc == AQ_OK && allocated == before && drains == drained, "%d, %zu bytes allocated, the stream drained %d times", rc, allocated - before,
                      drains - drained);
                const aq::TokArgs& a = log_[0].tok;
                calls++;
                if (ksplit < 0) ksplit = a.ksplit, share = a.share;
                CHECK(a.ksplit == ksplit && a.share == share, "bits %d group %d K %d N %d pair %d: %d shares from %d rows, %d at %d", bits, group, K, N,
                      pair, ksplit, from, a.ksplit, M);
                if (a.ksplit <= 1) continue;
                shared++;
                tiles_used(a.tile, (size_t)a.ksplit * M * N * (pair ? 8 : 4));
                CHECK(log_.size() == 2 && log_[1].is("tok_reduce"), "%zu launches", log_.size());
            }
        }
    }
    capturing = false;
    CHECK(calls > 5000 && shared > 1000, "%d calls, %d of them shared K out", calls, shared);
    for (int i = 0; i < 300; i++) {
        const int M = 9 + rnd(24), K = 4096 + 256 * rnd(48);
        const void *w[4] = {W, W, W, W}, *s[4] = {S, S, S, S}, *b[4] = {B, B, B, B};
        void* y[4] = {Y, Y, Y, Y};
        const int N[4] = {16 + rnd(4096), 1 + rnd(20000), 16 + rnd(20000), 1 + rnd(4096)};
        log_.clear();
        CHECK(aq_qmv_multi(ctx, X, 4, w, s, b, y, N, M, K, 64, 4, 0) == AQ_OK, "%s", aq_last_error());
        for (const Launch& l : log_) {
            if (l.is("qmv_tok16_kernel") && l.tok.ksplit > 1) tiles_used(l.tok.tile, (size_t)l.tok.ksplit * M * l.tok.N * 4);
            uintptr_t end = 0;
            for (int m = 0; l.is("qmv_tok16_multi") && m < l.multi.count; m++) {
                if (l.multi.ksplit[m] <= 1) continue;
                CHECK(reinterpret_cast<uintptr_t>(l.multi.tile[m]) >= end, "member %d overlaps the one before it", m);
                end = reinterpret_cast<uintptr_t>(l.multi.tile[m]) + (size_t)l.multi.ksplit[m] * M * l.multi.N[m] * 4;
                tiles_used(l.multi.tile[m], (size_t)l.multi.ksplit[m] * M * l.multi.N[m] * 4);
            }
        }
    }
    CHECK(tiles_hi - tiles_lo <= aq::kTokTileBytes, "partial tiles over %zu bytes", (size_t)(tiles_hi - tiles_lo));
}

// Members of a grid that fills the chip work through their shares by themselves: no tiles, no second launch.
static void test_shares_inside() {
    struct Case {
        int bits, group, M, K, N[3];
    };
    static const Case cases[] = {{4, 64, 9, 5376, {4096, 2048, 2048}}, {8, 64, 32, 5312, {2047, 4090, 2048}}, {8, 32, 8, 5376, {4096, 2048, 2048}},
                                 {4, 32, 21, 5376, {4096, 2048, 2048}}, {8, 32, 21, 5376, {4096, 2048, 2048}}, {4, 32, 21, 6144, {1024, 6144, 1001}}};
    for (const Case& c : cases) {
        const void *w[3] = {W, W, W}, *s[3] = {S, S, S}, *b[3] = {B, B, B};
        void* y[3] = {Y, Y, Y};
        log_.clear();
        CHECK(aq_qmv_multi(ctx, X, 3, w, s, b, y, c.N, c.M, c.K, c.group, c.bits, 0) == AQ_OK, "%s", aq_last_error());
        int inside = 0;
        for (const int n : log_[0].multi.inside) inside += n > 1;
        CHECK(log_.size() == 1 && inside > 0, "%d rows of %d: %zu launches, %d members with shares of their own", c.M, c.K, log_.size(), inside);
    }
    // Halves of 64 rows: bands of all members begin on the first XCD, whose CUs would have two of these workgroups after another.
    for (auto [group, K, wide, narrow] : {std::array{64, 9600, 5248, 1344}, {128, 13568, 6272, 832}}) {
        const void *w[3] = {W, W, W}, *s[3] = {S, S, S}, *b[3] = {B, B, B};
        void* y[3] = {Y, Y, Y};
        const int N[3] = {wide, narrow, narrow};
        log_.clear();
        CHECK(aq_qmv_multi(ctx, X, 3, w, s, b, y, N, 64, K, group, 4, 0) == AQ_OK, "%s", aq_last_error());
        CHECK(log_.size() == 2 && log_[1].is("tok_reduce"), "64 rows of %d: %zu launches", K, log_.size());
    }
}

// A pair has two sets of rows a workgroup or more: what one would take is no reason to leave K whole.
static void test_shares_of_pairs() {
    for (auto [bits, M, K, N] : {std::array{8, 32, 6208, 1920}, {4, 24, 6208, 1920}, {8, 9, 5120, 2048}}) {
        log_.clear();
        CHECK(aq_qmv_gate_up(ctx, X, W, S, B, W, S, B, Y, M, K, N, 64, bits, AQ_ACT_SILU, 0) == AQ_OK, "%s", aq_last_error());
        CHECK(log_.size() == 2 && log_[1].is("tok_reduce"), "gate|up, %d bit, %d x %d x %d: %zu launches", bits, M, K, N, log_.size());
    }
}

// The calls that tests/test_gpu_group32_infinities.py makes for the launch that adds partial tiles.
static void test_shares_of_the_infinities() {
    auto tiles = [](int i) { return i < (int)log_.size() && log_[i].is("tok_reduce"); };
    for (int bits : {4, 8}) {
        for (auto [M, K, N] : {std::array{21, 15360, 100}, {21, 15360, 101}, {40, 15360, 600}, {63, 15360, 545}}) {
            log_.clear();
            CHECK(qmv(M, K, N, 32, bits) == AQ_OK && tiles(1), "%d bit, %d x %d x %d", bits, M, K, N);
            if (M == 63) continue;
            log_.clear();
            CHECK(aq_qmv_gate_up(ctx, X, W, S, B, W, S, B, Y, M, K, N, 32, bits, AQ_ACT_SILU, 0) == AQ_OK && tiles(1), "gate|up, %d bit, %d x %d x %d",
                  bits, M, K, N);
        }
        for (auto [M, K, wide] : {std::array{21, 5120, 12000}, {40, 5120, 6000}}) {
            const void *w[2] = {W, W}, *s[2] = {S, S}, *b[2] = {B, B};
            void* y[2] = {Y, Y};
            const int N[2] = {wide, M == 21 ? 100 : 600};
            log_.clear();
            CHECK(aq_qmv_multi(ctx, X, 2, w, s, b, y, N, M, K, 32, bits, 0) == AQ_OK && tiles(1), "members, %d bit, %d x %d", bits, M, K);
            CHECK(log_[0].multi.count == 2 && log_[0].multi.ksplit[0] == 1 && log_[0].multi.ksplit[1] > 1, "members, %d bit, %d x %d: %d and %d shares", bits,
                  M, K, log_[0].multi.ksplit[0], log_[0].multi.ksplit[1]);
        }
    }
}

// Tiles and shares of K of prompts, where the costs of the tiles decide and measured far apart (us, the other form -> this one).
static void test_tiles_of_prompts() {
    auto prompt = [](int M, int K, int N, int group, int bits) {
        log_.clear();
        CHECK(aq_qmm(ctx, X, W, S, B, Y, M, K, N, group, bits, 0) == AQ_OK, "%s", aq_last_error());
        return log_.size();
    };
    // (pass over x, tiles, sums of shares)
    for (auto [M, K, N, group, bits] : {std::array{2048, 14336, 4096, 64, 4}, {999, 9920, 4032, 64, 8}, {509, 15360, 3840, 32, 4}})  // 255 -> 234, 159 -> 121
        CHECK(prompt(M, K, N, group, bits) == 3 && log_[2].is("qmmh_reduce"), "%d x %d x %d, %d bit: %zu launches", M, K, N, bits, log_.size());
    CHECK(prompt(333, 1024, 1024, 64, 8) == 2, "333 rows: %zu launches", log_.size());  // 15 -> 14
    // q|k|v of a prompt of 8 bit: 64 x 128 tiles, three workgroups a CU (55 -> 52)
    const void *w[3] = {W, W, W}, *s[3] = {S, S, S}, *b[3] = {B, B, B};
    void* y[3] = {Y, Y, Y};
    const int N[3] = {2048, 512, 512};
    log_.clear();
    CHECK(aq_qmm_multi(ctx, X, 3, w, s, b, y, N, 777, 2560, 64, 8, 0) == AQ_OK && log_.size() > 1, "%s", aq_last_error());
    CHECK(log_[1].is("qmmh_kernelILi8ELi1ELi2ELi2ELi2E"), "q|k|v of 777 rows: %s", log_[1].kernel.c_str());
    // a pair that three shares of either matrix would not shorten (24.5 -> 22)
    log_.clear();
    CHECK(aq_qmv_gate_up(ctx, X, W, S, B, W, S, B, Y, 128, 1152, 3840, 32, 8, AQ_ACT_SILU, 0) == AQ_OK && log_.size() == 2, "gate|up of 128 rows: %zu launches", log_.size());
    // k and v beside a q that fills the chip stay whole (64 -> 53)
    const int wide[3] = {2688, 576, 576};
    log_.clear();
    CHECK(aq_qmm_multi(ctx, X, 3, w, s, b, y, wide, 1966, 1920, 32, 4, 0) == AQ_OK && log_.size() == 2, "q|k|v of 1966 rows: %zu launches", log_.size());
}

// Who adds the shares of K in the calls of tests/test_gpu_share_sums.py: of each of the members, the last workgroup of a tile (T), a
// second kernel (K), or nobody (-).
static void test_who_adds_shares() {
    struct Case {
        int bits, group, M, K, N[3];
        const char* adds;
    };
    static const Case cases[] = {
        {4, 64, 65, 4096, {515, 130, 64}, "KKK"}, {4, 32, 96, 3840, {1100, 33, 257}, "KKK"}, {4, 128, 129, 8192, {1024, 512, 31}, "KKK"},
        {8, 64, 66, 3072, {3072, 96, 1000}, "KKK"}, {8, 32, 200, 2048, {640, 513, 64}, "TTT"}, {4, 64, 300, 2816, {704, 2050, 1}, "KKK"},
        {4, 32, 500, 8192, {2048, 72, 95}, "KKK"}, {8, 64, 777, 10240, {2560, 256, 17}, "KKK"}, {4, 64, 129, 2816, {3072, 96, 1000}, "TKK"},
        {4, 32, 300, 2048, {4096, 1024, 33}, "-TT"}, {4, 128, 777, 2048, {1100, 33, 257}, "TKK"}, {4, 64, 500, 4096, {3072, 96, 1000}, "TKK"},
        {4, 64, 777, 2048, {4096, 1024, 33}, "-TK"}, {8, 64, 300, 4096, {2048, 513, 513}, "TKK"}, {8, 32, 500, 2816, {3072, 96, 1000}, "-TK"}};
    for (const Case& c : cases) {
        const void *w[3] = {W, W, W}, *s[3] = {S, S, S}, *b[3] = {B, B, B};
        void* y[3] = {Y, Y, Y};
        log_.clear();
        CHECK(aq_qmm_multi(ctx, X, 3, w, s, b, y, c.N, c.M, c.K, c.group, c.bits, 0) == AQ_OK && log_.size() >= 2 && log_[1].is("qmmh_kernel"), "%s", aq_last_error());
        std::string adds;
        for (int i = 0; i < 3; i++) adds += !log_[1].half.seg[i].partial ? '-' : log_[1].half.seg[i].tickets ? 'T' : 'K';
        CHECK(adds == c.adds && log_.size() == (adds.find('K') == std::string::npos ? 2 : 3), "%d bit, %d rows of %d: %s, %zu launches", c.bits, c.M, c.K, adds.c_str(),
              log_.size());
    }
}

// A recorded call whose workspace holds a member at a time, not the grid: one pass over x, and a launch that clears the tickets ahead of a later
// member's tiles (tests/test_gpu_share_sums.py runs it).
static void test_tickets_of_members_one_by_one() {
    aq_ctx* own = nullptr;
    CHECK(aq_create(0, &own) == AQ_OK, "%s", aq_last_error());
    const void *w[3] = {W, W, W}, *s[3] = {S, S, S}, *b[3] = {B, B, B};
    void* y[3] = {Y, Y, Y};
    const int N[3] = {515, 500, 130};
    CHECK(aq_qmm(own, X, W, S, B, Y, 65, 2048, N[0], 64, 4, 0) == AQ_OK, "%s", aq_last_error());
    log_.clear();
    capturing = true;
    CHECK(aq_qmm_multi(own, X, 3, w, s, b, y, N, 65, 2048, 64, 4, 0) == AQ_OK, "%s", aq_last_error());
    capturing = false;
    std::string kernels;
    for (const Launch& l : log_) kernels += l.is("prep") ? 'x' : l.is("qmmh_kernel") ? l.half.seg[0].tickets ? 'T' : '-' : l.is("fill") ? '0' : '?';
    CHECK(kernels == "xT0T0T", "%s, the last %s", kernels.c_str(), log_.back().kernel.c_str());
    aq_destroy(own);
}

// The list of an expert block's routes: beside the pass over x while it takes up to 40 KiB of LDS, behind that a launch of its own.
static void test_lists_of_routes() {
    for (auto [routes, launches] : {std::array{5056, 2}, {5057, 3}}) {
        log_.clear();
        CHECK(aq_gather_qmv_gate_up(ctx, X, W, S, B, static_cast<int32_t*>(S), static_cast<int32_t*>(S), Y, routes, 1000, 256, 776, 128, 2 * 776, 0, 776, 64, 4, AQ_ACT_SILU, 0) == AQ_OK,
              "%s", aq_last_error());
        CHECK((int)log_.size() == launches && log_.back().is("qmmr_kernel"), "%d routes: %zu launches, the last %s", routes, log_.size(), log_.back().kernel.c_str());
    }
}

// What include/aq_mi355.h says of the launches of a few rows: of q|k|v, and of the gated pair (0: the projections apart).
static void test_launches_of_few_rows() {
    struct Case {
        int bits, group, M, K, members, pair;
    };
    static const Case cases[] = {
        {4, 64, 1, 4096, 1, 1}, {4, 64, 4, 1152, 1, 1}, {4, 64, 4, 8192, 1, 1}, {4, 64, 4, 16384, 1, 0}, {4, 64, 2, 8320, 1, 0}, {4, 64, 5, 1152, 1, 1},
        {4, 64, 8, 4096, 1, 1}, {4, 64, 5, 4224, 6, 2}, {4, 64, 8, 8192, 6, 2}, {4, 64, 8, 8320, 6, 0}, {4, 64, 6, 16384, 6, 0}, {4, 64, 4, 1024, 1, 1},
        {4, 64, 8, 1024, 2, 2}, {4, 64, 5, 4160, 2, 2}, {4, 64, 8, 16448, 2, 2}, {4, 64, 3, 14400, 1, 1}, {4, 32, 2, 1216, 1, 1}, {4, 32, 2, 1536, 3, 0},
        {4, 128, 4, 1152, 1, 1}, {4, 128, 4, 2048, 1, 1}, {8, 128, 4, 2048, 1, 1}, {8, 64, 4, 896, 1, 1}, {8, 64, 4, 4096, 1, 0}, {8, 64, 4, 3072, 1, 1},
        {8, 64, 5, 4096, 1, 1}, {4, 64, 32, 4096, 1, 1}, {4, 32, 3, 1216, 1, 1}};
    for (const Case& c : cases) {
        const void *w[3] = {W, W, W}, *s[3] = {S, S, S}, *b[3] = {B, B, B};
        void* y[3] = {Y, Y, Y};
        const int N[3] = {2048, 512, 512};
        log_.clear();
        CHECK(aq_qmv_multi(ctx, X, 3, w, s, b, y, N, c.M, c.K, c.group, c.bits, 0) == AQ_OK && (int)log_.size() == c.members,
              "q|k|v, %d bit, groups of %d, %d rows of %d: %zu launches", c.bits, c.group, c.M, c.K, log_.size());
        log_.clear();
        CHECK(aq_qmv_gate_up(ctx, X, W, S, B, W, S, B, Y, c.M, c.K, 2048, c.group, c.bits, AQ_ACT_SILU, 0) == AQ_OK, "%s", aq_last_error());
        const bool apart = log_.back().is("act_mul");
        CHECK(apart ? c.pair == 0 : (int)log_.size() == c.pair, "gate|up, %d bit, groups of %d, %d rows of %d: %zu launches, the last %s", c.bits, c.group,
              c.M, c.K, log_.size(), log_.back().kernel.c_str());
    }
}

int main() {
    for (int cus : {128, 512, 256}) {
        compute_units = cus;
        if (aq_create(0, &ctx) != AQ_OK) {
            printf("aq_create: %s\n", aq_last_error());
            return 1;
        }
        test_shares();
        if (cus == 256) test_calls_stay_whole(), test_shares_inside(), test_shares_of_pairs(), test_shares_of_the_infinities(), test_tiles_of_prompts(), test_launches_of_few_rows(), test_who_adds_shares(), test_tickets_of_members_one_by_one(), test_lists_of_routes();
        aq_destroy(ctx);
    }
    if (!failures) puts("ok");
    return failures ? 1 : 0;
}
