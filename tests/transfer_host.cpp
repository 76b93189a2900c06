// The host side of csrc/isph_transfer.hip against a stand-in for the HIP runtime
// that runs on the CPU: streams that can be held busy, devices that calls have to
// match, and kernel launches that do what k_pack does.  The first argument names
// the scenario; 0 is returned if it went as it should.
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstring>
#include <future>
#include <mutex>
#include <thread>
#include <vector>

#include "isph_host.h"

struct ihipStream_t {
    int device = 0;
    bool busy = false;
    std::mutex lock;
    std::condition_variable idle;
    void wait() {
        std::unique_lock<std::mutex> g(lock);
        idle.wait(g, [&] { return !busy; });
    }
    void release() {
        std::lock_guard<std::mutex> g(lock);
        busy = false;
        idle.notify_all();
    }
};
struct ihipEvent_t {
    int device = 0;
    ihipStream_t* stream = nullptr;
};
static bool no_pinned = false;
static thread_local int current = 0;
static thread_local struct { dim3 grid, block; size_t lds; hipStream_t stream; } config;

// k_pack's table of columns
struct PackCols {
    const char* src[isph::MAX_COLUMNS];
    int stride[isph::MAX_COLUMNS], size[isph::MAX_COLUMNS];
    size_t at[isph::MAX_COLUMNS];
    int ncol;
};

extern "C" {
hipError_t hipGetDevice(int* d) { *d = current; return hipSuccess; }
hipError_t hipSetDevice(int d) { current = d; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    if (no_pinned) return hipErrorOutOfMemory;
    *p = malloc(n);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
    st->wait();
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) { s->wait(); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = new ihipEvent_t;
    (*e)->device = current;
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    if (e->device != s->device) return hipErrorInvalidHandle;
    e->stream = s;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) { e->stream->wait(); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t l, hipStream_t s) {
    config = {g, b, l, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* l, hipStream_t* s) {
    *g = config.grid;
    *b = config.block;
    *l = config.lds;
    *s = config.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3 grid, dim3 block, void** a, size_t, hipStream_t s) {
    if (current != s->device) return hipErrorInvalidHandle;
    s->wait();
    const int64_t r0 = *(int64_t*)a[0];
    const int rows = *(int*)a[1];
    const PackCols& c = *(PackCols*)a[2];
    char* out = *(char**)a[3];
    if ((int)(grid.x * block.x) < rows) return hipErrorInvalidValue;
    for (int k = 0; k < c.ncol; ++k)
        for (int i = 0; i < rows; ++i)
            memcpy(out + c.at[k] + (size_t)i * c.size[k],
                   c.src[k] + (size_t)(r0 + i) * c.stride[k], c.size[k]);
    return hipSuccess;
}
void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*,
                           void*, int*) {}
void __hipUnregisterFatBinary(void**) {}
}

using namespace isph::host;

struct Particles {
    ihipStream_t stream;
    isph_ctx ctx;
    std::vector<double> pos;  // (x, y) pairs
    std::vector<int> id;
    std::vector<double> x, y;
    std::vector<int> id_out;
    Particles(int n, int device, int seed) : pos(2 * n), id(n), x(n), y(n), id_out(n) {
        for (int i = 0; i < 2 * n; ++i) pos[i] = seed + 0.5 * i;
        for (int i = 0; i < n; ++i) id[i] = seed - i;
        stream.device = device;
        ctx.stream = &stream;
        ctx.device = device;
        transfer_attach();
    }
    int get() {
        const Column c[] = {{pos.data(), 16, 8, x.data()},
                            {pos.data() + 1, 16, 8, y.data()},
                            {id.data(), 4, 4, id_out.data()}};
        return download(&ctx, (int64_t)id.size(), c, 3);
    }
    bool right() const {
        for (size_t i = 0; i < id.size(); ++i)
            if (x[i] != pos[2 * i] || y[i] != pos[2 * i + 1] || id_out[i] != id[i]) return false;
        return true;
    }
};

#define CHECK(e) \
    do { if (!(e)) { printf("line %d: %s\n", __LINE__, #e); fflush(stdout); _Exit(1); } } while (0)

// A context's queued work keeps neither another one's downloads nor its creation
// and destruction waiting.
static void busy(int rows) {
    Particles a(rows, 0, 3), b(rows, 0, 7);
    a.stream.busy = true;
    auto fa = std::async(std::launch::async, [&] { return a.get(); });
    std::this_thread::sleep_for(std::chrono::milliseconds(200));
    auto fb = std::async(std::launch::async, [&] {
        transfer_attach();
        const int rc = b.get();
        transfer_detach();
        return rc;
    });
    CHECK(fb.wait_for(std::chrono::seconds(20)) == std::future_status::ready);
    CHECK(fb.get() == ISPH_OK && b.right());
    CHECK(fa.wait_for(std::chrono::milliseconds(0)) != std::future_status::ready);
    a.stream.release();
    CHECK(fa.get() == ISPH_OK && a.right());
}

// More threads than slots, over and over.
static void crowd(int rows) {
    std::vector<std::thread> th;
    for (int t = 0; t < 6; ++t)
        th.emplace_back([=] {
            Particles p(rows + 13 * t, 0, 100 * t);
            for (int k = 0; k < 5; ++k) {
                std::fill(p.x.begin(), p.x.end(), -1.0);
                CHECK(p.get() == ISPH_OK && p.right());
            }
            transfer_detach();
        });
    for (auto& t : th) t.join();
}

// The calling thread's current device is another than the context's, and stays so.
static void device(int rows) {
    Particles p(rows, 1, 5);
    CHECK(hipSetDevice(2) == hipSuccess);
    CHECK(p.get() == ISPH_OK && p.right());
    int now = -1;
    CHECK(hipGetDevice(&now) == hipSuccess && now == 2);
    transfer_detach();
}

int main(int argc, char** argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    for (int rows : {1, 65, 200000, 700001}) {
        if (what == "busy") busy(rows);
        if (what == "busy_unpinned") {
            no_pinned = true;
            busy(rows);
        }
        if (what == "crowd") crowd(rows);
        if (what == "device") device(rows);
    }
    return 0;
}
