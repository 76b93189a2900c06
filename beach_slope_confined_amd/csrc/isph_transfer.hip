// isph_transfer.hip -- particle arrays and fields to host memory.
//
// The caller's arrays are pageable, and a copy to pageable memory goes through
// the runtime's own staging one array at a time: 80 MB of particles took 18 ms,
// a tenth of the link's 57 GB/s, most of it in the host's single-threaded
// copies, page faults and the splitting of (x, y) pairs.  Here a kernel writes
// the columns of a chunk of rows, pairs split, straight into pinned memory, and
// several threads each take chunk after chunk: launch, wait, copy out.  Their
// copies and page faults overlap with each other and with the link.  All
// particle arrays: 2.5k rows 0.30 -> 0.05 ms, 93k 0.59 -> 0.28 ms, 1.06M
// 18.4 -> 2.9 ms, 4.26M 65 -> 8.9 ms (36 GB/s of the link's 57).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

#include "isph_host.h"

namespace isph {

struct PackCols {
    const char* src[MAX_COLUMNS];
    int stride[MAX_COLUMNS];  // bytes from a row's value to the next one's
    int size[MAX_COLUMNS];    // 4 or 8
    size_t at[MAX_COLUMNS];   // byte offset of the column in the chunk
    int ncol;
};

// rows [r0, r0 + rows) of the columns, one after the other, into `out`
__global__ void __launch_bounds__(BLOCK) k_pack(int64_t r0, int rows, PackCols c, char* out) {
    const int i = blockIdx.x * BLOCK + threadIdx.x;
    if (i >= rows) return;
    for (int k = 0; k < c.ncol; ++k) {
        const char* s = c.src[k] + (size_t)(r0 + i) * c.stride[k];
        char* d = out + c.at[k] + (size_t)i * c.size[k];
        if (c.size[k] == 8)
            *reinterpret_cast<double*>(d) = *reinterpret_cast<const double*>(s);
        else
            *reinterpret_cast<int*>(d) = *reinterpret_cast<const int*>(s);
    }
}

namespace host {

namespace {

// Pinned staging of the process: slots that the downloads of all contexts share,
// a chunk at a time.  Allocated at the first download, kept while contexts live
// (10 MB), given back with the last one.  Whoever holds a slot waits for nothing
// but its own chunk, so contexts on other streams and GPUs go on meanwhile.
constexpr int SLOTS = 8;
constexpr size_t SLOT_BYTES = 1280 * 1024;
std::mutex pool_lock;
std::condition_variable pool_given;
char* pool = nullptr;
int pool_users = 0;
unsigned pool_free = (1u << SLOTS) - 1;

// the pool's memory; null if there is none to be had
char* pool_memory() {
    std::lock_guard<std::mutex> g(pool_lock);
    if (!pool && hipHostMalloc((void**)&pool, SLOTS * SLOT_BYTES, hipHostMallocPortable) != hipSuccess) {
        pool = nullptr;
        (void)hipGetLastError();
    }
    return pool;
}

int take_slot() {
    std::unique_lock<std::mutex> g(pool_lock);
    pool_given.wait(g, [] { return pool_free != 0; });
    const int slot = __builtin_ctz(pool_free);
    pool_free &= ~(1u << slot);
    return slot;
}

void give_slot(int slot) {
    {
        std::lock_guard<std::mutex> g(pool_lock);
        pool_free |= 1u << slot;
    }
    pool_given.notify_one();
}

// The calling thread works on a device for as long as this lives: a launch and
// an event belong to the current device, a copy on a stream did not need it.
class OnDevice {
public:
    explicit OnDevice(int device) {
        status = hipGetDevice(&before);
        if (status == hipSuccess && before != device) {
            status = hipSetDevice(device);
            moved = status == hipSuccess;
        }
    }
    ~OnDevice() {
        if (moved) (void)hipSetDevice(before);
    }
    hipError_t status;

private:
    int before = 0;
    bool moved = false;
};

}  // namespace

void transfer_attach() {
    std::lock_guard<std::mutex> g(pool_lock);
    ++pool_users;
}

void transfer_detach() {
    std::lock_guard<std::mutex> g(pool_lock);
    if (--pool_users == 0 && pool) {
        (void)hipHostFree(pool);
        pool = nullptr;
    }
}

int download(isph_ctx* c, int64_t rows, const Column* cols, int ncol) {
    if (rows <= 0 || ncol <= 0) return ISPH_OK;
    size_t bytes = 0;  // of a row
    for (int k = 0; k < ncol; ++k) bytes += cols[k].size;
    const OnDevice there(c->device);
    HIPCHK(c, there.status);
    HIPCHK(c, hipStreamSynchronize(c->stream));  // before a slot is held
    char* const mem = pool_memory();
    if (!mem) {  // no pinned memory: through the runtime's own staging
        std::vector<char> t;
        for (int k = 0; k < ncol; ++k) {
            const Column& q = cols[k];
            const bool dense = q.stride == q.size;
            const size_t len = (size_t)(rows - 1) * q.stride + q.size;
            if (!dense) t.resize(len);
            HIPCHK(c, hipMemcpyAsync(dense ? q.dst : t.data(), q.src, len, hipMemcpyDeviceToHost,
                                     c->stream));
            HIPCHK(c, hipStreamSynchronize(c->stream));
            for (int64_t i = 0; !dense && i < rows; ++i)
                memcpy(static_cast<char*>(q.dst) + i * q.size, t.data() + i * q.stride, q.size);
        }
        return ISPH_OK;
    }
    // rows of a chunk: columns begin at multiples of 64 rows
    const int64_t most = (int64_t)(SLOT_BYTES / bytes) & ~int64_t(63);
    const int64_t nchunk = (rows + most - 1) / most;
    const int64_t per = ((rows + nchunk - 1) / nchunk + 63) & ~int64_t(63);
    PackCols pc{};
    pc.ncol = ncol;
    size_t at = 0;
    for (int k = 0; k < ncol; ++k) {
        pc.src[k] = static_cast<const char*>(cols[k].src);
        pc.stride[k] = cols[k].stride;
        pc.size[k] = cols[k].size;
        pc.at[k] = at;
        at += (size_t)per * cols[k].size;
    }
    std::atomic<int64_t> next{0};
    std::atomic<int> status{hipSuccess};
    auto work = [&](int thread) {
        hipEvent_t ev = nullptr;
        // a thread of our own starts on device 0
        hipError_t e = thread ? hipSetDevice(c->device) : hipSuccess;
        if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
        while (e == hipSuccess && status.load() == hipSuccess) {
            const int64_t r0 = per * next.fetch_add(1);
            if (r0 >= rows) break;
            const int m = (int)std::min<int64_t>(per, rows - r0);
            const int slot = take_slot();
            char* buf = mem + (size_t)slot * SLOT_BYTES;
            k_pack<<<nblk(m), BLOCK, 0, c->stream>>>(r0, m, pc, buf);
            e = hipGetLastError();
            if (e == hipSuccess) e = hipEventRecord(ev, c->stream);
            if (e == hipSuccess) e = hipEventSynchronize(ev);
            for (int k = 0; e == hipSuccess && k < ncol; ++k)
                memcpy(static_cast<char*>(cols[k].dst) + (size_t)r0 * cols[k].size,
                       buf + pc.at[k], (size_t)m * cols[k].size);
            if (e != hipSuccess) (void)hipStreamSynchronize(c->stream);  // it may be written still
            give_slot(slot);
        }
        if (ev) (void)hipEventDestroy(ev);
        if (e != hipSuccess) status.store(e);
    };
    const int threads = (int)std::min<int64_t>(SLOTS, nchunk);
    std::thread th[SLOTS];
    int started = 1;  // the calling thread is the first
    try {
        for (; started < threads; ++started) th[started] = std::thread(work, started);
    } catch (...) {  // fewer threads then
    }
    work(0);
    for (int k = 1; k < started; ++k) th[k].join();
    HIPCHK(c, (hipError_t)status.load());
    return ISPH_OK;
}

}  // namespace host
}  // namespace isph
