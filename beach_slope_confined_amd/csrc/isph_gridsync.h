// isph_gridsync.h -- grid-wide sums for kernels whose blocks all stay resident
// (cooperative launches).  Worker blocks publish their part of a sum; one more
// block, the leader, reads all parts, finishes the reduction and broadcasts
// what the workers need of it.  The exchange is reduction and barrier in one.
// Small grids do without the leader: every block reads all parts.
//
// Every published 64-bit word carries 32 bits of data under a 32-bit epoch
// number, so it is valid by itself and no flag has to follow the data.  Words
// are written and read with agent-scope atomics, which go past the XCDs'
// private L2 caches.  Two buffers alternate by epoch: a worker publishes epoch
// e + 2 only after the broadcast of e + 1, for which the leader needed every
// worker's part of e + 1, and a worker publishes that after it has read the
// broadcast of e, or without a leader all parts of e; likewise for the
// leader's words.  The words are zeroed
// before each launch and epochs count from 1.
//
// Vector entries that other blocks read after an exchange are stored with
// agent-scope atomics (write-through, so nothing has to be written back) and
// are complete (vmcnt 0) before the block publishes; the readers load them
// with agent-scope atomics after the exchange.  Their owner may store to them
// again once it has passed a further exchange in which every reader published
// after its reads; a reader that has published is waited for by no one, so what
// it reads after that needs one exchange more.  No cache is written back or
// invalidated: at 256 blocks an exchange costs 2.0 us this way, 14 us with a
// release and an acquire fence of agent scope, and 3.4 us if every block reads
// every part itself.
//
// Every wait is bounded (GS_SPIN polls, about a second): a block that gives up
// raises ERR_SYNC and ends, the others run into their own bounds, and the grid
// drains.
#pragma once
#include "isph_kernels.h"

namespace isph {

constexpr int GS_MAXB = 256;      // blocks of a resident grid, one per CU, the leader included
constexpr int GS_PARTS = 5120 + 256;  // published parts of a sum, and room for partial sums
constexpr int GS_LINES = 32;      // copies of the broadcast, one per 128-byte line
constexpr int GS_LINE = 16;       // words of a line
constexpr int GS_SPIN = 1 << 20;  // polls before a block gives up

typedef unsigned long long gs_word;

// words of both buffers: the broadcast lines, then 4 per part
constexpr int gs_words(int parts) { return 2 * (GS_LINES * GS_LINE + 4 * parts); }

struct GridSync {
    gs_word* words;
    uint32_t* err;    // error bits
    uint32_t* state;  // GS_REFUSED, GS_WRITTEN; cleared with the words
    int parts;        // a multiple of 256
};
constexpr uint32_t GS_REFUSED = 1u;  // some block cannot hold its rows: nothing was done
constexpr uint32_t GS_WRITTEN = 2u;  // a block has written its part of the result

__device__ __forceinline__ gs_word* gs_part(const GridSync& g, uint32_t e, int part) {
    return g.words + 2 * GS_LINES * GS_LINE + (size_t)(e & 1) * 4 * g.parts + part;
}
__device__ __forceinline__ gs_word* gs_line(const GridSync& g, uint32_t e, int line) {
    return g.words + ((size_t)(e & 1) * GS_LINES + line) * GS_LINE;
}

template <class T>
__device__ __forceinline__ void gs_store(T* p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ T gs_load(const T* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ gs_word gs_hi(uint32_t e, double v) {
    return ((gs_word)e << 32) | ((gs_word)__double_as_longlong(v) >> 32);
}
__device__ __forceinline__ gs_word gs_lo(uint32_t e, double v) {
    return ((gs_word)e << 32) | ((gs_word)__double_as_longlong(v) & 0xffffffffull);
}
__device__ __forceinline__ double gs_value(gs_word hi, gs_word lo) {
    return __longlong_as_double((long long)((hi << 32) | (lo & 0xffffffffull)));
}

// worker: a thread publishes one part of epoch e
__device__ __forceinline__ void gs_publish(const GridSync& g, uint32_t e, int part, bool two,
                                           double v0, double v1) {
    gs_word* w = gs_part(g, e, part);
    gs_store(w, gs_hi(e, v0));
    gs_store(w + g.parts, gs_lo(e, v0));
    if (two) {
        gs_store(w + 2 * g.parts, gs_hi(e, v1));
        gs_store(w + 3 * g.parts, gs_lo(e, v1));
    }
}

// Words that a thread waits for besides an exchange's: they are requested with
// every poll, and the wait goes on until they are valid too.
struct GsNone {
    __device__ __forceinline__ void request() {}
    __device__ __forceinline__ bool valid() const { return true; }
    __device__ __forceinline__ bool wait() { return true; }
};

// leader: a thread reads the N parts first, first + stride, .. of epoch e that
// lie below `count` (the others are 0); false if one did not come
template <int N, class More>
__device__ __forceinline__ bool gs_collect(const GridSync& g, uint32_t e, int first, int stride,
                                           int count, bool two, double* v0, double* v1,
                                           More& more) {
    for (int spin = 0; spin < GS_SPIN; ++spin) {
        more.request();
        gs_word x[N][4];
#pragma unroll
        for (int m = 0; m < N; ++m) {
            const bool in = first + m * stride < count;
            const gs_word* w = gs_part(g, e, in ? first + m * stride : first);
#pragma unroll
            for (int q = 0; q < 4; ++q)
                x[m][q] = in && (q < 2 || two) ? gs_load(w + q * g.parts) : (gs_word)e << 32;
        }
        bool ok = more.valid();
#pragma unroll
        for (int m = 0; m < N; ++m)
#pragma unroll
            for (int q = 0; q < 4; ++q) ok = ok && (uint32_t)(x[m][q] >> 32) == e;
        if (ok) {
#pragma unroll
            for (int m = 0; m < N; ++m) {
                v0[m] = gs_value(x[m][0], x[m][1]);
                v1[m] = gs_value(x[m][2], x[m][3]);
            }
            return true;
        }
    }
    return false;
}

template <int N>
__device__ __forceinline__ bool gs_collect(const GridSync& g, uint32_t e, int first, int stride,
                                           int count, bool two, double* v0, double* v1) {
    GsNone none;
    return gs_collect<N>(g, e, first, stride, count, two, v0, v1, none);
}

// leader: threads 0 .. GS_LINES - 1 broadcast a value and a flag
__device__ __forceinline__ void gs_broadcast(const GridSync& g, uint32_t e, double v, int flag) {
    if (threadIdx.x < GS_LINES) {
        gs_word* w = gs_line(g, e, threadIdx.x);
        gs_store(w, gs_hi(e, v));
        gs_store(w + 1, gs_lo(e, v));
        gs_store(w + 2, ((gs_word)e << 32) | (uint32_t)flag);
    }
}

// worker: every wave reads the broadcast of epoch e for itself
__device__ __forceinline__ bool gs_receive(const GridSync& g, uint32_t e, int block, double& v,
                                           int& flag) {
    const int lane = threadIdx.x & 63;
    const gs_word* w = gs_line(g, e, block & (GS_LINES - 1)) + min(lane, 2);
    for (int spin = 0; spin < GS_SPIN; ++spin) {
        const gs_word x = gs_load(w);
        if (__all((uint32_t)(x >> 32) == e)) {
            const gs_word hi = __shfl(x, 0, 64), lo = __shfl(x, 1, 64), f = __shfl(x, 2, 64);
            v = gs_value(hi, lo);
            flag = (int)(uint32_t)f;
            // keeps the compiler from moving later loads up; no cache action
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
            return true;
        }
    }
    return false;
}
}  // namespace isph
