// isph_copy.hip -- several device arrays copied in one launch.
//
// A state is 19 arrays, a tape entry of the adjoint 68.  Small arrays are bound
// by the copies' launches (about 2.5 us each, whatever their size up to 1 MB), so
// one launch takes up to COPY_MAX arrays, a block per 16 KB piece; large ones
// are bound by memory either way.  2 steps of the 2.5k-particle dam with their
// restore 9.14 -> 8.92 ms, 8 steps forward and back at 133k particles about 1%.
#include <hip/hip_runtime.h>

#include "isph_host.h"

namespace isph {

constexpr int COPY_MAX = 24;
constexpr int COPY_PIECE = 16384;  // bytes of a block: four 16-byte words a thread

struct CopyTable {
    const char* src[COPY_MAX];
    char* dst[COPY_MAX];
    size_t bytes[COPY_MAX];   // a multiple of 4
    int first[COPY_MAX];      // first block of an array; past the last one, the number of blocks
};

__global__ void __launch_bounds__(BLOCK) k_copy_arrays(CopyTable t) {
    int a = 0;
#pragma unroll
    for (int k = 1; k < COPY_MAX; ++k)
        if ((int)blockIdx.x >= t.first[k]) a = k;
    const size_t at = (size_t)(blockIdx.x - t.first[a]) * COPY_PIECE;
    const size_t left = t.bytes[a] - at;
    const int len = left < (size_t)COPY_PIECE ? (int)left : COPY_PIECE;
    const char* s = t.src[a] + at;
    char* d = t.dst[a] + at;
    // whole words of 16 bytes where both addresses allow it, 4 bytes otherwise
    // and for the rest
    int done = 0;
    if ((((size_t)s | (size_t)d) & 15) == 0) {
        const int m = len / 16;
        const uint4* s4 = reinterpret_cast<const uint4*>(s);
        uint4* d4 = reinterpret_cast<uint4*>(d);
        constexpr int Q = COPY_PIECE / 16 / BLOCK;
        uint4 w[Q];
#pragma unroll
        for (int q = 0; q < Q; ++q)
            if ((int)threadIdx.x + q * BLOCK < m) w[q] = s4[threadIdx.x + q * BLOCK];
#pragma unroll
        for (int q = 0; q < Q; ++q)
            if ((int)threadIdx.x + q * BLOCK < m) d4[threadIdx.x + q * BLOCK] = w[q];
        done = m * 16;
    }
    for (int e = done + 4 * (int)threadIdx.x; e < len; e += 4 * BLOCK)
        *reinterpret_cast<uint32_t*>(d + e) = *reinterpret_cast<const uint32_t*>(s + e);
}

namespace host {

int copy_arrays(isph_ctx* c, const ArrayCopy* a, int n) {
    for (int i0 = 0; i0 < n; i0 += COPY_MAX) {
        CopyTable t;
        int64_t blocks = 0;
        for (int k = 0; k < COPY_MAX; ++k) {
            const bool in = i0 + k < n;
            const size_t b = in ? a[i0 + k].bytes : 0;
            t.src[k] = in ? static_cast<const char*>(a[i0 + k].src) : nullptr;
            t.dst[k] = in ? static_cast<char*>(a[i0 + k].dst) : nullptr;
            t.bytes[k] = b;
            t.first[k] = (int)blocks;
            blocks += (int64_t)((b + COPY_PIECE - 1) / COPY_PIECE);
        }
        if (blocks > 0) k_copy_arrays<<<(unsigned)blocks, BLOCK, 0, c->stream>>>(t);
    }
    HIPCHK(c, hipGetLastError());
    return ISPH_OK;
}

}  // namespace host
}  // namespace isph
