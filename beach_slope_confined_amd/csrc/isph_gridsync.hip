// isph_gridsync.hip -- launching grids whose blocks wait for each other.
#include <algorithm>

#include "isph_gridsync.h"
#include "isph_host.h"

namespace isph {

__global__ void k_gs_clear(int n, gs_word* w, uint32_t* state) {
    const int i = blockIdx.x * BLOCK + threadIdx.x;
    if (i < n) w[i] = 0ull;
    if (i == 0) *state = 0;
}

// in place of a grid: what is left when its blocks have waited in vain
__global__ void k_gs_lose(uint32_t* err) { atomicOr(err, ERR_SYNC); }

namespace host {

int grid_launch(isph_ctx* c, const void* kern, int blocks, int threads, void** args, size_t lds,
                int parts, bool& ran) {
    ran = false;
    if (lds > 64 * 1024)
        HIPCHK(c, hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    const int n = gs_words(parts);
    k_gs_clear<<<nblk(n), BLOCK, 0, c->stream>>>(n, c->gs_words, c->err + 1);
    hipError_t e = hipSuccess;
    if (c->lose > 0) {
        c->lose -= 1;
        k_gs_lose<<<1, 1, 0, c->stream>>>(c->err);
    } else {
        e = hipLaunchCooperativeKernel(kern, dim3(blocks), dim3(threads), args, (unsigned)lds,
                                       c->stream);
    }
    auto lost = [&] {
        c->hold = c->hold_next;
        c->hold_next = std::min(2 * c->hold_next, HOLD_MOST);
        c->forms[ISPH_FORM_LOST] += 1;
    };
    if (e != hipSuccess) {
        // One process at a time holds a GPU's cooperative queue; a second one
        // is refused, and its contexts keep to the launched kernels meanwhile.
        (void)hipGetLastError();
        lost();
        return ISPH_OK;
    }
    uint32_t word[2] = {0, 0};
    HIPCHK(c, hipMemcpyAsync(word, c->err, sizeof(word), hipMemcpyDeviceToHost, c->stream));
    if (int rc = read_sc(c)) return rc;
    if (word[0] & ERR_SYNC) {
        // Blocks waited in vain: something else holds their CUs.  Unless one
        // has written its part back, the launched kernels carry on from the
        // state the launch began with.
        lost();
        if (int rc = clear_errors(c, ERR_SYNC)) return rc;
        if (word[1] & GS_WRITTEN) return fail(c, ISPH_E_HIP, "a resident solve lost a block");
        return ISPH_OK;
    }
    if (word[1] & GS_REFUSED) {
        c->forms[ISPH_FORM_REFUSED] += 1;
        return ISPH_OK;
    }
    c->hold_next = HOLD_FIRST;
    ran = true;
    return ISPH_OK;
}

}  // namespace host
}  // namespace isph
