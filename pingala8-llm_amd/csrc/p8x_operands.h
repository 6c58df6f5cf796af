// p8x_operands.h -- device memory of the prompt GEMM's decoded fp16 weight operands. A call that gets none runs the
// kernel that decodes as it multiplies (k_mm): the same bits, slower. Templated on the device calls (HipApi in
// p8x_gemm.hip), so that the rules can be tested without a GPU.
#pragma once
#include <cstddef>

namespace p8x {

// A buffer of at least `need` bytes in *p (*have: its size), or false with the old one kept: running out of memory is no
// error here, and leaves none behind for the next launch's check. The new buffer is allocated before the old one is
// given back; the device is synchronized before that, since calls in flight may still use it.
template <class Api>
bool try_grow(void **p, size_t *have, size_t need) {
    if (*have >= need) return true;
    void *q = nullptr;
    if (!Api::alloc(&q, need)) {
        Api::clear_error();
        return false;
    }
    if (*p) {
        if (!Api::synchronize()) {
            Api::clear_error();
            Api::release(q);
            return false;
        }
        Api::release(*p);
    }
    *p = q;
    *have = need;
    return true;
}

}  // namespace p8x
