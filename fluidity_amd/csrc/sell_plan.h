// The plan of a sliced ELL operand on the device, built there.
#pragma once

#include "flgpu_internal.h"
#include "krylov_common.h"

namespace flgpu {

struct SellPlan {
    int nsl = 0;          // slices (0: no plan)
    int64_t nslot = 0;
    bool use16 = false;   // column indices as int16 offsets
    DevBuf<int32_t> sptr, col32, rows, off;
    DevBuf<int16_t> col16;
    DevBuf<uint64_t> mask;
    DevBuf<int32_t> src;  // per slot: the entry of the value array it takes, -1 for padding
    void release() {
        nsl = 0;
        nslot = 0;
        sptr.release();
        col32.release();
        rows.release();
        off.release();
        col16.release();
        mask.release();
        src.release();
    }
};

// Plans the n-row CSR pattern (device arrays, 0-based, columns ascending in a
// row), its rows in order or sorted; vmap (or null): the value array's entry
// for each CSR entry.  Waits for the stream.  A pattern whose slots would not
// fit 32-bit indices gets no plan (nsl = 0).
int sell_build(hipStream_t s, int n, int64_t nnz, const int32_t* rowptr, const int32_t* col, const int32_t* vmap,
               bool sorted, SellPlan& p);

// The operand with values in slot order.
template <typename AV, typename CT>
inline SellOp<AV, CT> sell_op(const SellPlan& p, int n, const AV* val, const CT* col, const float* rs = nullptr) {
    return SellOp<AV, CT>{p.nsl, n, p.sptr.p, col, val, rs, p.rows.p, p.off.p, p.mask.p};
}

}  // namespace flgpu
