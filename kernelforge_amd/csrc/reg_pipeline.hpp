// reg_pipeline.hpp -- products whose operands go from global memory straight into
// registers, one step ahead of the MFMAs (local_direct.hip, local_matvec.hip).
#pragma once

#include "kf_common.hpp"

namespace kf {

// n steps through two register buffers: load(buf, step) fills one while mul(buf) works on
// the other.  No load in the loop is conditional: behind a branch the compiler cannot tell
// how many loads are in flight and waits for all of them before the first product (the
// weighted sum of a 100 x 1,000 matvec 586 us instead of 507).
template <class Load, class Mul>
__device__ __forceinline__ void reg_pipeline(int n, Load load, Mul mul) {
    if (n <= 0) return;
    load(0, 0);
    int i = 0;
    for (; i + 2 < n; i += 2) {
        load(1, i + 1);
        mul(0);
        load(0, i + 2);
        mul(1);
    }
    if (i + 1 < n) {
        load(1, i + 1);
        mul(0);
        mul(1);
    } else {
        mul(0);
    }
}

}  // namespace kf
