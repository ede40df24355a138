// f32 values as sums of three bf16 values, the operands of exact products on
// the bf16 matrix cores: hi = rn(x), mid = rn(x - hi), lo = x - hi - mid.  Both
// differences are exact, and 24 significant bits are three times eight.  Below
// about 2^-110 lo falls under bf16's smallest subnormal and is lost in part: a
// linear whose inputs are all of that size is off by 1.2e-7 of the result at
// 2^-111, 3.7e-7 at 2^-114 and 6e-6 at 2^-118, against 1.0e-7 above.
#pragma once
#include "device_common.h"

namespace leafhip {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));

__device__ __forceinline__ void split8(const float (&f)[8], v8bf& hi, v8bf& mid, v8bf& lo) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const v2f v = v2f{f[2 * p], f[2 * p + 1]};
        const v2bf h = __builtin_convertvector(v, v2bf);
        const v2f r = v2f{v.x - (float)h.x, v.y - (float)h.y};
        const v2bf m = __builtin_convertvector(r, v2bf);
        const v2f s = v2f{r.x - (float)m.x, r.y - (float)m.y};
        const v2bf l = __builtin_convertvector(s, v2bf);
        hi[2 * p] = h.x; hi[2 * p + 1] = h.y;
        mid[2 * p] = m.x; mid[2 * p + 1] = m.y;
        lo[2 * p] = l.x; lo[2 * p + 1] = l.y;
    }
}

}  // namespace leafhip
