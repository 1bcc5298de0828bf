// fri_fold.h -- one element of the FRI arity-2 fold (fri.hip has its semantics).
#pragma once
#include "kernels.h"
#include "field.h"

namespace pg {
// out[i] = (v[2i] + v[2i+1]) / 2 + beta / (2 x_i) (v[2i] - v[2i+1]) + add[i] for
// ext4 vectors, i < 2^log_n_out; tw: w_n^e for n = 2^(log_n_out + 1); add may be
// null and, a caller's vector, at any word.
template <class F>
__device__ __forceinline__ u32x4 fri_fold_at(gcptr v, uint64_t i, int log_n_out, const uint32_t (&beta)[4], gcptr tw,
                                             gcptr add) {
    const u32x4 a4 = reinterpret_cast<const GLOBAL u32x4*>(v)[2 * i], b4 = reinterpret_cast<const GLOBAL u32x4*>(v)[2 * i + 1];
    const Ext4 a = {{a4.x, a4.y, a4.z, a4.w}}, b = {{b4.x, b4.y, b4.z, b4.w}};
    const uint32_t mask = (2u << log_n_out) - 1u;
    const uint32_t r = log_n_out == 0 ? 0u : (__brev((uint32_t)i) >> (32 - log_n_out));
    const uint32_t x_inv = tw[(0u - r) & mask];  // w_n^{-rev(i)}
    Ext4 s = eadd<F>(a, b);
#pragma unroll
    for (int k = 0; k < 4; k++) s.c[k] = fhalve<F>(s.c[k]);
    const Ext4 d = escale<F>(esub<F>(a, b), x_inv);
    Ext4 half_beta;
#pragma unroll
    for (int k = 0; k < 4; k++) half_beta.c[k] = fhalve<F>(beta[k]);
    Ext4 o = eadd<F>(s, emul<F>(d, half_beta));
    if (add) {
        const u32x4 w = reinterpret_cast<const GLOBAL u32x4u*>(add)[i];
        o = eadd<F>(o, Ext4{{w.x, w.y, w.z, w.w}});
    }
    return u32x4{o.c[0], o.c[1], o.c[2], o.c[3]};
}
}  // namespace pg
