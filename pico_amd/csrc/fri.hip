// fri.hip -- FRI arity-2 fold, and the element-wise helpers (representation conversion, seeded synthetic inputs).
//
// Fold semantics (p3 fold_even_odd; pinned in-tree by the query check at
// vm/src/compiler/recursion/circuit/fri.rs:288-387): the committed vector is
// in bit-reversed evaluation order over <w_n>, so v[2i] and v[2i+1] are the
// values at x_i and -x_i with x_i = w_n^{rev_{log(n/2)}(i)}; the folded value
// is the line through both points evaluated at beta:
//   out[i] = (v[2i] + v[2i+1]) / 2 + beta/2 * (v[2i] - v[2i+1]) * x_i^{-1}.
#include "kernels.h"
#include "field.h"
#include "fri_fold.h"

namespace pg {

// beta is read from device memory when `beta` is given (in the commit phase the
// tree's last launch has just sampled it, and no host round trip stands between
// two rounds), else it is `host_beta`.
template <class F>
__global__ void __launch_bounds__(256) fri_fold_kernel(const uint32_t* __restrict__ v, uint64_t n_out,
                                                       const uint32_t* __restrict__ beta, Ext4 host_beta,
                                                       const uint32_t* __restrict__ tw, int log_n_out, const uint32_t* __restrict__ add,
                                                       uint32_t* __restrict__ out) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_out) return;
    uint32_t bt[4];
#pragma unroll
    for (int k = 0; k < 4; k++) bt[k] = beta ? beta[k] : host_beta.c[k];
    reinterpret_cast<GLOBAL u32x4*>((gptr)out)[i] = fri_fold_at<F>((gcptr)v, i, log_n_out, bt, (gcptr)tw, (gcptr)add);
}

template <class F>
__global__ void convert_kernel(uint32_t* data, uint64_t n, int to) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) data[i] = to ? to_monty<F>(data[i]) : from_monty<F>(data[i]);
}

// Element i of seeded stream `seed`: the first of SplitMix64 outputs
// 4i .. 4i+3 of that seed whose top 31 bits are below p, else the last
// candidate reduced mod p.  Output j of SplitMix64 is its finaliser applied to
// seed + (j + 1) * golden, so elements are drawn independently in parallel.
__device__ __forceinline__ uint64_t splitmix_out(uint64_t seed, uint64_t j) {
    uint64_t z = seed + (j + 1) * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

template <class F>
__global__ void fill_random_kernel(uint64_t seed, uint32_t* out, uint64_t n, int monty) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint32_t x = 0;
    bool ok = false;
    for (int t = 0; t < 4 && !ok; t++) {
        x = (uint32_t)(splitmix_out(seed, 4 * i + t) >> 33);
        ok = x < F::P;
    }
    if (!ok) x %= F::P;
    out[i] = monty ? to_monty<F>(x) : x;
}

static unsigned blocks(uint64_t n) { return (unsigned)((n + 255) / 256); }

hipError_t launch_fri_fold(int field, const uint32_t* v, size_t n_out, const uint32_t* beta, const uint32_t* host_beta,
                           const uint32_t* tw, const uint32_t* add, uint32_t* out, hipStream_t stream) {
    if (n_out == 0) return hipSuccess;
    Ext4 hb{{0, 0, 0, 0}};
    for (int k = 0; k < 4 && host_beta; k++) hb.c[k] = host_beta[k];
    int log_n_out = 0;
    while ((1ull << log_n_out) < n_out) log_n_out++;
    if (field == FIELD_KOALABEAR)
        fri_fold_kernel<KoalaBear><<<blocks(n_out), 256, 0, stream>>>(v, n_out, beta, hb, tw, log_n_out, add, out);
    else
        fri_fold_kernel<BabyBear><<<blocks(n_out), 256, 0, stream>>>(v, n_out, beta, hb, tw, log_n_out, add, out);
    return hipGetLastError();
}

// dst row r (r < nrows) = src row rev_q(r0 + r), w words per row: a run of
// natural-order rows of a matrix stored in bit-reversed row order.  One
// thread per word, adjacent threads on adjacent columns (coalesced).
__global__ void rows_bitrev_kernel(const uint32_t* __restrict__ src, uint64_t ld, uint32_t w, int q, uint64_t r0,
                                   uint64_t nrows, uint32_t* __restrict__ dst) {
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nrows * w) return;
    const uint64_t r = t / w, c = t % w;
    const uint64_t j = r0 + r;
    const uint64_t sr = q ? (uint64_t)(__brevll(j) >> (64 - q)) : 0;
    dst[t] = ((gcptr)src)[sr * ld + c];
}

hipError_t launch_rows_bitrev(const uint32_t* src, uint64_t ld, uint32_t w, int q, uint64_t r0, uint64_t nrows,
                              uint32_t* dst, hipStream_t stream) {
    if (nrows == 0 || w == 0) return hipSuccess;
    rows_bitrev_kernel<<<blocks(nrows * w), 256, 0, stream>>>(src, ld, w, q, r0, nrows, dst);
    return hipGetLastError();
}

hipError_t launch_convert(int field, uint32_t* data, size_t n, int to_monty_, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    if (field == FIELD_KOALABEAR)
        convert_kernel<KoalaBear><<<blocks(n), 256, 0, stream>>>(data, n, to_monty_);
    else
        convert_kernel<BabyBear><<<blocks(n), 256, 0, stream>>>(data, n, to_monty_);
    return hipGetLastError();
}

hipError_t launch_fill_random(int field, uint64_t seed, uint32_t* out, size_t n, int monty,
                              hipStream_t stream) {
    if (n == 0) return hipSuccess;
    if (field == FIELD_KOALABEAR)
        fill_random_kernel<KoalaBear><<<blocks(n), 256, 0, stream>>>(seed, out, n, monty);
    else
        fill_random_kernel<BabyBear><<<blocks(n), 256, 0, stream>>>(seed, out, n, monty);
    return hipGetLastError();
}

}  // namespace pg
