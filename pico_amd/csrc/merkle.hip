// merkle.hip -- Poseidon2 Merkle kernels for the mixed-height MMCS:
// leaf hashing (sponge over concatenated same-height rows), compress/inject
// layers and the opening gather.
//
// Semantics (p3 MerkleTreeMmcs, pinned in-tree by the inverse verify_batch at
// vm/src/compiler/recursion/circuit/fri.rs:389-436):
//   layer0[i] = H(concat of row i of every matrix of the tallest height)
//   next[i]   = C(prev[2i], prev[2i+1]); if matrices of height len(next)
//               exist: next[i] = C(next[i], H(concat of their row i))
//   H = PaddingFreeSponge<16, 8, 8> (overwrite mode, circuit/hash.rs:40-52)
//   C = TruncatedPermutation (circuit/hash.rs:89-94)
// The linear layers run on the matrix cores (poseidon2_mx.h).  Layers of more
// than SMALL_MAX_NODES rows or nodes take 64 states per wave, smaller ones 16:
// the grid deals groups of that many rows or nodes to waves.
#include <algorithm>

#include "kernels.h"
#include "poseidon2.h"
#include "poseidon2_mx.h"
#include "fri_fold.h"

namespace pg {

// ---- hashing on the matrix cores --------------------------------------------
// What bounds it: VALU issue, now of the S-boxes and the layer reductions.
// A wave's two tiles of 32 states share every table read from LDS (31 KB per
// workgroup, read once per permutation and wave).
constexpr int MX_WAVES = 4;  // waves per workgroup
constexpr int MX_THREADS = 64 * MX_WAVES;
// Three waves per SIMD (168 registers): at four (128) every kernel spills, at two
// the issue slots are not all filled (leaf hash of 2^21 x 256: 4.53 ms, 4.82 and
// 4.70).  At three a few spill 2 to 6 registers (the batched leaves for KoalaBear,
// the segment absorb and the injecting compress for BabyBear).
#define MX_KERNEL __global__ void __launch_bounds__(MX_THREADS) __attribute__((amdgpu_waves_per_eu(3, 3)))

// The lane's place in its wave: state 32 t + n of tile t, words 4 h + i of the
// rate and of the capacity.
struct MxLane {
    uint32_t n, h;
    __device__ __forceinline__ MxLane() : n(threadIdx.x & 31u), h((threadIdx.x & 63u) >> 5) {}
};
// index of the wave in the grid (uniform)
__device__ __forceinline__ uint64_t mx_wave() {
    return (uint64_t)blockIdx.x * MX_WAVES + (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
}
__device__ __forceinline__ mx4 mx_op(u32x4 v) { return __builtin_bit_cast(mx4, v ^ MX_BIAS); }
__device__ __forceinline__ mx4 mx_op_words(const uint32_t* st) { return mx_op(u32x4{st[0], st[1], st[2], st[3]}); }

// A cursor over the concatenation of one row of mats[0..n): the words
// 8 c + 4 h .. + 3 of chunk c for the wave's two tiles.  The cursor (k, j) is
// wave-uniform, so the matrix descriptors are read through the scalar cache.
struct MxRows {
    const MatRef* mats;
    int n, k;
    uint32_t j;
    __device__ __forceinline__ MxRows(const MatRef* m, int nm) : mats(m), n(nm), k(0), j(0) {}
    __device__ __forceinline__ void skip_ended() {
        while (j >= mats[k].width && k + 1 < n) {
            k++;
            j = 0;
        }
    }
    // cnt words of the chunk exist; the others read as word 0
    template <int T>
    __device__ __forceinline__ void chunk(u32x4 (&out)[T], const uint64_t (&row)[T], uint32_t cnt, uint32_t h) {
        skip_ended();
        if (cnt == 8 && j + 8 <= mats[k].width) {  // within one matrix
            const gcptr base = (gcptr)mats[k].data + (j + 4 * h);
#pragma unroll
            for (int t = 0; t < T; t++)
                out[t] = *reinterpret_cast<const GLOBAL u32x4u*>(base + row[t] * mats[k].stride);
            j += 8;
            return;
        }
        const uint32_t* p[8];
        uint64_t st[8];
#pragma unroll
        for (int w = 0; w < 8; w++) {
            if ((uint32_t)w < cnt) {
                skip_ended();
                p[w] = mats[k].data + j;
                st[w] = mats[k].stride;
                j++;
            } else {
                p[w] = p[0];
                st[w] = st[0];
            }
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const gcptr q = (gcptr)(h ? p[4 + i] : p[i]);
            const uint64_t ld = h ? st[4 + i] : st[i];
#pragma unroll
            for (int t = 0; t < T; t++) out[t][i] = q[row[t] * ld];
        }
    }
};

// Sponge state of 64 rows between permutations: `b`, the last S-boxes'
// outputs (the zero state: S-box outputs of zero); the state words themselves
// are formed only where a chunk is partial and at the end.
template <class F>
struct MxSponge {
    mx4 b[2][2];
    __device__ __forceinline__ MxSponge() {
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int s = 0; s < 2; s++) b[t][s] = mx_op(u32x4{0});
    }
    // Absorbs a whole chunk
    __device__ __forceinline__ void absorb8(const u32x4 (&in)[2], MxView<F>& v) {
        int x[2][8];
        v.fresh();
        const mx4 rate[2] = {mx_op(in[0]), mx_op(in[1])};
        mx_next<F>(x, rate, b, v);
        mx_rounds<F>(b, x, v);
    }
    // Absorbs one chunk: cnt of its 8 words overwrite the rate words.
    __device__ __forceinline__ void absorb(const u32x4 (&in)[2], uint32_t cnt, uint32_t h, MxView<F>& v) {
        const uint32_t each[2] = {cnt, cnt};
        absorb(in, cnt == 8, each, h, v);
    }
    // The same with a count per state: cnt[t] for the lane's state of tile t, 8
    // in all of them where `whole`.
    __device__ __forceinline__ void absorb(const u32x4 (&in)[2], bool whole, const uint32_t (&cnt)[2], uint32_t h,
                                           MxView<F>& v) {
        int x[2][8];
        v.fresh();
        if (whole) {
            const mx4 rate[2] = {mx_op(in[0]), mx_op(in[1])};
            mx_next<F>(x, rate, b, v);
        } else {
            uint32_t st[2][8];
            mx_last<F>(st, b, v);
            mx4 full[2][2];
#pragma unroll
            for (int t = 0; t < 2; t++) {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (4 * h + i < cnt[t]) st[t][i] = in[t][i];
                full[t][0] = mx_op_words(&st[t][0]);
                full[t][1] = mx_op_words(&st[t][4]);
            }
            mx_init<F>(x, full, v);
        }
        mx_rounds<F>(b, x, v);
    }
    // absorbs the concatenated rows; total > 0
    __device__ __forceinline__ void absorb_rows(MxRows src, const uint64_t (&row)[2], uint32_t total, uint32_t h,
                                                MxView<F>& v) {
        u32x4 next[2];
        src.chunk(next, row, total < 8u ? total : 8u, h);
        for (uint32_t off = 0; off < total; off += 8) {
            const u32x4 cur[2] = {next[0], next[1]};
            const uint32_t left = total - off;
            // the next chunk's words are in flight during the permutation
            if (left > 8) src.chunk(next, row, left - 8 < 8u ? left - 8 : 8u, h);
            absorb(cur, left < 8u ? left : 8u, h, v);
        }
    }
};

// Row addresses of the wave's group; rows past the end shadow the last one.
__device__ __forceinline__ void mx_group_rows(uint64_t (&row)[2], uint64_t group, uint64_t rows, const MxLane& l) {
#pragma unroll
    for (int t = 0; t < 2; t++) {
        const uint64_t r = 64 * group + 32 * t + l.n;
        row[t] = r < rows ? r : rows - 1;
    }
}
__device__ __forceinline__ void mx_store_digests(uint32_t* digests, uint64_t group, uint64_t rows, const MxLane& l,
                                                 const uint32_t (&st)[2][8]) {
#pragma unroll
    for (int t = 0; t < 2; t++) {
        const uint64_t r = 64 * group + 32 * t + l.n;
        if (r < rows)
            *reinterpret_cast<GLOBAL u32x4*>((gptr)digests + 8 * r + 4 * l.h) =
                u32x4{st[t][0], st[t][1], st[t][2], st[t][3]};
    }
}

// General leaf hash: any number of matrices, any widths.
template <class F>
MX_KERNEL leaf_hash_kernel(const MatRef* mats, int n, uint32_t total,
                                                               uint64_t rows, uint32_t* digests) {
    __shared__ MxTable<F> tab;
    mx_load<F>(tab);
    const uint64_t group = mx_wave();
    if (64 * group >= rows) return;
    MxView<F> v(tab);
    const MxLane l;
    uint32_t st[2][8] = {};
    if (total) {
        uint64_t row[2];
        mx_group_rows(row, group, rows, l);
        MxSponge<F> sp;
        sp.absorb_rows(MxRows(mats, n), row, total, l.h, v);
        mx_last<F>(st, sp.b, v);
    }
    mx_store_digests(digests, group, rows, l, st);
}

// One matrix whose width is a multiple of 8 and whose rows are 16-byte
// aligned: every sponge chunk is one 16-byte load per lane and tile.
template <class F>
MX_KERNEL leaf_hash_w8_kernel(const uint32_t* data, uint64_t stride,
                                                                  uint32_t chunks, uint64_t rows,
                                                                  uint32_t* digests) {
    __shared__ MxTable<F> tab;
    mx_load<F>(tab);
    const uint64_t group = mx_wave();
    if (64 * group >= rows) return;
    MxView<F> v(tab);
    const MxLane l;
    uint64_t row[2];
    mx_group_rows(row, group, rows, l);
    const GLOBAL u32x4* rp[2];
#pragma unroll
    for (int t = 0; t < 2; t++) rp[t] = reinterpret_cast<const GLOBAL u32x4*>((gcptr)data + row[t] * stride + 4 * l.h);
    u32x4 next[2] = {rp[0][0], rp[1][0]};
    MxSponge<F> sp;
    for (uint32_t c = 0; c < chunks; c++) {
        const u32x4 cur[2] = {next[0], next[1]};
        const uint32_t cn = c + 1 < chunks ? c + 1 : c;
        next[0] = rp[0][2 * cn];  // in flight during the permutation
        next[1] = rp[1][2 * cn];
        sp.absorb8(cur, v);
    }
    uint32_t st[2][8];
    mx_last<F>(st, sp.b, v);
    mx_store_digests(digests, group, rows, l, st);
}

// One segment of the leaf sponge: columns [0, width) of a matrix view are
// the next `width` inputs of every row's sponge, whose state lives in
// `state` (16 words per row) between segments.  pos0 = inputs already
// written into the pending chunk (the running input count mod 8): in
// overwrite mode a chunk's inputs go to st[0..8) and the permutation runs
// when it is full, so st itself carries a partial chunk across segments.
// first: start from the zero state; last: run the final partial chunk's
// permutation (if any) and write the digest instead of the state.  The
// segments of a row, concatenated, give the same digest as one pass of
// absorb_rows over the whole row.
template <class F>
MX_KERNEL absorb_segment_kernel(const uint32_t* data, uint64_t stride,
                                                                    uint32_t width, uint32_t pos0, int first,
                                                                    int last, uint64_t rows, uint32_t* state,
                                                                    uint32_t* digests) {
    __shared__ MxTable<F> tab;
    mx_load<F>(tab);
    const uint64_t group = mx_wave();
    if (64 * group >= rows) return;
    MxView<F> v(tab);
    const MxLane l;
    uint64_t row[2];
    mx_group_rows(row, group, rows, l);
    // st holds the state while a chunk is pending, b after a permutation
    uint32_t st[2][8] = {};
    if (!first) {
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int s = 0; s < 2; s++) {
                const u32x4 w = *reinterpret_cast<const GLOBAL u32x4*>((gcptr)state + 16 * row[t] + 8 * s + 4 * l.h);
#pragma unroll
                for (int i = 0; i < 4; i++) st[t][4 * s + i] = w[i];
            }
    }
    mx4 b[2][2];
    bool words = true;  // st is valid
    uint32_t pos = pos0, e = 0;
    while (e < width || (last && pos > 0)) {  // pos, e and words are the same in every lane
        const uint32_t take = width - e < 8 - pos ? width - e : 8 - pos;
        int x[2][8];
        v.fresh();
        if (!words && take == 8) {
            mx4 rate[2];
#pragma unroll
            for (int t = 0; t < 2; t++)
                rate[t] = mx_op(*reinterpret_cast<const GLOBAL u32x4u*>((gcptr)data + row[t] * stride + e + 4 * l.h));
            mx_next<F>(x, rate, b, v);
            e += 8;
        } else {
            if (!words) mx_last<F>(st, b, v);
            words = true;
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const uint32_t w = 4 * l.h + i;
                    if (w >= pos && w < pos + take) st[t][i] = ((gcptr)data)[row[t] * stride + e + w - pos];
                }
            e += take;
            pos += take;
            if (pos < 8 && !(last && e >= width)) break;  // pending: the next segment fills it
            mx4 full[2][2];
#pragma unroll
            for (int t = 0; t < 2; t++) {
                full[t][0] = mx_op_words(&st[t][0]);
                full[t][1] = mx_op_words(&st[t][4]);
            }
            mx_init<F>(x, full, v);
            pos = 0;
        }
        mx_rounds<F>(b, x, v);
        words = false;
    }
    if (!words) mx_last<F>(st, b, v);
    if (last) {
        mx_store_digests(digests, group, rows, l, st);
        return;
    }
#pragma unroll
    for (int t = 0; t < 2; t++) {
        const uint64_t r = 64 * group + 32 * t + l.n;
        if (r >= rows) continue;
#pragma unroll
        for (int s = 0; s < 2; s++)
            *reinterpret_cast<GLOBAL u32x4*>((gptr)state + 16 * r + 8 * s + 4 * l.h) =
                u32x4{st[t][4 * s], st[t][4 * s + 1], st[t][4 * s + 2], st[t][4 * s + 3]};
    }
}

// next[i] = C(prev[2i], prev[2i+1]), then with INJ: C(next[i], H(rows i of inj))
template <class F, bool INJ>
MX_KERNEL compress_kernel(const uint32_t* prev, uint32_t* next,
                                                              uint64_t n_out, const MatRef* inj,
                                                              int n_inj, uint32_t inj_width) {
    __shared__ MxTable<F> tab;
    mx_load<F>(tab);
    MxView<F> v(tab);
    const MxLane l;
    const uint64_t stride = (uint64_t)gridDim.x * MX_WAVES;
    for (uint64_t group = mx_wave(); 64 * group < n_out; group += stride) {
        uint64_t row[2];
        mx_group_rows(row, group, n_out, l);
        u32x4 hash[2] = {u32x4{0}, u32x4{0}};
        MxSponge<F> sp;
        if constexpr (INJ) {
            if (inj_width) {
                uint32_t st[2][8];
                sp.absorb_rows(MxRows(inj, n_inj), row, inj_width, l.h, v);
                mx_last<F>(st, sp.b, v);
#pragma unroll
                for (int t = 0; t < 2; t++) hash[t] = u32x4{st[t][0], st[t][1], st[t][2], st[t][3]};
            }
        }
        uint32_t st[2][8];
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int s = 0; s < 2; s++) {
                const u32x4 w = *reinterpret_cast<const GLOBAL u32x4*>((gcptr)prev + 16 * row[t] + 8 * s + 4 * l.h);
#pragma unroll
                for (int i = 0; i < 4; i++) st[t][4 * s + i] = w[i];
            }
#pragma clang loop unroll(disable)
        for (int k = 0; k < (INJ ? 2 : 1); k++) {
            if (k) {
#pragma unroll
                for (int t = 0; t < 2; t++)
#pragma unroll
                    for (int i = 0; i < 4; i++) st[t][4 + i] = hash[t][i];
            }
            mx4 full[2][2];
#pragma unroll
            for (int t = 0; t < 2; t++) {
                full[t][0] = mx_op_words(&st[t][0]);
                full[t][1] = mx_op_words(&st[t][4]);
            }
            int x[2][8];
            v.fresh();
            mx_init<F>(x, full, v);
            mx_rounds<F>(sp.b, x, v);
            mx_last<F>(st, sp.b, v);
        }
        mx_store_digests(next, group, n_out, l, st);
    }
}

// The same with the injected rows already hashed: C(C(prev[2i], prev[2i+1]), inj[i])
template <class F>
MX_KERNEL compress_digest_kernel(const uint32_t* prev, const uint32_t* inj,
                                                                     uint32_t* next, uint64_t n_out) {
    __shared__ MxTable<F> tab;
    mx_load<F>(tab);
    MxView<F> v(tab);
    const MxLane l;
    const uint64_t stride = (uint64_t)gridDim.x * MX_WAVES;
    for (uint64_t group = mx_wave(); 64 * group < n_out; group += stride) {
        uint64_t row[2];
        mx_group_rows(row, group, n_out, l);
        u32x4 hash[2];
        uint32_t st[2][8];
#pragma unroll
        for (int t = 0; t < 2; t++) {
            hash[t] = *reinterpret_cast<const GLOBAL u32x4*>((gcptr)inj + 8 * row[t] + 4 * l.h);
#pragma unroll
            for (int s = 0; s < 2; s++) {
                const u32x4 w = *reinterpret_cast<const GLOBAL u32x4*>((gcptr)prev + 16 * row[t] + 8 * s + 4 * l.h);
#pragma unroll
                for (int i = 0; i < 4; i++) st[t][4 * s + i] = w[i];
            }
        }
#pragma clang loop unroll(disable)
        for (int k = 0; k < 2; k++) {
            if (k) {
#pragma unroll
                for (int t = 0; t < 2; t++)
#pragma unroll
                    for (int i = 0; i < 4; i++) st[t][4 + i] = hash[t][i];
            }
            mx4 full[2][2], b[2][2];
#pragma unroll
            for (int t = 0; t < 2; t++) {
                full[t][0] = mx_op_words(&st[t][0]);
                full[t][1] = mx_op_words(&st[t][4]);
            }
            int x[2][8];
            v.fresh();
            mx_init<F>(x, full, v);
            mx_rounds<F>(b, x, v);
            mx_last<F>(st, b, v);
        }
        mx_store_digests(next, group, n_out, l, st);
    }
}

// ---- small layers: 16 states per wave ------------------------------------------
// A layer costs a permutation's latency however few nodes it has: 2.2 us this
// way, 7 us with 64 states per wave.  Up to SMALL_MAX_NODES (2^15: two waves
// per SIMD) it is the faster form: one layer of 2^15 nodes 6.7 against 8.1 us,
// two-chunk leaves of 2^15 rows 10.8 against 14.8 us; at 2^16 the 64-state form
// still takes one wave per SIMD (8.8 us) and this one four.
constexpr int S_WAVES = 4;
constexpr int S_THREADS = 64 * S_WAVES;
#define MX16_KERNEL __global__ void __launch_bounds__(S_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2)))
// the lane's state in its wave and its quarter of the words
struct Mx16Lane {
    uint32_t n, q;
    __device__ __forceinline__ Mx16Lane() : n(threadIdx.x & 15u), q((threadIdx.x & 63u) >> 4) {}
};
__device__ __forceinline__ uint32_t mx16_wave() { return (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); }

// Digest (lane groups 0 and 1) of row `row` of the concatenated matrices; the
// whole wave calls it.
template <class F>
__device__ __forceinline__ u32x4 mx16_hash_rows(const Mx16<F>& P, MxRows src, uint64_t row, uint32_t total, uint32_t q) {
    const uint64_t rows1[1] = {row};
    const uint32_t h = q & 1u;
    u32x4 next[1] = {u32x4{0}};
    if (total) src.chunk<1>(next, rows1, total < 8u ? total : 8u, h);
    mx4 st = mx4{0};
#pragma clang loop unroll(disable)
    for (uint32_t off = 0; off < total; off += 8) {
        const u32x4 cur = next[0];
        const uint32_t left = total - off;
        if (left > 8) src.chunk<1>(next, rows1, left - 8 < 8u ? left - 8 : 8u, h);  // in flight
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (4 * q + i < (left < 8u ? left : 8u)) st[i] = (int)cur[i];
        st = P.permute(Mx16<F>::op(st));
    }
    return mx16_words<F>(st);
}

template <class F>
MX16_KERNEL leaf_hash_small_kernel(const MatRef* mats, int n, uint32_t total, uint64_t rows, uint32_t* digests) {
    const Mx16<F> P;
    const Mx16Lane l;
    const uint64_t r = ((uint64_t)blockIdx.x * S_WAVES + mx16_wave()) * 16 + l.n;
    const u32x4 d = mx16_hash_rows<F>(P, MxRows(mats, n), r < rows ? r : rows - 1, total, l.q);
    if (r < rows && l.q < 2) *reinterpret_cast<GLOBAL u32x4*>((gptr)digests + 8 * r + 4 * l.q) = d;
}

// next[i] = C(C(prev[2i], prev[2i+1]), x_i): x_i the hash of rows i of inj, or
// inj_digests[i] when that is given
template <class F>
MX16_KERNEL compress_small_kernel(const uint32_t* prev, uint32_t* next, uint64_t n_out, const MatRef* inj, int n_inj,
                                  uint32_t inj_width, const uint32_t* inj_digests) {
    const Mx16<F> P;
    const Mx16Lane l;
    const uint64_t r = ((uint64_t)blockIdx.x * S_WAVES + mx16_wave()) * 16 + l.n;
    const uint64_t rr = r < n_out ? r : n_out - 1;
    u32x4 d;  // group q: words 4 (q & 1) .. of x_i
    if (inj_digests) {
        d = *reinterpret_cast<const GLOBAL u32x4*>((gcptr)inj_digests + 8 * rr + 4 * (l.q & 1u));
    } else {
        d = mx16_hash_rows<F>(P, MxRows(inj, n_inj), rr, inj_width, l.q);
#pragma unroll
        for (int i = 0; i < 4; i++)  // groups 2 and 3 read groups 0 and 1
            d[i] = __builtin_amdgcn_permlane32_swap(d[i], d[i], false, false)[0];
    }
    const u32x4 w = *reinterpret_cast<const GLOBAL u32x4*>((gcptr)prev + 16 * rr + 4 * l.q);
    mx4 st = __builtin_bit_cast(mx4, w);
#pragma clang loop unroll(disable)
    for (int k = 0; k < 2; k++) {
        if (k && l.q >= 2) st = __builtin_bit_cast(mx4, d);
        st = P.permute(Mx16<F>::op(st));
    }
    if (r < n_out && l.q < 2) *reinterpret_cast<GLOBAL u32x4*>((gptr)next + 8 * r + 4 * l.q) = mx16_words<F>(st);
}

// Several layers of a tree in one launch.  The first layer's n0 nodes are
// C(in[2i], in[2i+1]) or, with TREE_ROWS, the hashes of n0 rows of one matrix (a
// launch and the wait for a table of matrix descriptors less: commit of 2^8 x
// 13, 512 leaves, 78.7 -> 74.4 us) or, with TREE_FOLDED, of the pairs of a FRI
// vector folded here (a launch of 4.5 us less a round; commit phase of 2^18 with
// an injected 2^15: 694 -> 651 us); layers n0, n0/2, ... follow each other at `out`,
// as a tree stores them.  A workgroup computes the `layers` layers
// over its 2^log_per nodes of the first one: their children pass through LDS,
// so a layer costs one permutation's latency instead of a launch (4.3 us and
// the gap before it).
constexpr int TREE_MAX_PER = 128;  // first-layer nodes of a workgroup

// The duplex challenger (vm/src/compiler/recursion/circuit/challenger.rs:
// 89-175) observes 8 words and samples an ext4 element: the wave's 16 columns
// all hold the one state.  `root` and `pend` (16 words) are in LDS.  With k < 8
// inputs pending, the 8 words fill one duplexing and leave k for the one that
// sampling makes; the samples are output words 7, 6, 5, 4.
template <class F>
__device__ __forceinline__ void challenge_root(const Mx16<F>& P, const Mx16Lane& l, const TreeChallenge& ch,
                                               const uint32_t* root, uint32_t* pend) {
    const gptr st = (gptr)ch.state + 1, input = (gptr)ch.state + 17, n_input = (gptr)ch.state + 25,
               output = (gptr)ch.state + 26, n_output = (gptr)ch.state + 34;
    const uint32_t t = threadIdx.x, k = (uint32_t)__builtin_amdgcn_readfirstlane((int)*n_input);
    if (t < 8) {
        ((gptr)ch.root)[t] = root[t];
        if (t < k) pend[t] = input[t];
        pend[k + t] = root[t];
    }
    __threadfence_block();
    u32x4 w;
#pragma unroll
    for (int i = 0; i < 4; i++) w[i] = l.q < 2 ? pend[4 * l.q + i] : st[4 * l.q + i];
    w = mx16_words<F>(P.permute(Mx16<F>::op(__builtin_bit_cast(mx4, w))));
    if (k) {
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (4 * l.q + i < k) w[i] = pend[8 + 4 * l.q + i];
        w = mx16_words<F>(P.permute(Mx16<F>::op(__builtin_bit_cast(mx4, w))));
    }
    if (l.n == 0) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            st[4 * l.q + i] = w[i];
            if (l.q < 2) output[4 * l.q + i] = w[i];
            if (l.q == 1) ((gptr)ch.beta)[3 - i] = w[i];
        }
    }
    if (t < 8) input[t] = pend[t < k ? 8 + t : t];
    if (t == 0) {
        *n_input = 0;
        *n_output = 4;
    }
}

// Digest (lane groups 0 and 1) of one row of one matrix; the whole wave calls it.
template <class F>
__device__ __forceinline__ u32x4 mx16_hash_row(const Mx16<F>& P, gcptr row, uint32_t width, uint32_t q) {
    auto chunk = [&](uint32_t off) {  // words off + 4 (q & 1) ..; past the row: its last word
        const uint32_t j = off + 4 * (q & 1u);
        u32x4 v;
        if (off + 8 <= width) {
            v = *reinterpret_cast<const GLOBAL u32x4u*>(row + j);
        } else {
#pragma unroll
            for (uint32_t i = 0; i < 4; i++) v[i] = row[j + i < width ? j + i : width - 1];
        }
        return v;
    };
    u32x4 next = chunk(0);
    mx4 st = mx4{0};
#pragma clang loop unroll(disable)
    for (uint32_t off = 0; off < width; off += 8) {
        const u32x4 cur = next;
        const uint32_t left = width - off;
        if (left > 8) next = chunk(off + 8);  // in flight
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (4 * q + i < (left < 8u ? left : 8u)) st[i] = (int)cur[i];
        st = P.permute(Mx16<F>::op(st));
    }
    return mx16_words<F>(st);
}

// The job whose range of the prefix array (njobs + 1 entries) holds i
__device__ __forceinline__ int find_job(const uint64_t* __restrict__ prefix, int njobs, uint64_t i) {
    int lo = 0, hi = njobs;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (prefix[mid] <= i) lo = mid; else hi = mid;
    }
    return lo;
}

// What the first layer hashes.  TREE_JOBS: the nodes of one of several trees: `in`
// is the table of n0 jobs and `stride` the address of the prefix array over their
// workgroups (arguments of their own cost the other forms 1%: a cache line more).
enum { TREE_NODES, TREE_ROWS, TREE_FOLDED, TREE_JOBS };
template <class F, int FIRST>
MX16_KERNEL tree_layers_kernel(const uint32_t* in, uint64_t stride, uint32_t width, uint64_t n0, int log_per, int layers,
                               uint32_t* out, TreeChallenge ch, TreeFold fold) {
    __shared__ u32x4 buf[2][2 * TREE_MAX_PER];
    uint32_t block = blockIdx.x;  // of the tree's first layer
    if constexpr (FIRST == TREE_JOBS) {
        const uint64_t* const prefix = reinterpret_cast<const uint64_t*>(stride);
        const int j = __builtin_amdgcn_readfirstlane(find_job(prefix, (int)n0, block));
        const TreeJob* const jb = reinterpret_cast<const TreeJob*>(in) + j;
        block -= (uint32_t)prefix[j];
        in = jb->in;
        out = jb->out;
        n0 = jb->n0;
        log_per = (int)jb->log_per;
        layers = (int)jb->layers;
    }
    if constexpr (FIRST == TREE_FOLDED) {  // before the hash tables fill the registers
        uint32_t beta[4];
#pragma unroll
        for (int k = 0; k < 4; k++) beta[k] = ((gcptr)fold.beta)[k];
        const int log_n_out = 64 - __builtin_clzll(n0);  // of 2 n0 elements
        const uint32_t cnt = 2u << log_per;
        for (uint32_t t = threadIdx.x; t < cnt; t += blockDim.x) {
            const uint64_t i = (uint64_t)block * cnt + t;
            const u32x4 o = fri_fold_at<F>((gcptr)fold.prev, i, log_n_out, beta, (gcptr)fold.tw, (gcptr)fold.add);
            reinterpret_cast<GLOBAL u32x4*>((gptr)fold.out)[i] = o;
            buf[1][t] = o;
        }
        __syncthreads();
    }
    const Mx16<F> P;
    const Mx16Lane l;
    const uint32_t wave = mx16_wave(), waves = blockDim.x >> 6;
    gptr layer = (gptr)out;
    for (int i = 0; i < layers; i++) {
        const uint32_t cnt = (1u << log_per) >> i;
        const uint64_t base = (uint64_t)block * cnt;
        for (uint32_t g = wave; 16 * g < cnt; g += waves) {  // the wave's group of 16 nodes
            const uint32_t nd = 16 * g + l.n, nr = nd < cnt ? nd : cnt - 1;
            u32x4 w;
            if (FIRST == TREE_ROWS && i == 0) {
                w = mx16_hash_row<F>(P, (gcptr)in + (base + nr) * stride, width, l.q);
            } else {
                if (i > 0)
                    w = buf[(i - 1) & 1][4 * nr + l.q];
                else if constexpr (FIRST == TREE_FOLDED)
                    w = l.q < 2 ? buf[1][2 * nr + l.q] : u32x4{0};
                else
                    w = *reinterpret_cast<const GLOBAL u32x4*>((gcptr)in + 16 * (base + nr) + 4 * l.q);
                w = mx16_words<F>(P.permute(Mx16<F>::op(__builtin_bit_cast(mx4, w))));
            }
            if (l.q < 2 && nd < cnt) {
                buf[i & 1][2 * nd + l.q] = w;
                *reinterpret_cast<GLOBAL u32x4*>(layer + 8 * (base + nd) + 4 * l.q) = w;
            }
        }
        __syncthreads();
        layer += 8 * (n0 >> i);
    }
    if (ch.state && wave == 0) {  // one workgroup: the last layer is the root
        __shared__ uint32_t pend[16];
        challenge_root<F>(P, l, ch, reinterpret_cast<const uint32_t*>(buf[(layers - 1) & 1]), pend);
    }
}

__global__ void open_gather_kernel(const MatRef* mats, const uint32_t* shift,
                                   const uint32_t* col_off, int n_mats, uint32_t total_width,
                                   const uint32_t* digests, const uint64_t* layer_off, int log_h,
                                   const uint64_t* idx, uint32_t* rows_out, uint32_t* paths_out) {
    const int q = blockIdx.x;
    const uint64_t index = idx[q];
    for (int k = 0; k < n_mats; k++) {
        const uint64_t r = index >> shift[k];
        const MatRef m = mats[k];
        uint32_t* dst = rows_out + (uint64_t)q * total_width + col_off[k];
        for (uint32_t c = threadIdx.x; c < m.width; c += blockDim.x) dst[c] = m.data[r * m.stride + c];
    }
    for (int t = threadIdx.x; t < log_h * 8; t += blockDim.x) {
        const int j = t >> 3, e = t & 7;
        const uint64_t sib = (index >> j) ^ 1u;
        paths_out[((uint64_t)q * log_h + j) * 8 + e] = digests[(layer_off[j] + sib) * 8 + e];
    }
}

__global__ void fri_open_kernel(const FriOpenRound* rounds, const uint64_t* idx, uint32_t path_words, uint32_t* siblings,
                                uint32_t* paths) {
    const uint32_t q = blockIdx.x, r = blockIdx.y;
    const FriOpenRound rd = rounds[r];
    const uint64_t i = idx[q] >> r, leaf = i >> 1, H = 1ull << rd.log_h;
    if (threadIdx.x < 4) siblings[((uint64_t)q * gridDim.y + r) * 4 + threadIdx.x] = rd.vec[4 * (i ^ 1u) + threadIdx.x];
    for (uint32_t t = threadIdx.x; t < rd.log_h * 8; t += blockDim.x) {
        const uint32_t j = t >> 3;
        const uint64_t off = 2 * (H - (H >> j));  // layer j's first digest
        paths[(uint64_t)q * path_words + rd.path_off + t] = rd.digests[(off + ((leaf >> j) ^ 1u)) * 8 + (t & 7)];
    }
}

hipError_t launch_fri_open(const FriOpenRound* rounds, int nrounds, const uint64_t* idx, int nq, uint32_t path_words,
                           uint32_t* siblings, uint32_t* paths, hipStream_t stream) {
    if (nq == 0 || nrounds == 0) return hipSuccess;
    fri_open_kernel<<<dim3((unsigned)nq, (unsigned)nrounds), 128, 0, stream>>>(rounds, idx, path_words, siblings, paths);
    return hipGetLastError();
}

// ---- batched single-matrix commits --------------------------------------
// Leaf layer of many jobs: wave -> (job, group of 64 rows); rows of any width.
// A permutation takes a wave the same time with one row as with 64, so matrices
// of fewer than 64 rows share waves (PACKS): 4096 of 16 rows x 50 hash in 65 us,
// with a wave each in 143 us (one row per lane without matrix instructions: 74).
// A batch without such matrices takes the form without packs, whose widths are
// the same in every lane (64 jobs of 2^11 rows and more: 92.0 ms, 92.7 with packs).
template <class F, bool PACKS>
MX_KERNEL leaf_hash_batch_kernel(const LeafJob* __restrict__ jobs, const uint64_t* __restrict__ prefix, int njobs,
                                 uint64_t total, const LeafRow* __restrict__ pack_rows) {
    __shared__ MxTable<F> tab;
    mx_load<F>(tab);
    const uint64_t wave = mx_wave();
    if (wave >= total) return;
    const int j = __builtin_amdgcn_readfirstlane(find_job(prefix, njobs, wave));
    const LeafJob* jb = jobs + j;
    const uint64_t group = wave - prefix[j];
    MxView<F> v(tab);
    const MxLane l;
    const uint32_t widest = jb->width;
    gcptr rp[2];
    uint32_t width[2] = {widest, widest};
    bool pack = false;
    if constexpr (PACKS) pack = jb->pack != LeafJob::NO_PACK;
    if (pack) {
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const LeafRow* const r = pack_rows + jb->pack + 32 * t + l.n;
            rp[t] = (gcptr)r->src + 4 * l.h;
            width[t] = r->width;
        }
    } else {
        uint64_t row[2];
        mx_group_rows(row, group, jb->rows, l);
#pragma unroll
        for (int t = 0; t < 2; t++) rp[t] = (gcptr)jb->data + row[t] * jb->stride + 4 * l.h;
    }
    const bool whole = pack ? jb->whole != 0 : widest % 8 == 0;
    MxSponge<F> sp;
    auto load = [&](uint32_t off, u32x4 (&out)[2]) {  // words past a row's end read as word 0
        if (whole || off + 8 < widest) {
#pragma unroll
            for (int t = 0; t < 2; t++) out[t] = *reinterpret_cast<const GLOBAL u32x4u*>(rp[t] + off);
        } else {
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    out[t][i] = rp[t][off + 4 * l.h + i < width[t] ? (int64_t)(off + i) : -(int64_t)(4 * l.h)];
        }
    };
    u32x4 next[2];
    load(0, next);
    for (uint32_t off = 0; off < widest; off += 8) {
        const u32x4 cur[2] = {next[0], next[1]};
        if (off + 8 < widest) load(off + 8, next);
        const uint32_t cnt[2] = {width[0] - off, width[1] - off};
        sp.absorb(cur, whole || off + 8 < widest, cnt, l.h, v);
    }
    uint32_t st[2][8];
    mx_last<F>(st, sp.b, v);
    if (!pack) {
        mx_store_digests(jb->digests, group, jb->rows, l, st);
        return;
    }
#pragma unroll
    for (int t = 0; t < 2; t++)
        if (uint32_t* const d = pack_rows[jb->pack + 32 * t + l.n].digest)
            *reinterpret_cast<GLOBAL u32x4*>((gptr)d + 4 * l.h) = u32x4{st[t][0], st[t][1], st[t][2], st[t][3]};
}

template <class F>
MX_KERNEL compress_batch_kernel(const CompressJob* __restrict__ jobs,
                                                                    const uint64_t* __restrict__ prefix,
                                                                    int njobs, uint64_t total) {
    __shared__ MxTable<F> tab;
    mx_load<F>(tab);
    MxView<F> v(tab);
    const MxLane l;
    const uint64_t stride = (uint64_t)gridDim.x * MX_WAVES;
    for (uint64_t group = mx_wave(); 64 * group < total; group += stride) {
        uint64_t node[2];
        mx_group_rows(node, group, total, l);
        uint32_t* dst[2];
        mx4 full[2][2], b[2][2];
#pragma unroll
        for (int t = 0; t < 2; t++) {  // each lane finds its own nodes' jobs
            const int j = find_job(prefix, njobs, node[t]);
            const uint64_t i = node[t] - prefix[j];
            const gcptr src = (gcptr)jobs[j].prev + 16 * i + 4 * l.h;
            dst[t] = jobs[j].next + 8 * i + 4 * l.h;
#pragma unroll
            for (int s = 0; s < 2; s++) full[t][s] = mx_op(*reinterpret_cast<const GLOBAL u32x4*>(src + 8 * s));
        }
        int x[2][8];
        uint32_t st[2][8];
        v.fresh();
        mx_init<F>(x, full, v);
        mx_rounds<F>(b, x, v);
        mx_last<F>(st, b, v);
#pragma unroll
        for (int t = 0; t < 2; t++)
            if (64 * group + 32 * t + l.n < total)
                *reinterpret_cast<GLOBAL u32x4*>((gptr)dst[t]) = u32x4{st[t][0], st[t][1], st[t][2], st[t][3]};
    }
}

template <class F>
MX16_KERNEL compress_batch_small_kernel(const CompressJob* __restrict__ jobs, const uint64_t* __restrict__ prefix,
                                        int njobs, uint64_t total) {
    const Mx16<F> P;
    const Mx16Lane l;
    const uint64_t r = ((uint64_t)blockIdx.x * S_WAVES + mx16_wave()) * 16 + l.n;
    const uint64_t rr = r < total ? r : total - 1;
    const int j = find_job(prefix, njobs, rr);
    const uint64_t i = rr - prefix[j];
    const u32x4 w = *reinterpret_cast<const GLOBAL u32x4*>((gcptr)jobs[j].prev + 16 * i + 4 * l.q);
    const u32x4 d = mx16_words<F>(P.permute(Mx16<F>::op(__builtin_bit_cast(mx4, w))));
    if (r < total && l.q < 2) *reinterpret_cast<GLOBAL u32x4*>((gptr)jobs[j].next + 8 * i + 4 * l.q) = d;
}

__global__ void gather_roots_kernel(const uint32_t* const* __restrict__ src, uint32_t* __restrict__ dst, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n * 8) dst[i] = src[i >> 3][i & 7];
}

static unsigned grid_for(uint64_t n, unsigned block) { return (unsigned)((n + block - 1) / block); }
// workgroups for n rows, 64 per wave
static unsigned mx_grid(uint64_t n) { return (unsigned)((n + 64 * MX_WAVES - 1) / (64 * MX_WAVES)); }
// workgroups for n rows or nodes, 16 per wave
static unsigned small_grid(uint64_t n) { return (unsigned)((n + 16 * S_WAVES - 1) / (16 * S_WAVES)); }
// Compress kernels loop over the nodes with at most four workgroups per CU,
// so the table load of a workgroup is shared by its waves' nodes.
static unsigned mx_grid_loop(uint64_t n) { return std::min(mx_grid(n), 1024u); }

// ---- proof of work ------------------------------------------------------------
// check_witness (circuit/challenger.rs:210-222): observe(w), then sample_bits(bits)
// == 0.  Either way the n_in pending inputs and w overwrite words 0..n_in of the
// state, one permutation runs, and the sample is word 7.  64 candidates per wave,
// ascending over the grid; a wave stops once a smaller witness is known, so a
// launch costs what the smallest witness needs and not its whole range (2^22
// candidates, one thread each, took 500 us whatever the witness; 16 bits now 26).
template <class F>
MX_KERNEL pow_kernel(const uint32_t* state, const uint32_t* in, int n_in, uint32_t mask, uint32_t start,
                     uint32_t count, uint32_t* result) {
    __shared__ MxTable<F> tab;
    mx_load<F>(tab);
    MxView<F> v(tab);
    const MxLane l;
    uint32_t word[2][4];  // of the lane: words 4 h + i and 8 + 4 h + i
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int j = 4 * (int)l.h + i;
        word[0][i] = j < n_in ? in[j] : state[j];
        word[1][i] = state[8 + j];
    }
    const uint64_t stride = (uint64_t)gridDim.x * MX_WAVES;
    for (uint64_t group = mx_wave(); 64 * group < count; group += stride) {
        const uint32_t w0 = start + (uint32_t)(64 * group);
        const uint32_t known = __hip_atomic_load(result, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if ((uint32_t)__builtin_amdgcn_readfirstlane((int)known) < w0) return;
        mx4 st[2][2], b[2][2];
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const uint32_t wm = to_monty<F>(w0 + 32 * t + l.n);  // past count: computed, not reported
            u32x4 rate;
#pragma unroll
            for (int i = 0; i < 4; i++) rate[i] = 4 * (int)l.h + i == n_in ? wm : word[0][i];
            st[t][0] = mx_op(rate);
            st[t][1] = mx_op(u32x4{word[1][0], word[1][1], word[1][2], word[1][3]});
        }
        int x[2][8];
        uint32_t out[2][8];
        v.fresh();
        mx_init<F>(x, st, v);
        mx_rounds<F>(b, x, v);
        mx_last<F>(out, b, v);
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const uint64_t c = 64 * group + 32 * t + l.n;
            if (l.h && c < count && (from_monty<F>(out[t][3]) & mask) == 0) atomicMin(result, start + (uint32_t)c);
        }
    }
}

hipError_t launch_pow_search(int field, const uint32_t* state, const uint32_t* in, int n_in, int bits,
                             uint32_t start, uint32_t count, uint32_t* result, hipStream_t stream) {
    if (count == 0) return hipSuccess;
    const uint32_t mask = (1u << bits) - 1u;
    if (field == FIELD_KOALABEAR)
        pow_kernel<KoalaBear><<<mx_grid_loop(count), MX_THREADS, 0, stream>>>(state, in, n_in, mask, start, count, result);
    else
        pow_kernel<BabyBear><<<mx_grid_loop(count), MX_THREADS, 0, stream>>>(state, in, n_in, mask, start, count, result);
    return hipGetLastError();
}

hipError_t launch_gather_roots(const uint32_t* const* src, uint32_t* dst, int n, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    gather_roots_kernel<<<grid_for((uint64_t)n * 8, 256), 256, 0, stream>>>(src, dst, n);
    return hipGetLastError();
}

template <class F>
static hipError_t leaf_hash_batch_t(const LeafJob* jobs, const uint64_t* prefix, int njobs, uint64_t total,
                                    const LeafRow* pack_rows, hipStream_t stream) {
    const unsigned g = grid_for(total, MX_WAVES);
    if (pack_rows)
        leaf_hash_batch_kernel<F, true><<<g, MX_THREADS, 0, stream>>>(jobs, prefix, njobs, total, pack_rows);
    else
        leaf_hash_batch_kernel<F, false><<<g, MX_THREADS, 0, stream>>>(jobs, prefix, njobs, total, nullptr);
    return hipGetLastError();
}
hipError_t launch_leaf_hash_batch(int field, const LeafJob* jobs, const uint64_t* prefix, int njobs, uint64_t total,
                                  const LeafRow* pack_rows, hipStream_t stream) {
    if (total == 0) return hipSuccess;
    return field == FIELD_KOALABEAR ? leaf_hash_batch_t<KoalaBear>(jobs, prefix, njobs, total, pack_rows, stream)
                                    : leaf_hash_batch_t<BabyBear>(jobs, prefix, njobs, total, pack_rows, stream);
}

hipError_t launch_compress_batch(int field, const CompressJob* jobs, const uint64_t* prefix, int njobs,
                                 uint64_t total, hipStream_t stream) {
    if (total == 0) return hipSuccess;
    if (total <= SMALL_MAX_NODES) {
        const unsigned g = small_grid(total);
        if (field == FIELD_KOALABEAR)
            compress_batch_small_kernel<KoalaBear><<<g, S_THREADS, 0, stream>>>(jobs, prefix, njobs, total);
        else
            compress_batch_small_kernel<BabyBear><<<g, S_THREADS, 0, stream>>>(jobs, prefix, njobs, total);
        return hipGetLastError();
    }
    if (field == FIELD_KOALABEAR)
        compress_batch_kernel<KoalaBear><<<mx_grid_loop(total), MX_THREADS, 0, stream>>>(jobs, prefix, njobs, total);
    else
        compress_batch_kernel<BabyBear><<<mx_grid_loop(total), MX_THREADS, 0, stream>>>(jobs, prefix, njobs, total);
    return hipGetLastError();
}

// Nodes (or rows) of the first layer, at most SMALL_MAX_NODES: 64 per workgroup
// and seven layers a launch, one workgroup for all the rest once a layer has at
// most 128 nodes (rows of several chunks stay at 64: a wave would hash its two
// groups of rows one after the other).
TreeStep tree_step(uint64_t n0, int layers, uint32_t leaf_width) {
    TreeStep t;
    t.log_per = 6;
    if (n0 <= (uint64_t)(leaf_width > 8 ? 64 : TREE_MAX_PER)) t.log_per = __builtin_ctzll(n0);
    t.layers = std::min(layers, t.log_per + 1);
    t.threads = std::min((unsigned)S_THREADS, std::max(64u, 4u << t.log_per));
    t.blocks = (unsigned)(n0 >> t.log_per);
    return t;
}

hipError_t launch_tree_layers_batch(int field, const TreeJob* jobs, const uint64_t* prefix, int njobs, unsigned blocks,
                                    unsigned threads, hipStream_t stream) {
    if (blocks == 0) return hipSuccess;
    const uint32_t* const in = reinterpret_cast<const uint32_t*>(jobs);
    const uint64_t at = reinterpret_cast<uint64_t>(prefix);
    if (field == FIELD_KOALABEAR)
        tree_layers_kernel<KoalaBear, TREE_JOBS><<<blocks, threads, 0, stream>>>(in, at, 0, njobs, 0, 0, nullptr, {}, {});
    else
        tree_layers_kernel<BabyBear, TREE_JOBS><<<blocks, threads, 0, stream>>>(in, at, 0, njobs, 0, 0, nullptr, {}, {});
    return hipGetLastError();
}

hipError_t launch_leaf_hash(int field, const MatRef* mats, int n, uint32_t total_width,
                            size_t rows, uint32_t* digests, hipStream_t stream) {
    if (rows == 0) return hipSuccess;
    if (rows <= SMALL_MAX_NODES) {
        if (field == FIELD_KOALABEAR)
            leaf_hash_small_kernel<KoalaBear><<<small_grid(rows), S_THREADS, 0, stream>>>(mats, n, total_width, rows, digests);
        else
            leaf_hash_small_kernel<BabyBear><<<small_grid(rows), S_THREADS, 0, stream>>>(mats, n, total_width, rows, digests);
        return hipGetLastError();
    }
    const unsigned g = mx_grid(rows);
    if (field == FIELD_KOALABEAR)
        leaf_hash_kernel<KoalaBear><<<g, MX_THREADS, 0, stream>>>(mats, n, total_width, rows, digests);
    else
        leaf_hash_kernel<BabyBear><<<g, MX_THREADS, 0, stream>>>(mats, n, total_width, rows, digests);
    return hipGetLastError();
}

hipError_t launch_absorb_segment(int field, const uint32_t* data, uint64_t stride, uint32_t width, uint32_t pos0,
                                 int first, int last, uint64_t rows, uint32_t* state, uint32_t* digests,
                                 hipStream_t stream) {
    if (rows == 0) return hipSuccess;
    if (pos0 > 7 || (!last && !state) || (last && !digests) || (!first && !state)) return hipErrorInvalidValue;
    const unsigned g = mx_grid(rows);
    if (field == FIELD_KOALABEAR)
        absorb_segment_kernel<KoalaBear><<<g, MX_THREADS, 0, stream>>>(data, stride, width, pos0, first, last, rows, state, digests);
    else
        absorb_segment_kernel<BabyBear><<<g, MX_THREADS, 0, stream>>>(data, stride, width, pos0, first, last, rows, state, digests);
    return hipGetLastError();
}

// For a height group that is one matrix with width % 8 == 0 and 16-byte aligned rows.
hipError_t launch_leaf_hash_w8(int field, const uint32_t* data, uint64_t stride, uint32_t width,
                               size_t rows, uint32_t* digests, hipStream_t stream) {
    if (rows == 0) return hipSuccess;
    const unsigned g = mx_grid(rows);
    if (field == FIELD_KOALABEAR)
        leaf_hash_w8_kernel<KoalaBear><<<g, MX_THREADS, 0, stream>>>(data, stride, width / 8, rows, digests);
    else
        leaf_hash_w8_kernel<BabyBear><<<g, MX_THREADS, 0, stream>>>(data, stride, width / 8, rows, digests);
    return hipGetLastError();
}

template <class F>
static hipError_t tree_layers_t(const uint32_t* in, uint64_t stride, uint32_t leaf_width, uint64_t n0, int layers,
                                uint32_t* out, hipStream_t s, const TreeChallenge* ch, const TreeFold* fold) {
    while (layers > 0) {
        const TreeStep t = tree_step(n0, layers, leaf_width);
        const int log_per = t.log_per, now = t.layers;
        const unsigned threads = t.threads, g = t.blocks;
        const TreeChallenge c = ch && now == layers ? *ch : TreeChallenge{};
        if (fold)
            tree_layers_kernel<F, TREE_FOLDED><<<g, threads, 0, s>>>(nullptr, 0, 0, n0, log_per, now, out, c, *fold);
        else if (leaf_width)
            tree_layers_kernel<F, TREE_ROWS><<<g, threads, 0, s>>>(in, stride, leaf_width, n0, log_per, now, out, c, {});
        else
            tree_layers_kernel<F, TREE_NODES><<<g, threads, 0, s>>>(in, 0, 0, n0, log_per, now, out, c, {});
        for (int i = 0; i < now; i++) {  // the last layer written feeds the next launch
            in = out;
            out += 8 * n0;
            n0 >>= 1;
        }
        leaf_width = 0;
        fold = nullptr;
        layers -= now;
    }
    return hipGetLastError();
}

hipError_t launch_tree_layers(int field, const uint32_t* in, uint64_t stride, uint32_t leaf_width, uint64_t n0,
                              int layers, uint32_t* out, hipStream_t stream, const TreeChallenge* ch,
                              const TreeFold* fold) {
    if (layers <= 0) return hipSuccess;
    if (ch && (n0 >> (layers - 1)) != 1) return hipErrorInvalidValue;  // sampled from the root
    if (n0 == 0 || n0 > SMALL_MAX_NODES || (n0 & (n0 - 1)) || (n0 >> (layers - 1)) == 0) return hipErrorInvalidValue;
    return field == FIELD_KOALABEAR ? tree_layers_t<KoalaBear>(in, stride, leaf_width, n0, layers, out, stream, ch, fold)
                                    : tree_layers_t<BabyBear>(in, stride, leaf_width, n0, layers, out, stream, ch, fold);
}

hipError_t launch_compress(int field, const uint32_t* prev, uint32_t* next, size_t n_out,
                           const MatRef* inj, int n_inj, uint32_t inj_width, hipStream_t stream) {
    if (n_out == 0) return hipSuccess;
    if (n_inj > 0 && n_out <= SMALL_MAX_NODES) {
        if (field == FIELD_KOALABEAR)
            compress_small_kernel<KoalaBear><<<small_grid(n_out), S_THREADS, 0, stream>>>(prev, next, n_out, inj, n_inj, inj_width, nullptr);
        else
            compress_small_kernel<BabyBear><<<small_grid(n_out), S_THREADS, 0, stream>>>(prev, next, n_out, inj, n_inj, inj_width, nullptr);
        return hipGetLastError();
    }
    const unsigned g = mx_grid_loop(n_out);
    if (field == FIELD_KOALABEAR) {
        if (n_inj > 0)
            compress_kernel<KoalaBear, true><<<g, MX_THREADS, 0, stream>>>(prev, next, n_out, inj, n_inj, inj_width);
        else
            compress_kernel<KoalaBear, false><<<g, MX_THREADS, 0, stream>>>(prev, next, n_out, inj, n_inj, inj_width);
    } else {
        if (n_inj > 0)
            compress_kernel<BabyBear, true><<<g, MX_THREADS, 0, stream>>>(prev, next, n_out, inj, n_inj, inj_width);
        else
            compress_kernel<BabyBear, false><<<g, MX_THREADS, 0, stream>>>(prev, next, n_out, inj, n_inj, inj_width);
    }
    return hipGetLastError();
}

hipError_t launch_compress_digest(int field, const uint32_t* prev, uint32_t* next, size_t n_out,
                                  const uint32_t* inj, hipStream_t stream) {
    if (n_out == 0) return hipSuccess;
    if (n_out <= SMALL_MAX_NODES) {
        if (field == FIELD_KOALABEAR)
            compress_small_kernel<KoalaBear><<<small_grid(n_out), S_THREADS, 0, stream>>>(prev, next, n_out, nullptr, 0, 0, inj);
        else
            compress_small_kernel<BabyBear><<<small_grid(n_out), S_THREADS, 0, stream>>>(prev, next, n_out, nullptr, 0, 0, inj);
        return hipGetLastError();
    }
    const unsigned g = mx_grid_loop(n_out);
    if (field == FIELD_KOALABEAR)
        compress_digest_kernel<KoalaBear><<<g, MX_THREADS, 0, stream>>>(prev, inj, next, n_out);
    else
        compress_digest_kernel<BabyBear><<<g, MX_THREADS, 0, stream>>>(prev, inj, next, n_out);
    return hipGetLastError();
}

hipError_t launch_open_gather(const MatRef* mats, const uint32_t* shift, const uint32_t* col_off,
                              int n_mats, uint32_t total_width, const uint32_t* digests,
                              const uint64_t* layer_off, int log_h, const uint64_t* idx, int nq,
                              uint32_t* rows_out, uint32_t* paths_out, hipStream_t stream) {
    if (nq == 0) return hipSuccess;
    open_gather_kernel<<<nq, 128, 0, stream>>>(mats, shift, col_off, n_mats, total_width, digests,
                                               layer_off, log_h, idx, rows_out, paths_out);
    return hipGetLastError();
}

}  // namespace pg
