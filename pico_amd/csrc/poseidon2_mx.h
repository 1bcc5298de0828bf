// poseidon2_mx.h -- the Poseidon2 permutation of poseidon2.h with its linear
// layers on the matrix cores: one wave permutes 64 states.
//
// The permutation is bound by VALU issue (one state per lane: 3787 issue
// slots for KoalaBear, 4654 for BabyBear, three quarters of them 32x32
// multiplies and 64-bit adds), and about 60% of them are linear algebra mod
// p.  Here every linear layer is an exact integer matrix product on
// v_mfma_i32_32x32x32_i8, and the VALU is left with the S-boxes, a 3.5-slot
// reduction per layer output and the partial rounds' short recurrences: 1697
// slots (KoalaBear; BabyBear 2438) beside 102 (90) matrix instructions of 32
// cycles for 64 states.  Leaf hash of 2^21 rows x 256 columns: KoalaBear 6.93
// -> 4.53 ms, BabyBear 9.55 -> 5.62 ms.  What bounds it now: with the matrix
// instructions taken out the rest runs 8080 cycles per wave and permutation at
// 2.39 GHz; with them 9280 cycles at 2.05 GHz (each takes 10-16 cycles of
// issue, and the clock drops under their load).
//
// A matrix product mod p in bytes.  A state word x (any int32) is four bytes
// x = sum_b x_b 2^8b, the top one signed; x ^ 0x00808080 makes the lower three
// signed as well (x_b - 128; the constant 128 (1 + 2^8 + 2^16) = 0x808080 per
// unit of coefficient goes to the bias).  A coefficient c enters once per
// byte: D = c 2^8b 2^16 mod p, taken in (-p/2, p/2) and split into four
// balanced base-256 digits D = sum_a d_a 2^8a.  The i8 product accumulates
// plane a: acc_a = sum_{in, b} d_a x_b, at most 40 words x 4 bytes x 2^14 <
// 2^22, and
//   v = (acc_0 + 2^8 acc_1) + 2^16 (acc_2 + 2^8 acc_3) = t + 2^16 u
// is 2^16 times the wanted sum mod p.  Both primes are 1 mod 2^16, so 2^-16 =
// -(p-1)/2^16 mod p, a 15-bit number (32512 and 30720), and the output is
//   u + round(t / 2^16) - (p-1)/2^16 * (t's low half, signed),
// below 2^30 + 2^30 in size: an int32 that is the sum mod p.  With 0x8000 in
// the bias of plane 0 the rounding is a plain high half, so an output takes
// v_lshl_add_u32 twice, v_xor_b32 0x8000 and one v_dot2c_i32_i16.  Biases
// (round constants, the byte offsets) enter as the matrix instruction's C
// operand in planes 0 and 2.
//
// S-boxes use signed Montgomery products: |a b| <= 2^62 gives |a b 2^-32| <=
// 2^30 + p/2 < 2^31, so every int32 is a valid operand and no product needs a
// final correction.
//
// Partial rounds.  Only s_0 passes an S-box, so the state before partial
// round r is P^r S + sum_{j<r} P^(r-1-j) q x'_j, with S the state at the first
// partial round, x'_j the S-box output of round j, q the internal matrix's
// column 0 and P the internal matrix with that column cleared.  Round r's
// S-box input is the 0th entry plus a constant: a linear form of S and of the
// earlier x'.  S itself is the external layer of the fourth full round's
// S-box outputs, so the forms are taken of those directly and that layer is
// never computed.  Rounds go in blocks of four: a matrix product gives the
// forms of a block over everything before it, the at most three x' of the
// same block are added on the VALU; after the last block one product gives
// all 16 words of the state, with the next round's constants.
//
// Lanes.  A wave's 64 states are two tiles of 32.  In the matrix
// instruction's layout lane l holds column (state) l % 32 of both B and D;
// half h = l / 32 holds state words 8 s + 4 h + i as register 4 s + i (s = 0
// rate, 1 capacity): 16 bytes per 32-deep step, so a step multiplies the rate
// or the capacity words, and D's rows can be dealt so that every half receives
// all planes of its own words: no data moves between layers.  For the partial
// rounds the two tiles' forms are exchanged by v_permlane32_swap so that half
// h holds all four rounds of its lane's state of tile h.
#pragma once
#include "kernels.h"
#include "poseidon2.h"

namespace pg {

typedef int mx4 __attribute__((ext_vector_type(4)));
typedef int mx16 __attribute__((ext_vector_type(16)));

// ---- tables (compile time) -------------------------------------------------
// Operand A blocks of 64 lanes x 16 bytes, then the C biases (two halves x 16
// words each).
template <class F>
struct MxShape {
    static constexpr int RP = F::ROUNDS_P;
    static constexpr int PAIRS = (RP + 7) / 8;  // pairs of 4-round blocks
    static constexpr bool has_second(int m) { return 8 * m + 4 < RP; }
    // A blocks
    static constexpr int EXT = 0;                    // [step 2][y 2]
    static constexpr int MERGED = 4;                 // [step 2][y 2]
    static constexpr int FORMS = 8;                  // pair m: 2 state steps, m earlier pairs, 1 within the pair
    static constexpr int forms(int m) {
        int k = FORMS;
        for (int i = 0; i < m; i++) k += 2 + i + (has_second(i) ? 1 : 0);
        return k;
    }
    static constexpr int FINAL = forms(PAIRS);       // [2 state steps + PAIRS][y 2]
    static constexpr int NA = FINAL + 2 * (2 + PAIRS);
    // C biases
    static constexpr int B_INIT = 0, B_MERGED = 1, B_EXT = 2 /* + r: after full round r = 0..7 (3: unused) */,
                         B_FINAL = 5 /* in the place of round 3 */, B_FORMS = 10;
    static constexpr int NB = B_FORMS + PAIRS;
};

template <class F>
struct alignas(64) MxTable {
    uint32_t a[MxShape<F>::NA][64][4];
    int32_t c[MxShape<F>::NB][2][16];
};

// one linear layer over at most 16 + 8 PAIRS input words
struct MxLin {
    uint64_t m[16][40];  // [output][input]: inputs 0..15 state words, 16 + r partial round r
    uint64_t k[16];      // constants added
};

// digit `plane` of c 2^16 mod p, balanced
constexpr int32_t mx_centered(uint64_t v, uint32_t p) { return v > p / 2 ? (int32_t)(v - p) : (int32_t)v; }
constexpr int mx_digit(int32_t v, int plane) {
    int64_t x = v;
    int d = 0;
    for (int a = 0; a <= plane; a++) {
        d = (int)(x & 255);
        if (d >= 128) d -= 256;
        x = (x - d) >> 8;
    }
    return d;
}

// the four bytes by which coefficient c enters digit plane `plane`
template <class F>
constexpr uint32_t mx_operand_word(uint64_t c, int plane) {
    uint32_t word = 0;
    for (int b = 0; b < 4 && c; b++) {
        const uint64_t v = ((c << (16 + 8 * (b & 1))) % F::P << (b >= 2 ? 16 : 0)) % F::P;
        word |= (uint32_t)(mx_digit(mx_centered(v, F::P), plane) & 255) << (8 * b);
    }
    return word;
}

template <class F>
constexpr uint64_t mx_external(int r, int c) {
    return M4_COEF[r % 4][c % 4] * ((r / 4 == c / 4) ? 2u : 1u);
}

template <class F>
constexpr uint64_t mx_diag(int i) {  // canonical internal diagonal
    uint64_t r = P2<F>::K.diag[i];   // Montgomery: multiply by 2^-32
    return r * cpow_canon(F::P, (uint32_t)((1ull << 32) % F::P), F::P - 2) % F::P;
}

// A block of one step: `input(half, i)` is the input index of word i of half,
// -1: none; `row(r)` sets the output and the plane of D row r, output -1: none
template <class F, class In, class Row>
constexpr void mx_fill(uint32_t (&a)[64][4], const MxLin& L, In input, Row row) {
    for (int lane = 0; lane < 64; lane++) {
        int out = -1, plane = 0;
        row(lane % 32, out, plane);
        for (int i = 0; i < 4; i++) {
            const int in = input(lane / 32, i);
            a[lane][i] = out >= 0 && in >= 0 ? mx_operand_word<F>(L.m[out][in], plane) : 0;
        }
    }
}

// D row of accumulator register j in half h, and back
constexpr int mx_row_j(int r) { return 4 * (r / 8) + r % 4; }
constexpr int mx_row_h(int r) { return (r / 4) % 2; }
// state words 8 s + 4 h + i: output register o = 4 s + i of half h
constexpr int mx_word(int h, int o) { return 8 * (o / 4) + 4 * h + o % 4; }

// Bias of output `out` (its constant plus 0x808080 per unit of coefficient
// over the inputs [0, nin)), 2^16-scaled and split into a signed low half and
// a high half; plane 0's includes the rounding.
template <class F>
constexpr void mx_bias(const MxLin& L, int out, int nin, int32_t& lo, int32_t& hi) {
    uint64_t s = L.k[out];
    for (int i = 0; i < nin; i++) s = (s + L.m[out][i] * 0x808080u) % F::P;
    const int32_t v = mx_centered((s << 16) % F::P, F::P);
    int32_t l = v & 0xffff;
    if (l >= 0x8000) l -= 0x10000;
    lo = l + 0x8000;
    hi = (int32_t)(((int64_t)v - l) >> 16);
}

template <class F>
constexpr void mx_state_bias(int32_t (&c)[2][16], const MxLin& L, int nin) {
    for (int h = 0; h < 2; h++)
        for (int o = 0; o < 8; o++) mx_bias<F>(L, mx_word(h, o), nin, c[h][o], c[h][8 + o]);
}

// state-to-state layers: y = 0 holds planes 0 and 2, y = 1 planes 1 and 3;
// register j = o + 8 (plane / 2)
template <class F>
constexpr void mx_state_step(uint32_t (&a)[64][4], const MxLin& L, int in0, int y) {
    mx_fill<F>(
        a, L, [&](int h, int i) { return in0 + 4 * h + i; },
        [&](int r, int& out, int& plane) {
            const int j = mx_row_j(r);
            out = mx_word(mx_row_h(r), j % 8);
            plane = y + 2 * (j / 8);
        });
}
// partial-round inputs of pair n: word i of half h is round 8 n + 4 (i / 2) +
// 2 h + i % 2
constexpr int mx_round(int pair, int h, int i) { return 8 * pair + 4 * (i / 2) + 2 * h + i % 2; }

// The permutation's linear layers (see above); `forms` row r: round r's form
// over the state words and the x' of the blocks of four before its own.
template <class F>
struct MxParts {
    MxLin ext, merged, fin;
    uint64_t forms[F::ROUNDS_P][40];
};
template <class F>
constexpr MxParts<F> make_mx_parts() {
    constexpr uint64_t p = F::P;
    constexpr int RP = F::ROUNDS_P;
    MxParts<F> t{};
    for (int r = 0; r < 16; r++)
        for (int c = 0; c < 16; c++) t.ext.m[r][c] = mx_external<F>(r, c);
    // the last external layer of one permutation and the first of the next,
    // whose rate words are overwritten: the capacity words' share
    for (int r = 0; r < 16; r++) {
        for (int e = 0; e < 16; e++) {
            uint64_t v = 0;
            for (int c = 8; c < 16; c++) v += t.ext.m[r][c] * t.ext.m[c][e];
            t.merged.m[r][e] = v % p;
        }
        t.merged.k[r] = P2<F>::K.ext_rc[0][r];
        for (int c = 0; c < 8; c++)  // the new rate words' byte offsets
            t.merged.k[r] = (t.merged.k[r] + t.ext.m[r][c] * 0x808080u) % p;
    }
    // partial rounds: columns P^k q, rows e_0 P^r and P^RP over the state
    uint64_t d[16] = {};
    for (int i = 0; i < 16; i++) d[i] = mx_diag<F>(i);
    uint64_t pq[24][16] = {};
    for (int i = 0; i < 16; i++) pq[0][i] = i == 0 ? (d[0] + 1) % p : 1;
    for (int k = 1; k < RP; k++) {
        uint64_t sum = 0;
        for (int i = 1; i < 16; i++) sum += pq[k - 1][i];
        for (int i = 0; i < 16; i++) pq[k][i] = (sum + (i ? d[i] * pq[k - 1][i] : 0)) % p;
    }
    uint64_t pw[16][16] = {};  // P^r
    for (int i = 0; i < 16; i++) pw[i][i] = 1;
    for (int r = 0; r <= RP; r++) {
        for (int o = 0; o < (r < RP ? 1 : 16); o++)
            for (int c = 0; c < 16; c++) {
                uint64_t v = 0;
                for (int k = 0; k < 16; k++) v += pw[o][k] * t.ext.m[k][c] % p;
                if (r < RP)
                    t.forms[r][c] = v % p;
                else
                    t.fin.m[o][c] = v % p;
            }
        for (int c = 0; c < 16; c++) {  // pw <- P pw
            uint64_t sum = 0;
            for (int i = 1; i < 16; i++) sum += pw[i][c];
            for (int i = 0; i < 16; i++) pw[i][c] = (sum + (i ? d[i] * pw[i][c] : 0)) % p;
        }
    }
    for (int r = 0; r < RP; r++)
        for (int j = 0; j < r / 4 * 4; j++) t.forms[r][16 + j] = pq[r - 1 - j][0];
    for (int o = 0; o < 16; o++) {
        for (int j = 0; j < RP; j++) t.fin.m[o][16 + j] = pq[RP - 1 - j][o];
        t.fin.k[o] = P2<F>::K.ext_rc[4][o];
    }
    return t;
}

template <class F>
constexpr MxTable<F> make_mx_table() {
    using S = MxShape<F>;
    constexpr int RP = F::ROUNDS_P;
    MxTable<F> t{};
    const MxParts<F> parts = make_mx_parts<F>();
    MxLin ext = parts.ext;
    for (int s = 0; s < 2; s++)
        for (int y = 0; y < 2; y++) {
            mx_state_step<F>(t.a[S::EXT + 2 * s + y], ext, 8 * s, y);
            mx_state_step<F>(t.a[S::MERGED + 2 * s + y], parts.merged, 8 * s, y);
        }
    // the external layer's biases with each round's constants (words are in
    // Montgomery form)
    auto ext_bias = [&](int slot, int round) {
        for (int i = 0; i < 16; i++) ext.k[i] = round < 0 ? 0 : P2<F>::K.ext_rc[round][i];
        mx_state_bias<F>(t.c[slot], ext, 16);
    };
    ext_bias(S::B_INIT, 0);
    for (int r = 0; r < 8; r++)
        if (r != 3) ext_bias(S::B_EXT + r, r == 7 ? -1 : r + 1);
    mx_state_bias<F>(t.c[S::B_MERGED], parts.merged, 16);
    for (int s = 0; s < 2 + S::PAIRS; s++)
        for (int y = 0; y < 2; y++)
            mx_fill<F>(
                t.a[S::FINAL + 2 * s + y], parts.fin,
                [&](int h, int i) {
                    if (s < 2) return 8 * s + 4 * h + i;
                    const int r = mx_round(s - 2, h, i);
                    return r < RP ? 16 + r : -1;
                },
                [&](int r, int& out, int& plane) {
                    const int j = mx_row_j(r);
                    out = mx_word(mx_row_h(r), j % 8);
                    plane = y + 2 * (j / 8);
                });
    mx_state_bias<F>(t.c[S::B_FINAL], parts.fin, 16 + RP);
    // forms of pair m: output 4 beta + o is round 8 m + 4 beta + o (o = 2 h +
    // g), register j = 8 beta + 2 plane + g
    for (int m = 0; m < S::PAIRS; m++) {
        MxLin f{};
        for (int q = 0; q < 8; q++) {
            const int r = 8 * m + q;
            if (r >= RP) continue;
            for (int c = 0; c < 40; c++) f.m[q][c] = parts.forms[r][c];
            f.k[q] = P2<F>::K.int_rc[r];
        }
        auto rows = [&](bool second_only) {
            return [&, second_only](int r, int& out, int& plane) {
                const int j = mx_row_j(r), beta = j / 8, g = j % 2;
                plane = (j % 8) / 2;
                out = 4 * beta + 2 * mx_row_h(r) + g;
                if (second_only && beta == 0) out = -1;
            };
        };
        const int base = S::forms(m);
        for (int s = 0; s < 2; s++)
            mx_fill<F>(t.a[base + s], f, [&](int h, int i) { return 8 * s + 4 * h + i; }, rows(false));
        for (int n = 0; n < m; n++)
            mx_fill<F>(t.a[base + 2 + n], f, [&](int h, int i) { return 16 + mx_round(n, h, i); }, rows(false));
        if (S::has_second(m))
            mx_fill<F>(t.a[base + 2 + m], f, [&](int h, int i) { return i < 2 ? 16 + mx_round(m, h, i) : -1; }, rows(true));
        for (int h = 0; h < 2; h++)
            for (int beta = 0; beta < 2; beta++)
                for (int g = 0; g < 2; g++)
                    mx_bias<F>(f, 4 * beta + 2 * h + g, 16 + 8 * m + 4 * beta, t.c[S::B_FORMS + m][h][8 * beta + g],
                               t.c[S::B_FORMS + m][h][8 * beta + 4 + g]);
    }
    return t;
}

// ---- 16 states per wave ------------------------------------------------------
// For layers that do not fill the GPU a permutation costs its latency, which
// is the instructions a wave issues (one in 4.2 cycles, dependent or not).
// Here a wave holds 16 states, four lanes each, on v_mfma_i32_16x16x64_i8:
// lane l holds column (state) l % 16 and, with q = l / 16, state words 4 q + i
// as register i: the 16 words of a state are one 64-deep step.  D row 4 q + i
// is the same word of the same lane, so a layer is one matrix instruction per
// plane.  A block of partial rounds is one instruction per step: row 4 o +
// plane, so lane group q holds all planes of the block's form q; the four
// forms are spread over the lane groups by permlane swaps and every group runs
// the four S-boxes.  x'_r is operand word r % 16 -> group r % 4, register r / 4
// of step r / 16.  The tables stay in registers (192 for KoalaBear).
// A tree layer of at most 64 nodes per CU: 3.2 us with one state on 16 lanes
// (additions by DPP moves), 7 us with 64 states per wave, 2.2 us this way;
// the 8 layers above 2^8 digests 36.5 -> 21.2 us, a leaf layer of 512 rows x
// 16 13.7 -> 6.9 us.
template <class F>
struct Mx16Shape {
    static constexpr int RP = F::ROUNDS_P;
    static constexpr int BLOCKS = (RP + 3) / 4;
    static constexpr int STEPS = 1 + (RP + 15) / 16;  // of the layer after the partial rounds
    static_assert(BLOCKS <= 5, "the forms read at most one step of x'");
    static constexpr int EXT = 0;    // [plane 4]
    static constexpr int FORMS = 4;  // block 0: one step; the others: state, x'
    static constexpr int forms(int b) { return FORMS + (b ? 2 * b - 1 : 0); }
    static constexpr int FINAL = FORMS + 2 * BLOCKS - 1;  // [step][plane 4]
    static constexpr int NA = FINAL + 4 * STEPS;
    // biases: before full rounds 0..7 (4: after the partial rounds), after the last
    static constexpr int NC = 9;
};
template <class F>
struct alignas(64) Mx16Table {
    uint32_t a[Mx16Shape<F>::NA][64][4];
    int32_t c[Mx16Shape<F>::NC][2][16];             // planes 0 and 2 of word w
    int32_t f[Mx16Shape<F>::BLOCKS][16];            // plane i of form q at 4 q + i
};
template <class F>
constexpr Mx16Table<F> make_mx16_table() {
    using S = Mx16Shape<F>;
    constexpr int RP = F::ROUNDS_P;
    Mx16Table<F> t{};
    const MxParts<F> parts = make_mx_parts<F>();
    // one step: input(q, i), row(r) -> output and plane
    auto fill = [&](uint32_t (&a)[64][4], const MxLin& L, auto input, auto row) {
        for (int lane = 0; lane < 64; lane++) {
            int out = -1, plane = 0;
            row(lane % 16, out, plane);
            for (int i = 0; i < 4; i++) {
                const int in = input(lane / 16, i);
                a[lane][i] = out >= 0 && in >= 0 ? mx_operand_word<F>(L.m[out][in], plane) : 0;
            }
        }
    };
    auto state = [](int q, int i) { return 4 * q + i; };
    auto rounds = [](int step) {
        return [step](int q, int i) {
            const int r = 16 * step + 4 * i + q;
            return r < RP ? 16 + r : -1;
        };
    };
    for (int p = 0; p < 4; p++) {
        auto rows = [p](int r, int& out, int& plane) {
            out = r;
            plane = p;
        };
        fill(t.a[S::EXT + p], parts.ext, state, rows);
        fill(t.a[S::FINAL + p], parts.fin, state, rows);
        for (int s = 1; s < S::STEPS; s++) fill(t.a[S::FINAL + 4 * s + p], parts.fin, rounds(s - 1), rows);
    }
    for (int b = 0; b < S::BLOCKS; b++) {
        MxLin f{};
        for (int o = 0; o < 4; o++) {
            if (4 * b + o >= RP) continue;
            for (int c = 0; c < 40; c++) f.m[o][c] = parts.forms[4 * b + o][c];
            f.k[o] = P2<F>::K.int_rc[4 * b + o];
        }
        auto rows = [](int r, int& out, int& plane) {
            out = r / 4;
            plane = r % 4;
        };
        fill(t.a[S::forms(b)], f, state, rows);
        if (b) fill(t.a[S::forms(b) + 1], f, rounds(0), rows);
        for (int o = 0; o < 4; o++) mx_bias<F>(f, o, 16 + 4 * b, t.f[b][4 * o], t.f[b][4 * o + 2]);
    }
    MxLin ext = parts.ext;
    for (int k = 0; k < S::NC; k++) {
        for (int w = 0; w < 16; w++) ext.k[w] = k == 8 ? 0 : P2<F>::K.ext_rc[k][w];
        for (int w = 0; w < 16; w++)
            if (k == 4)
                mx_bias<F>(parts.fin, w, 16 + RP, t.c[k][0][w], t.c[k][1][w]);
            else
                mx_bias<F>(ext, w, 16, t.c[k][0][w], t.c[k][1][w]);
    }
    return t;
}

// Coefficients of x'_{r-k} in round r's S-box input within a block, in
// Montgomery form and centered: c_1 = d_0 + 1 = -1, c_2 = 15, c_3 = e_0 P^2 q
template <class F>
struct MxRec {
    static constexpr int32_t ONE = mx_centered(F::R1, F::P);
    static constexpr int32_t C1 = -ONE;
    static constexpr int32_t C2 = mx_centered(15ull * F::R1 % F::P, F::P);
    static constexpr int32_t c3() {
        uint64_t s = 15ull * 15;
        for (int i = 1; i < 16; i++) s += mx_diag<F>(i);
        return mx_centered(s % F::P * F::R1 % F::P, F::P);
    }
    static constexpr int32_t C3 = c3();
    static constexpr int64_t mag(int64_t v) { return v < 0 ? -v : v; }
    // every operand is an int32: the sum's Montgomery reduction is one too
    static_assert((mag(ONE) + mag(C1) + mag(C2) + mag(C3)) / 2 + F::P / 2 < (1ll << 31), "block recurrence fits int32");
};

// ---- device ------------------------------------------------------------------
// The recurrence's constants in scalar registers, one v_mad_i64_i32 a product.
// They pass through an empty asm, which hides their values: the compiler makes
// products by constants near powers of two shifts and 64-bit subtractions.  A set
// is made for each block of rounds: one for the whole kernel lets the sign
// extensions leave loops, and each product becomes a full 64-bit one.  The
// instruction itself is left to the compiler, because between a matrix
// instruction and a vector instruction that touches its registers the program has
// to wait (the hardware does not), and the compiler places those waits only for
// instructions it knows.
template <class F>
struct MxConst {
    int one = MxRec<F>::ONE, c1 = MxRec<F>::C1, c2 = MxRec<F>::C2, c3 = MxRec<F>::C3;
    __device__ __forceinline__ MxConst() { asm("" : "+s"(one), "+s"(c1), "+s"(c2), "+s"(c3)); }
};

static __device__ const MxTable<KoalaBear> kMxKb = make_mx_table<KoalaBear>();
static __device__ const MxTable<BabyBear> kMxBb = make_mx_table<BabyBear>();

template <class F>
__device__ __forceinline__ const MxTable<F>& mx_table() {
    if constexpr (F::P == KoalaBear::P)
        return kMxKb;
    else
        return kMxBb;
}

constexpr uint32_t MX_BIAS = 0x00808080u;  // signed bytes

// Copies the tables to LDS (every thread of the block; ends with a barrier).
template <class F>
__device__ __forceinline__ void mx_load(MxTable<F>& lds) {
    const uint4* src = reinterpret_cast<const uint4*>(&mx_table<F>());
    uint4* dst = reinterpret_cast<uint4*>(&lds);
    for (uint32_t i = threadIdx.x; i < sizeof(MxTable<F>) / 16; i += blockDim.x) dst[i] = src[i];
    __syncthreads();
}

// Montgomery product of any two int32, in [-2^31, 2^31)
template <class F>
__device__ __forceinline__ int mx_redc(int64_t v) {
    constexpr uint32_t PINV = inv_mod_2_32(F::P);
    const int m = (int)((uint32_t)v * PINV);
    return (int)((v - (int64_t)m * (int)F::P) >> 32);
}
template <class F>
__device__ __forceinline__ int mx_sbox(int x) {
    const int x2 = mx_redc<F>((int64_t)x * x);
    const int x3 = mx_redc<F>((int64_t)x2 * x);
    if constexpr (F::SBOX == 3) return x3;
    return mx_redc<F>((int64_t)mx_redc<F>((int64_t)x2 * x2) * x3);
}
// S-box output as a matrix operand word
template <class F>
__device__ __forceinline__ int mx_sbox_op(int x) {
    return (int)((uint32_t)mx_sbox<F>(x) ^ MX_BIAS);
}

// The four planes of one output -> an int32 congruent to it
template <class F>
__device__ __forceinline__ int mx_join(int a0, int a1, int a2, int a3) {
    typedef short s16x2 __attribute__((ext_vector_type(2)));
    const uint32_t t = ((uint32_t)a1 << 8) + (uint32_t)a0;
    const uint32_t u = ((uint32_t)a3 << 8) + (uint32_t)a2;
    const s16x2 k = {(short)-(int)((F::P - 1) >> 16), 1};
    return __builtin_amdgcn_sdot2(__builtin_bit_cast(s16x2, t ^ 0x8000u), k, (int)u, false);
}

// Largest size of an output over `words` inputs: two planes of `words` 4-byte
// words in u, the rounded high half of t, the low half times (p-1)/2^16.
template <class F>
constexpr int64_t mx_bound(int words) {
    const int64_t acc = (int64_t)words * 4 * 128 * 128 + (1 << 16);
    return acc * 257 + (acc * 257 >> 16) + 1 + (int64_t)32768 * ((F::P - 1) >> 16);
}
static_assert(mx_bound<KoalaBear>(16) < KoalaBear::P && mx_bound<BabyBear>(16) < BabyBear::P, "state words in (-p, p)");
static_assert(mx_bound<KoalaBear>(16 + 20) < (1ll << 31) && mx_bound<BabyBear>(16 + 13) < (1ll << 31), "int32");
static_assert(mx_bound<KoalaBear>(24) < (1ll << 31) && mx_bound<BabyBear>(24) < (1ll << 31), "int32");

__device__ __forceinline__ mx16 mx_mma(mx4 a, mx4 b, mx16 c) {
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
}

// The wave's view of the tables in LDS.  Offsets are opaque (`fresh`) inside
// loops: hoisting the table reads would take more registers than there are.
template <class F>
struct MxView {
    const MxTable<F>& t;
    uint32_t ao, co;
    __device__ __forceinline__ explicit MxView(const MxTable<F>& tab)
        : t(tab), ao(16 * (threadIdx.x & 63u)), co(64 * ((threadIdx.x & 63u) >> 5)) {}
    __device__ __forceinline__ void fresh() { asm volatile("" : "+v"(ao), "+v"(co)); }
    __device__ __forceinline__ mx4 A(int k) const {
        return *reinterpret_cast<const mx4*>(reinterpret_cast<const char*>(&t.a[k][0][0]) + ao);
    }
    __device__ __forceinline__ mx16 C(int k) const {
        return *reinterpret_cast<const mx16*>(reinterpret_cast<const char*>(&t.c[k][0][0]) + co);
    }
};

// One linear layer of NS steps on T tiles: x[tile][o] from the operands
// in[tile][step] with blocks base + 2 step + y and bias k.
template <class F, int T, int NS>
__device__ __forceinline__ void mx_layer(int (&x)[T][8], const mx4 (&in)[T][NS], const MxView<F>& v, int base, int k) {
    const mx16 c = v.C(k);
    mx16 y0[T], y1[T];
#pragma unroll
    for (int t = 0; t < T; t++) {
        y0[t] = c;
        y1[t] = mx16{0};
    }
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const mx4 a0 = v.A(base + 2 * s), a1 = v.A(base + 2 * s + 1);
#pragma unroll
        for (int t = 0; t < T; t++) {
            y0[t] = mx_mma(a0, in[t][s], y0[t]);
            y1[t] = mx_mma(a1, in[t][s], y1[t]);
        }
    }
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
        for (int o = 0; o < 8; o++) x[t][o] = mx_join<F>(y0[t][o], y1[t][o], y0[t][8 + o], y1[t][8 + o]);
}

template <class F, int T>
__device__ __forceinline__ void mx_full_sbox(mx4 (&b)[T][2], const int (&x)[T][8]) {
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
        for (int o = 0; o < 8; o++) b[t][o / 4][o % 4] = mx_sbox_op<F>(x[t][o]);
}

// Exchange between the halves: afterwards a holds (a's low half, b's low
// half), b (a's high half, b's high half); its own inverse.
__device__ __forceinline__ void mx_swap(int& a, int& b) {
    const auto r = __builtin_amdgcn_permlane32_swap((unsigned)a, (unsigned)b, false, false);
    a = (int)r[0];
    b = (int)r[1];
}

// The four S-boxes of a block of partial rounds: u the forms over everything
// before the block, x' out
template <class F>
__device__ __forceinline__ void mx_block(int (&u)[4], int rounds) {
    const MxConst<F> k;
#pragma unroll
    for (int o = 0; o < 4; o++) {
        if (o >= rounds) continue;
        int v = u[o];
        if (o > 0) {
            int64_t w = (int64_t)v * k.one + (int64_t)u[o - 1] * k.c1;
            if (o > 1) w += (int64_t)u[o - 2] * k.c2;
            if (o > 2) w += (int64_t)u[o - 3] * k.c3;
            v = mx_redc<F>(w);
        }
        u[o] = mx_sbox<F>(v);
    }
}

// Rounds of the permutation from the first full round's S-boxes to the last
// one's.  In: x = the initial external layer's outputs plus round 0's
// constants.  Out: b = the last S-boxes' outputs as matrix operands (the last
// external layer is left to the caller).
template <class F>
__device__ __forceinline__ void mx_rounds(mx4 (&b)[2][2], int (&x)[2][8], const MxView<F>& v) {
    using S = MxShape<F>;
    mx_full_sbox<F>(b, x);
#pragma unroll
    for (int r = 0; r < 3; r++) {
        mx_layer<F, 2, 2>(x, b, v, S::EXT, S::B_EXT + r);
        mx_full_sbox<F>(b, x);
    }
    mx4 in[2][2 + S::PAIRS];
#pragma unroll
    for (int t = 0; t < 2; t++) {
        in[t][0] = b[t][0];
        in[t][1] = b[t][1];
#pragma unroll
        for (int m = 0; m < S::PAIRS; m++) in[t][2 + m] = mx4{0};
    }
#pragma unroll
    for (int m = 0; m < S::PAIRS; m++) {
        const int base = S::forms(m);
        mx16 f[2];
        f[0] = f[1] = v.C(S::B_FORMS + m);
#pragma unroll
        for (int s = 0; s < 2 + m; s++) {
            const mx4 a = v.A(base + s);
#pragma unroll
            for (int t = 0; t < 2; t++) f[t] = mx_mma(a, in[t][s], f[t]);
        }
#pragma unroll
        for (int beta = 0; beta < 2; beta++) {
            const int rounds = S::RP - 8 * m - 4 * beta;
            if (rounds <= 0) continue;
            if (beta) {
                const mx4 a = v.A(base + 2 + m);
#pragma unroll
                for (int t = 0; t < 2; t++) f[t] = mx_mma(a, in[t][2 + m], f[t]);
            }
            int u[2][2];
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int g = 0; g < 2; g++)
                    u[t][g] = mx_join<F>(f[t][8 * beta + g], f[t][8 * beta + 2 + g], f[t][8 * beta + 4 + g],
                                         f[t][8 * beta + 6 + g]);
            // tile t's forms of rounds 2 h + g sit in half h: gather tile h's
            // four rounds in half h, and put the results back
            mx_swap(u[0][0], u[1][0]);
            mx_swap(u[0][1], u[1][1]);
            int q[4] = {u[0][0], u[0][1], u[1][0], u[1][1]};
            mx_block<F>(q, rounds);
#pragma unroll
            for (int o = 0; o < 4; o++) q[o] = (int)((uint32_t)q[o] ^ MX_BIAS);
            mx_swap(q[0], q[2]);
            mx_swap(q[1], q[3]);
            in[0][2 + m][2 * beta] = q[0];
            in[0][2 + m][2 * beta + 1] = q[1];
            in[1][2 + m][2 * beta] = q[2];
            in[1][2 + m][2 * beta + 1] = q[3];
        }
    }
    mx_layer<F, 2, 2 + S::PAIRS>(x, in, v, S::FINAL, S::B_FINAL);
    mx_full_sbox<F>(b, x);
#pragma unroll
    for (int r = 4; r < 7; r++) {
        mx_layer<F, 2, 2>(x, b, v, S::EXT, S::B_EXT + r);
        mx_full_sbox<F>(b, x);
    }
}

// Whole state (as operand words) -> mx_rounds' input
template <class F>
__device__ __forceinline__ void mx_init(int (&x)[2][8], const mx4 (&st)[2][2], const MxView<F>& v) {
    mx_layer<F, 2, 2>(x, st, v, MxShape<F>::EXT, MxShape<F>::B_INIT);
}
// The last external layer of b and the first of the next permutation, whose
// rate words are `rate` (operand words) -> mx_rounds' input
template <class F>
__device__ __forceinline__ void mx_next(int (&x)[2][8], const mx4 (&rate)[2], const mx4 (&b)[2][2], const MxView<F>& v) {
    using S = MxShape<F>;
    const mx16 c = v.C(S::B_MERGED);
    mx16 y0[2], y1[2];
#pragma unroll
    for (int t = 0; t < 2; t++) {
        y0[t] = c;
        y1[t] = mx16{0};
    }
#pragma unroll
    for (int s = 0; s < 3; s++) {
        const int k = s < 2 ? S::MERGED + 2 * s : S::EXT;
        const mx4 a0 = v.A(k), a1 = v.A(k + 1);
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const mx4 in = s < 2 ? b[t][s < 2 ? s : 0] : rate[t];
            y0[t] = mx_mma(a0, in, y0[t]);
            y1[t] = mx_mma(a1, in, y1[t]);
        }
    }
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int o = 0; o < 8; o++) x[t][o] = mx_join<F>(y0[t][o], y1[t][o], y0[t][8 + o], y1[t][8 + o]);
}
// The last external layer: state words, reduced
template <class F>
__device__ __forceinline__ void mx_last(uint32_t (&st)[2][8], const mx4 (&b)[2][2], const MxView<F>& v) {
    int x[2][8];
    mx_layer<F, 2, 2>(x, b, v, MxShape<F>::EXT, MxShape<F>::B_EXT + 7);
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int o = 0; o < 8; o++) {  // in (-p, p): mx_bound
            const uint32_t r = (uint32_t)x[t][o], s = r + F::P;
            st[t][o] = s < r ? s : r;
        }
}

// ---- device: 16 states per wave ---------------------------------------------
static __device__ const Mx16Table<KoalaBear> kMx16Kb = make_mx16_table<KoalaBear>();
static __device__ const Mx16Table<BabyBear> kMx16Bb = make_mx16_table<BabyBear>();

template <class F>
struct Mx16 {
    using S = Mx16Shape<F>;
    mx4 a[S::NA], c[S::NC][2], f[S::BLOCKS];
    bool q1, q2;  // bits of the lane group q

    __device__ __forceinline__ Mx16() {
        const int lane = threadIdx.x & 63, q = lane >> 4;
        const Mx16Table<F>* t;
        if constexpr (F::P == KoalaBear::P)
            t = &kMx16Kb;
        else
            t = &kMx16Bb;
#pragma unroll
        for (int k = 0; k < S::NA; k++) a[k] = *reinterpret_cast<const mx4*>(&t->a[k][lane][0]);
#pragma unroll
        for (int k = 0; k < S::NC; k++)
#pragma unroll
            for (int p = 0; p < 2; p++) c[k][p] = *reinterpret_cast<const mx4*>(&t->c[k][p][4 * q]);
#pragma unroll
        for (int b = 0; b < S::BLOCKS; b++) f[b] = *reinterpret_cast<const mx4*>(&t->f[b][4 * q]);
        q1 = q & 1;
        q2 = q & 2;
    }
    static __device__ __forceinline__ mx4 mma(mx4 x, mx4 y, mx4 z) {
        return __builtin_amdgcn_mfma_i32_16x16x64_i8(x, y, z, 0, 0, 0);
    }
    // operand word of a state word
    static __device__ __forceinline__ mx4 op(mx4 w) { return w ^ (int)MX_BIAS; }

    // one linear layer of NS steps: this lane's four outputs
    template <int NS>
    __device__ __forceinline__ mx4 layer(const mx4 (&in)[NS], int base, int k) const {
        mx4 y[4] = {c[k][0], mx4{0}, c[k][1], mx4{0}};
#pragma unroll
        for (int s = 0; s < NS; s++)
#pragma unroll
            for (int p = 0; p < 4; p++) y[p] = mma(a[base + 4 * s + p], in[s], y[p]);
        mx4 x;
#pragma unroll
        for (int i = 0; i < 4; i++) x[i] = mx_join<F>(y[0][i], y[1][i], y[2][i], y[3][i]);
        return x;
    }
    static __device__ __forceinline__ mx4 sbox(mx4 x) {
#pragma unroll
        for (int i = 0; i < 4; i++) x[i] = mx_sbox_op<F>(x[i]);
        return x;
    }
    // The permutation: operand words of the state in, state words (any int32) out
    __device__ __forceinline__ mx4 permute(mx4 st) const {
        mx4 in[S::STEPS];
        {
            const mx4 one[1] = {st};
            in[0] = sbox(layer<1>(one, S::EXT, 0));
        }
#pragma unroll
        for (int r = 1; r < 4; r++) {
            const mx4 one[1] = {in[0]};
            in[0] = sbox(layer<1>(one, S::EXT, r));
        }
#pragma unroll
        for (int s = 1; s < S::STEPS; s++) in[s] = mx4{0};
#pragma unroll
        for (int b = 0; b < S::BLOCKS; b++) {
            mx4 y = mma(a[S::forms(b)], in[0], f[b]);
            if (b) y = mma(a[S::forms(b) + 1], in[1], y);
            // group q holds form q: give every group all four
            const unsigned u = (unsigned)mx_join<F>(y[0], y[1], y[2], y[3]);
            const auto h = __builtin_amdgcn_permlane32_swap(u, u, false, false);
            const auto lo = __builtin_amdgcn_permlane16_swap(h[0], h[0], false, false);
            const auto hi = __builtin_amdgcn_permlane16_swap(h[1], h[1], false, false);
            int w[4] = {(int)lo[0], (int)lo[1], (int)hi[0], (int)hi[1]};
            mx_block<F>(w, S::RP - 4 * b);
            // all four are made in every lane: the compiler would move some under the
            // selects' conditions, as branches
            asm("" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3]));
            in[1 + b / 4][b % 4] = (int)((uint32_t)(q1 ? (q2 ? w[3] : w[1]) : (q2 ? w[2] : w[0])) ^ MX_BIAS);
        }
        in[0] = sbox(layer<S::STEPS>(in, S::FINAL, 4));
#pragma unroll
        for (int r = 5; r < 8; r++) {
            const mx4 one[1] = {in[0]};
            in[0] = sbox(layer<1>(one, S::EXT, r));
        }
        const mx4 one[1] = {in[0]};
        return layer<1>(one, S::EXT, 8);
    }
};
// state words of a permutation, reduced
template <class F>
__device__ __forceinline__ u32x4 mx16_words(mx4 x) {
    u32x4 w;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t r = (uint32_t)x[i], s = r + F::P;
        w[i] = s < r ? s : r;
    }
    return w;
}

}  // namespace pg
