// f32 products on the bf16 matrix cores, by an exact three-way split (the method of
// Henry, Tang and Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype
// For Higher-Precision Computations", ARITH 2019).
//
// v_mfma_f32_16x16x4_f32 peaks at 157 TFLOP/s on gfx950 and, as measured here,
// shares the SIMD with the vector ALU; v_mfma_f32_16x16x32_bf16 runs at 16
// times that rate: 2.24 PFLOP/s measured with two waves per SIMD on the parts of N(0, 1)
// values (2.48 on zeros: power), 1.87 with two vector instructions beside each MFMA,
// 1.58 with four.  So an f32 operand x is written as
// x = h + m + l, three bf16 values of 8 significant bits each (h = bf16(x), m =
// bf16(x - h), l = x - h - m: together all 24 bits of x, both subtractions
// exact), and a product as the six partial products above 2^-24 of it,
//   h h' + (h m' + m h') + (m m' + h l' + l h'),
// each exact in the f32 accumulator's input; the dropped m l' + l m' + l l' is
// at most 2^-24 and typically 2^-27 of the product.  Six MFMAs at 16 times the
// rate: 2.6 times the f32 MFMA's.  Every sum is still an f32 sum.  Error
// against 64-bit sums for N(0, 1) operands over K terms, f32 MFMA chain / six
// products in one chain / six products per 32 terms then one f32 add:
//   K = 128   2.1e-7 / 1.5e-7 / 5.7e-8
//   K = 512   4.0e-7 / 3.4e-7 / 8.8e-8
//   K = 4096  1.1e-6 / 1.0e-6 / 2.2e-7
// (fewer roundings of the long accumulator), so a chain of at most 256 terms
// accumulates in the MFMA and a longer one adds 32-term sums on the vector ALU.
//
// Range, below: bf16's smallest bit is 2^-133 and f32's 2^-149, so l loses bits of
// an x under 2^-110 (the error of a product against 64-bit sums, 2.0e-7 on f32 MFMAs,
// was 2.2e-6 with an operand of 2^-116 and 5.7e-4 at 2^-124).  Operands are
// therefore split as 2^16 x (split8), which makes the split exact for denormal
// values too (the conversion and the MFMA keep bf16 denormals; 5.6e-8 at every
// scale), and the f32 add that takes a sum of products into its accumulator is a
// multiply-add with 2^-32.  Scores and softmax weights are split without the
// factor (split8_as_is), since only their absolute error counts: the exponential
// sees the scores', under 2^-80, and the weights', 2^-134, is below the 2^-126 under
// which the exponential returns 0.  (With it on the weights 333 rows over 2340
// keys, 32 over 8 heads, d = 128, took 131 us instead of 128.)
// What the factor costs (us, without / with): nothing in the forward; 32 over 8
// heads, d = 128, T = 4096, dk/dv 1515 / 1531, dq product 439 / 445; MHA d = 64, 4 x 1024
// rows x 8 heads, dk/dv 82.9 / 85.6.
//
// Range, above: an operand of magnitude 2^40 or more, infinities among them, could
// overflow so scaled or turn into NaN in the split (inf - inf), so it enters the split
// as 0 and its products are added by f32 MFMAs from the full value ("big"
// below; NaN needs no care, every part of it is NaN).  Kernels flag a staged
// tile that holds one, and only flagged tiles take that slow path; elements
// that are not big keep the same arithmetic, bit for bit, with or without one
// beside them (but where both operands of a tile hold one, the whole tile's
// product is formed in f32).
#pragma once
#include "common.h"
#include "shapes.h"
#include <utility>

typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef unsigned u2 __attribute__((ext_vector_type(2)));
typedef unsigned u4 __attribute__((ext_vector_type(4)));
typedef short s4i __attribute__((ext_vector_type(4)));

constexpr int kSplitExp = 16;         // a split operand is 2^16 x
constexpr float kUnscale = 0x1p-32f;  // takes that back off a product of two
constexpr float kUnscale1 = 0x1p-16f; // off a product with one operand as it is
constexpr float kBig = 0x1p40f;       // 256 products of such operands, scaled: 2^120

// x again, as a value the compiler knows nothing about: what a rarely taken
// branch computes from it stays in the branch instead of being hoisted out of
// the loop around it into registers the loop needs.
DEVI int opaque(int x) {
    asm volatile("" : "+v"(x));
    return x;
}

// Eight f32 values split: an MFMA operand's eight consecutive k slots.
struct Tri {
    u4 h, m, l;
};

// Two f32 rounded to bf16 (nearest even, v_cvt_pk_bf16_f32), x0 in the low half.
DEVI unsigned pack_bf16(float x0, float x1) {
    return __builtin_bit_cast(unsigned, __builtin_convertvector((f2{x0, x1}), bf2));
}
DEVI void split2(float x0, float x1, unsigned &h, unsigned &m, unsigned &l) {
    h = pack_bf16(x0, x1);
    x0 -= __uint_as_float(h << 16);
    x1 -= __uint_as_float(h & 0xffff0000u);
    m = pack_bf16(x0, x1);
    x0 -= __uint_as_float(m << 16);
    x1 -= __uint_as_float(m & 0xffff0000u);
    l = pack_bf16(x0, x1);
}
DEVI float scale_up(float x) { return __builtin_amdgcn_ldexpf(x, kSplitExp); }  // (an inline constant: no register)
DEVI Tri split8_as_is(const float (&x)[8]) {
    Tri t;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        unsigned h, m, l;
        split2(x[2 * i], x[2 * i + 1], h, m, l);
        t.h[i] = h; t.m[i] = m; t.l[i] = l;
    }
    return t;
}

DEVI Tri split8(const float (&x)[8]) {
    float y[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = scale_up(x[i]);
    return split8_as_is(y);
}

// The f32 value whose parts are in the low (hi = 0) or high halves of h, m, l.
DEVI float join_bf16(unsigned h, unsigned m, unsigned l, int hi) {
    const int sh = hi ? 0 : 16;
    const auto part = [&](unsigned x) { return __uint_as_float((x << sh) & 0xffff0000u); };
    return part(h) + part(m) + part(l);
}

// max(m, |a|, |b|); a NaN counts as nothing.
DEVI float vmax3_abs(float m, float a, float b) {
    float r;
    asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(r) : "v"(m), "v"(a), "v"(b));
    return r;
}
template <int N>
DEVI float max_abs(const float (&x)[N], float m = 0.f) {
    static_assert(N % 2 == 0, "pairs");
#pragma unroll
    for (int i = 0; i < N; i += 2) m = vmax3_abs(m, x[i], x[i + 1]);
    return m;
}
// Whether any lane of the wave holds a big value (wave-uniform).
DEVI bool any_big(float max_abs_of_lane) { return __builtin_amdgcn_ballot_w64(max_abs_of_lane >= kBig) != 0; }
DEVI float big_part(float x) { return __builtin_fabsf(x) >= kBig ? x : 0.f; }
DEVI float small_part(float x) { return __builtin_fabsf(x) >= kBig ? 0.f : x; }

DEVI f4 mfma_bf16(u4 a, u4 b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, a), __builtin_bit_cast(bf8, b), c, 0, 0, 0);
}

// The partial products that take part C (0 = l, 1 = m, 2 = h) of an operand
// `a` streamed from LDS, against the parts of N operands b(n) held in
// registers, the N chains interleaved: l h', m m', m h', h l', h m', h h' in
// the order of the parts -- smallest first, nearly.
template <int C, int N, class B>
DEVI void mfma_parts(f4 (&c)[N], u4 a, B b) {
    if constexpr (C == 2) {
#pragma unroll
        for (int n = 0; n < N; ++n) c[n] = mfma_bf16(a, b(n).l, c[n]);
    }
    if constexpr (C >= 1) {
#pragma unroll
        for (int n = 0; n < N; ++n) c[n] = mfma_bf16(a, b(n).m, c[n]);
    }
#pragma unroll
    for (int n = 0; n < N; ++n) c[n] = mfma_bf16(a, b(n).h, c[n]);
}

// Runs step(i, part, operand) for i = 0..STEPS-1 and the parts l, m, h of each,
// the operand parts read by load(i, part) RING - 1 parts ahead: 4 RING
// registers instead of the 24 that two whole operands take, and still 100 cycles
// or more of MFMAs between a read and its use.  The scheduling fences keep the
// reads where they are put.
template <int STEPS, int RING, class Load, class Step>
DEVI void stream_parts(Load load, Step step) {
    u4 ring[RING];
#pragma unroll
    for (int k = 0; k < RING - 1; ++k) ring[k] = load(k / 3, k % 3);
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
        [&]<int... C>(std::integer_sequence<int, C...>) {
            ((
                 [&] {
                     const int k = 3 * i + C;
                     if (k + RING - 1 < 3 * STEPS)
                         ring[(k + RING - 1) % RING] = load((k + RING - 1) / 3, (k + RING - 1) % 3);
                     step(i, std::integral_constant<int, C>{}, ring[k % RING]);
                     __builtin_amdgcn_sched_barrier(0);
                 }()),
             ...);
        }(std::make_integer_sequence<int, 3>{});
    }
}

template <int DP>
DEVI void put_tri(char *tile, int rows, int row, int col, const Tri &t) {  // col a multiple of 8
    char *p = tile + row * split_stride(DP) + 2 * col;
    *reinterpret_cast<u4 *>(p) = t.h;
    *reinterpret_cast<u4 *>(p + rows * split_stride(DP)) = t.m;
    *reinterpret_cast<u4 *>(p + 2 * rows * split_stride(DP)) = t.l;
}
// Part C (0 = l, 1 = m, 2 = h) of an operand with the contraction along the row:
// lane l16 = row, k slot 8 grp + j = column c0 + 8 grp + j.
template <int DP>
DEVI u4 get_row(const char *tile, int rows, int row0, int c0, int l16, int grp, int part) {
    return *reinterpret_cast<const u4 *>(tile + ((2 - part) * rows + row0 + l16) * split_stride(DP) + 2 * (c0 + 8 * grp));
}
// gfx950's transposing LDS read: 16 lanes read four rows of 16 values (lane i
// at row i / 4, values 4 (i % 4)) and lane i gets column i of the four.
DEVI u2 lds_tr16(const char *p) {
    typedef __attribute__((address_space(3))) s4i lds_s4;
    return __builtin_bit_cast(u2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4 *)p));
}
// Part C of an operand with the contraction across the rows: lane l16 = column
// c0 + l16, k slot 8 grp + j = row r0 + 4 grp + j for j < 4, row r0 + 16 + 4 grp + j
// - 4 for j >= 4 -- the slots in which two 16 x 16 C tiles (rows r0.., r0 + 16..)
// hold their rows, so a C tile pair split by split8 is the other operand as it stands.
template <int DP>
DEVI u4 get_col(const char *tile, int rows, int r0, int c0, int lane, int part) {
    const int i = lane & 15, grp = lane >> 4;
    constexpr int S = split_stride(DP);
    const char *p = tile + ((2 - part) * rows + r0 + 4 * grp + (i >> 2)) * S + 2 * (c0 + 4 * (i & 3));
    const u2 x = lds_tr16(p), y = lds_tr16(p + 16 * S);
    return u4{x.x, x.y, y.x, y.y};
}
