// BLS12-381 scalar field in a radix-2^29 form, for the inner loops of the sumcheck round kernels on gfx950.
//
// A value is 9 limbs: limbs 0..7 in [0, 2^29), limb 8 takes what is left (non-negative in everything below).  The limbs
// are those of the integer itself: a tensor element (8 x 32-bit words, fr-tensor.cu:181-184) is repacked by shifts, with
// no multiplication.  A product is a Montgomery product with radix 2^261, fr29_mul(a, b) = a b 2^-261 mod r, so one
// operand of every product carries the factor 2^261 (the challenges, converted once per lane) or the result's scale is
// accounted for at the end (the eq weights, which arrive with 2^256).
//
// Why: with 29-bit limbs a column of the schoolbook product (9 products below 2^58) fits a 64-bit accumulator, so a limb
// product is ONE v_mad_u64_u32 with no add-with-carry behind it and no carry flag to wait for; r = 1 mod 2^29, so the
// reduction's multiplier is the low limb or its negative (no product, fr29_redc), and its result needs no conditional subtraction.  About 220
// vector instructions per product against 370 in the 32-bit form (field.hpp: 120 multiply-adds, 120 add-with-carry, 130
// others), and a product that is only summed (Wide29) costs its 81 multiply-adds and a share of a carry pass.
#pragma once
#include "field.hpp"

namespace zk {

struct Fr29 { int32_t l[9]; };
static constexpr uint32_t R29M = (1u << 29) - 1u;

ZK_HD constexpr int32_t fr29_p(int i) {                 // r
    constexpr int32_t t[9] = {1, 536870904, 529989567, 457704959, 494949691, 201589968, 354471143, 174404527, 7597479};
    return t[i];
}
ZK_HD constexpr int32_t fr29_n(int i) {                 // ((2^29 - 1) r + 1) / 2^29
    constexpr int32_t t[9] = {9, 6881336, 72284608, 499626180, 293359722, 383989737, 180066615, 166807048, 7597479};
    return t[i];
}
ZK_HD Fr29 fr29_const(const int32_t (&t)[9]) {
    Fr29 r;
#pragma unroll
    for (int i = 0; i < 9; ++i) r.l[i] = t[i];
    return r;
}
ZK_HD Fr29 fr29_r() { constexpr int32_t t[9] = {1, 536870904, 529989567, 457704959, 494949691, 201589968, 354471143, 174404527, 7597479}; return fr29_const(t); }
ZK_HD Fr29 fr29_2_261() { constexpr int32_t t[9] = {536870842, 559, 481694080, 172907520, 250130850, 384216799, 419952827, 139714039, 5047359}; return fr29_const(t); }     // 2^261 mod r
ZK_HD Fr29 fr29_2_527() { constexpr int32_t t[9] = {238450677, 105123874, 285095421, 524243062, 304996105, 406999561, 483795002, 430521147, 293893}; return fr29_const(t); }     // 2^527 mod r
ZK_HD Fr29 fr29_2_266() { constexpr int32_t t[9] = {536868651, 18087, 526333248, 216203804, 294598241, 8484555, 89016444, 271483280, 1968430}; return fr29_const(t); }     // 2^266 mod r
ZK_HD Fr29 fr29_2_271() { constexpr int32_t t[9] = {536798552, 578879, 254716416, 35656607, 98837070, 269398762, 12757061, 312906888, 2209941}; return fr29_const(t); }     // 2^271 mod r
ZK_HD Fr29 fr29_2_522() { constexpr int32_t t[9] = {175223744, 489824382, 375642521, 475708563, 62229572, 199455800, 136968049, 375395230, 2620817}; return fr29_const(t); }   // 2^522 mod r
ZK_HD Fr29 fr29_2_532() { constexpr int32_t t[9] = {114228895, 142738518, 3129318, 211945681, 138120195, 474365025, 94583408, 180499405, 1807122}; return fr29_const(t); }     // 2^532 mod r
ZK_HD Fr29 fr29_zero() {
    Fr29 r;
#pragma unroll
    for (int i = 0; i < 9; ++i) r.l[i] = 0;
    return r;
}

// Montgomery reduction interleaved with the columns: col(k), k = 0..17, is the k-th column of the value to reduce (a product:
// columns 0..16; a Wide29 sum: 18 limbs).  Returns value * 2^-261 mod r as a non-negative integer below value / 2^261 + (1 + 2^-29) r.
// The first seven limbs go by N = (2^29 - 1) r, which ends in -1: the multiple of N that clears a limb is the limb itself, and what it adds to the columns
// above is fr29_n, with nothing to negate and nothing to add to the column.  N is 2^29 times r, so the last two limbs go by r: the seven add less than 2^(29 * 7) N = 2^-29 2^261 r.
// All nine by r: a lookup of 2^22 queries took 491 us instead of 483, an attention head of 2048 tokens 3.16 ms instead of 3.13 (medians of four).
template <int NCOL, typename Col> ZK_HD Fr29 fr29_redc(Col col) {
    constexpr int FAST = 7;
    int32_t m[9];
    Fr29 t;
    int64_t carry = 0;
#pragma unroll
    for (int k = 0; k < 9; ++k) {
        int64_t q = carry;
#pragma unroll
        for (int i = 0; i < k; ++i) q += (int64_t)m[i] * (i < FAST ? fr29_n(k - i - 1) : fr29_p(k - i));
        q += col(k);
        if (k < FAST) m[k] = (int32_t)((uint32_t)q & R29M);
        else {
            m[k] = (int32_t)((0u - (uint32_t)q) & R29M);   // r = 1 mod 2^29: -r^-1 = -1
            q += (int64_t)m[k];
        }
        carry = q >> 29;
    }
#pragma unroll
    for (int k = 9; k < 18; ++k) {
        int64_t q = carry;
#pragma unroll
        for (int i = k - 9; i < 9; ++i) {
            if (i < FAST) q += (int64_t)m[i] * fr29_n(k - i - 1);
            else if (i > k - 9) q += (int64_t)m[i] * fr29_p(k - i);
        }
        if (k < NCOL) q += col(k);
        if (k < 17) {
            t.l[k - 9] = (int32_t)((uint32_t)q & R29M);
            carry = q >> 29;
        } else {
            t.l[8] = (int32_t)q;
        }
    }
    return t;
}
// a b 2^-261 mod r; limbs 0..7 of both below 2^29, limb 8 below 2^30, a b below 2^523.  Result below a b / 2^261 + (1 + 2^-29) r, limbs normalised.
ZK_HD Fr29 fr29_mul(const Fr29& a, const Fr29& b) {
    return fr29_redc<17>([&](int k) {
        int64_t s = 0;
#pragma unroll
        for (int i = 0; i < 9; ++i)
            if (k - i >= 0 && k - i < 9) s += (int64_t)a.l[i] * b.l[k - i];
        return s;
    });
}
// a k 2^-58 mod r for a small k = k0 + k1 2^29 (two limbs: any k below 2^58): a Montgomery product with radix 2^58 -- eighteen
// limb products for a k and eighteen for the two reduction steps, against 162 of fr29_mul.  a as for fr29_mul (limb 8 below
// 2^30); the result is non-negative and below a k / 2^58 + r, limbs normalised.
ZK_HD Fr29 fr29_mul_small(const Fr29& a, uint32_t k0, uint32_t k1) {
    Fr29 t;
    auto col = [&](int j) {
        int64_t s = 0;
        if (j < 9) s += (int64_t)a.l[j] * (int64_t)k0;
        if (j >= 1) s += (int64_t)a.l[j - 1] * (int64_t)k1;
        return s;
    };
    int64_t q = col(0);
    const int32_t m0 = (int32_t)((0u - (uint32_t)q) & R29M);      // r = 1 mod 2^29
    q += (int64_t)m0;
    int64_t carry = q >> 29;
    q = carry + col(1) + (int64_t)m0 * fr29_p(1);
    const int32_t m1 = (int32_t)((0u - (uint32_t)q) & R29M);
    q += (int64_t)m1;
    carry = q >> 29;
#pragma unroll
    for (int j = 2; j <= 10; ++j) {
        q = carry;
        if (j <= 9) q += col(j);
        if (j <= 8) q += (int64_t)m0 * fr29_p(j);
        if (j - 1 <= 8) q += (int64_t)m1 * fr29_p(j - 1);
        if (j < 10) {
            t.l[j - 2] = (int32_t)((uint32_t)q & R29M);
            carry = q >> 29;
        } else {
            t.l[8] = (int32_t)q;
        }
    }
    return t;
}
// x mod r for an integer of magnitude below 2^58, canonical (x itself, or r - |x|)
ZK_HD Fr29 fr29_from_small(int64_t x) {
    Fr29 t = fr29_r();
    const bool ng = x < 0;
    const uint64_t y = ng ? 0ull - (uint64_t)x : (uint64_t)x;
    const int32_t y0 = (int32_t)((uint32_t)y & R29M), y1 = (int32_t)((uint32_t)(y >> 29) & R29M);
    if (ng) {
        const int32_t s0 = t.l[0] - y0;
        t.l[0] = (int32_t)((uint32_t)s0 & R29M);
        const int32_t s1 = t.l[1] - y1 + (s0 >> 29);
        t.l[1] = (int32_t)((uint32_t)s1 & R29M);
        t.l[2] += s1 >> 29;                                 // limb 2 of r is far above 1: no further borrow
    } else {
#pragma unroll
        for (int i = 2; i < 9; ++i) t.l[i] = 0;
        t.l[0] = y0;
        t.l[1] = y1;
    }
    return t;
}
// limb-wise with a carry pass; the results are non-negative where the value is
ZK_HD Fr29 fr29_add(const Fr29& a, const Fr29& b) {
    Fr29 r;
    int32_t c = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int32_t s = a.l[i] + b.l[i] + c;
        r.l[i] = (int32_t)((uint32_t)s & R29M);
        c = s >> 29;
    }
    r.l[8] = a.l[8] + b.l[8] + c;
    return r;
}
// a - b + r: non-negative for b <= a + r (both canonical: a value in (0, 2r))
ZK_HD Fr29 fr29_sub_plus_r(const Fr29& a, const Fr29& b) {
    Fr29 r;
    int32_t c = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int32_t s = a.l[i] - b.l[i] + fr29_p(i) + c;
        r.l[i] = (int32_t)((uint32_t)s & R29M);
        c = s >> 29;
    }
    r.l[8] = a.l[8] - b.l[8] + fr29_p(8) + c;
    return r;
}
// a - b + 3 r: non-negative for b < 3 r (operands that are sums of a canonical value and a product, below 2.1 r)
ZK_HD Fr29 fr29_sub_plus_3r(const Fr29& a, const Fr29& b) {
    Fr29 r;
    int32_t c = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int32_t s = a.l[i] - b.l[i] + 3 * fr29_p(i) + c;
        r.l[i] = (int32_t)((uint32_t)s & R29M);
        c = s >> 29;
    }
    r.l[8] = a.l[8] - b.l[8] + 3 * fr29_p(8) + c;
    return r;
}
// the same integer in 29-bit limbs (any 256-bit value)
ZK_HD Fr29 fr29_repack(const Big<8>& a) {
    Fr29 r;
#pragma unroll
    for (int i = 0; i < 9; ++i) {
        const int off = 29 * i, w = off >> 5, sh = off & 31;
        uint32_t v = a.v[w] >> sh;
        if (sh > 3 && w + 1 < 8) v |= a.v[w + 1] << (32 - sh);
        r.l[i] = (int32_t)(i < 8 ? (v & R29M) : v);
    }
    return r;
}
// canonical residue of a non-negative value below (PASSES + 1) r
template <int PASSES = 2> ZK_HD Fr29 fr29_canon(const Fr29& a) {
    Fr29 v = a;
#pragma unroll
    for (int pass = 0; pass < PASSES; ++pass) {
        Fr29 t;
        int32_t c = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int32_t s = v.l[i] - fr29_p(i) + c;
            t.l[i] = (int32_t)((uint32_t)s & R29M);
            c = s >> 29;
        }
        t.l[8] = v.l[8] - fr29_p(8) + c;
        if (t.l[8] >= 0) v = t;
    }
    return v;
}
// a canonical value as 8 x 32-bit words
ZK_HD Big<8> fr29_pack(const Fr29& v) {
    Big<8> r;
#pragma unroll
    for (int w = 0; w < 8; ++w) {
        const int off = 32 * w, i = off / 29, sh = off % 29;
        uint64_t x = (uint64_t)(uint32_t)v.l[i] >> sh;
        if (i + 1 < 9) x |= (uint64_t)(uint32_t)v.l[i + 1] << (29 - sh);
        if (i + 2 < 9) x |= (uint64_t)(uint32_t)v.l[i + 2] << (58 - sh);
        r.v[w] = (uint32_t)x;
    }
    return r;
}
template <int PASSES = 2> ZK_HD Big<8> fr29_canon_pack(const Fr29& a) { return fr29_pack(fr29_canon<PASSES>(a)); }
// a b mod r, canonical, for any two 256-bit integers: Barrett's reduction on the limbs of the whole product t.  With t1 the limbs of t
// from the eighth on and mu = floor(2^522 / r), q = floor(t1 mu / 2^290) without the columns below the eighth is floor(t / r) or one
// less: what the low limbs of t, the fraction of mu and the dropped columns add to t / r stays below 2^-9.  So t - q r, of which only
// the nine low limbs are formed, lies below 2 r.  190 limb products, where two Montgomery products (a b, then times 2^512) take 240
// with as many add-with-carry: 8.4 M products (805 MB) stream in 137 us = 5.9 TB/s against 163.
ZK_HD Big<8> fr_mul_barrett(const Big<8>& x, const Big<8>& y) {
    constexpr int32_t mu[10] = {361647168, 255869313, 225526387, 363197021, 349782287, 235913501, 59465163, 527375294, 356668343, 70};
    const Fr29 a = fr29_repack(x), b = fr29_repack(y);
    int32_t t[18], q[9];
    uint64_t s = 0;
#pragma unroll
    for (int k = 0; k < 17; ++k) {
#pragma unroll
        for (int i = 0; i < 9; ++i)
            if (k - i >= 0 && k - i < 9) s += (uint64_t)(uint32_t)a.l[i] * (uint32_t)b.l[k - i];
        t[k] = (int32_t)((uint32_t)s & R29M);
        s >>= 29;
    }
    t[17] = (int32_t)s;
    s = 0;
#pragma unroll
    for (int k = 8; k < 19; ++k) {
#pragma unroll
        for (int i = 0; i < 10; ++i)
            if (k - i >= 0 && k - i < 10) s += (uint64_t)(uint32_t)t[8 + i] * (uint32_t)mu[k - i];
        if (k >= 10) q[k - 10] = (int32_t)((uint32_t)s & R29M);
        s >>= 29;
    }
    Fr29 v;
    int64_t c = 0;
#pragma unroll
    for (int k = 0; k < 9; ++k) {
        c += t[k] - q[k];                                   // r = 1 mod 2^29
#pragma unroll
        for (int i = 0; i < k; ++i) c -= (int64_t)q[i] * fr29_p(k - i);
        v.l[k] = (int32_t)((uint32_t)c & R29M);
        c >>= 29;
    }
    return fr29_pack(fr29_canon<1>(v));
}

// A sum of products that is reduced once.  Columns 0..16 take the limb products of every term, column 17 what carries out of
// them; the operands' limbs are non-negative, so a column grows by less than 9 * 2^58 per term and wide29_carry must run at
// least every FOUR terms (4 * 9 * 2^58 + 2^29 < 2^64).  The whole sum must stay below 2^522 (18 limbs).
struct Wide29 { uint64_t c[18]; };
ZK_HD Wide29 wide29_zero() {
    Wide29 w;
#pragma unroll
    for (int i = 0; i < 18; ++i) w.c[i] = 0;
    return w;
}
ZK_HD void wide29_mac(Wide29& w, const Fr29& a, const Fr29& b) {
#pragma unroll
    for (int k = 0; k < 17; ++k) {
        uint64_t s = w.c[k];
#pragma unroll
        for (int i = 0; i < 9; ++i)
            if (k - i >= 0 && k - i < 9) s += (uint64_t)(uint32_t)a.l[i] * (uint32_t)b.l[k - i];
        w.c[k] = s;
    }
}
ZK_HD void wide29_carry(Wide29& w) {
#pragma unroll
    for (int k = 0; k < 17; ++k) {
        w.c[k + 1] += w.c[k] >> 29;
        w.c[k] &= (uint64_t)R29M;
    }
}
// sum * 2^-261 mod r, below sum / 2^261 + (1 + 2^-29) r (the carry pass runs first: every column below 2^29 but the last)
ZK_HD Fr29 wide29_redc(Wide29& w) {
    wide29_carry(w);
    return fr29_redc<18>([&](int k) { return (int64_t)w.c[k]; });
}

#if defined(__HIPCC__)
// ---- sums over lanes -----------------------------------------------------------------------------------------------------
template <int CTRL, int ROWS = 0xF> __device__ __forceinline__ uint32_t dpp_plus(uint32_t x) {
    return x + (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, ROWS, 0xF, false);
}
__device__ __forceinline__ void fr29_carry_u(uint32_t (&l)[9]) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        l[i + 1] += l[i] >> 29;
        l[i] &= R29M;
    }
}
// limb-wise sums over the rows of sixteen lanes (every lane of the wave active), in each row's last lane; limbs 0..7 below 2^29
__device__ __forceinline__ void fr29_row_sum(uint32_t (&l)[9]) {
#pragma unroll
    for (int i = 0; i < 9; ++i) l[i] = dpp_plus<0x112>(dpp_plus<0x111>(l[i]));      // one, then two lanes to the left
    fr29_carry_u(l);
#pragma unroll
    for (int i = 0; i < 9; ++i) l[i] = dpp_plus<0x118>(dpp_plus<0x114>(l[i]));      // four, eight
    fr29_carry_u(l);
}
// and over the wave, in its last lane
__device__ __forceinline__ void fr29_wave_sum(uint32_t (&l)[9]) {
    fr29_row_sum(l);
#pragma unroll
    for (int i = 0; i < 9; ++i) l[i] = dpp_plus<0x143, 0xC>(dpp_plus<0x142, 0xA>(l[i]));      // row 0 into 1, 2 into 3, then the lower half into the upper
    fr29_carry_u(l);
}

// ---- sums over a workgroup that are reduced once -------------------------------------------------------------------------
// A lane's sums stay integers in 29-bit limbs while they are added up over the lanes; the residues are taken of the workgroup's sums, a lane
// a sum in one of its waves.  (Reduced a lane first, the five sums of a round took 4000 instructions a wave, what two pairs cost.)
static constexpr int RAW_LIMBS = 19;                      // 2^522 a lane, 256 lanes
// the wave's sum of N limbs (the top one small enough for 64 of it) to slot; every lane of the wave active
template <int N> __device__ __forceinline__ void raw_wave_sum(uint32_t (&l)[N], uint32_t* slot) {
    auto carry = [&]() {
#pragma unroll
        for (int i = 0; i < N - 1; ++i) {
            l[i + 1] += l[i] >> 29;
            l[i] &= R29M;
        }
    };
#pragma unroll
    for (int i = 0; i < N; ++i) l[i] = dpp_plus<0x112>(dpp_plus<0x111>(l[i]));
    carry();
#pragma unroll
    for (int i = 0; i < N; ++i) l[i] = dpp_plus<0x118>(dpp_plus<0x114>(l[i]));
    carry();
#pragma unroll
    for (int i = 0; i < N; ++i) l[i] = dpp_plus<0x143, 0xC>(dpp_plus<0x142, 0xA>(l[i]));
    carry();
    if ((threadIdx.x & 63u) == 63u) {
#pragma unroll
        for (int i = 0; i < RAW_LIMBS; ++i) slot[i] = i < N ? l[i] : 0u;
    }
}
__device__ __forceinline__ void raw_put(Wide29& w, uint32_t* slot) {      // below 2^522
    wide29_carry(w);
    uint32_t l[19];
#pragma unroll
    for (int i = 0; i < 18; ++i) l[i] = (uint32_t)w.c[i];
    l[18] = 0u;
    raw_wave_sum(l, slot);
}
__device__ __forceinline__ void raw_put(const uint32_t (&words)[9], uint32_t* slot) {      // a sum of up to 2^12 elements as nine 32-bit words
    uint32_t l[10];
#pragma unroll
    for (int i = 0; i < 10; ++i) {
        const int off = 29 * i, w = off >> 5, sh = off & 31;
        uint32_t v = words[w] >> sh;
        if (sh > 3 && w + 1 < 9) v |= words[w + 1] << (32 - sh);
        l[i] = i < 9 ? v & R29M : v;
    }
    raw_wave_sum(l, slot);
}
__device__ __forceinline__ void raw_put(const Fr29& x, uint32_t* slot) {      // limb 8 below 2^31
    uint32_t l[10];
#pragma unroll
    for (int i = 0; i < 9; ++i) l[i] = (uint32_t)x.l[i];
    l[9] = l[8] >> 29;
    l[8] &= R29M;
    raw_wave_sum(l, slot);
}
// V fix 2^-522 mod r, canonical, of a workgroup's sum V; slot: its first wave's, the others' `stride` words apart
template <int WAVES> __device__ __forceinline__ Fr raw_residue(const uint32_t* slot, uint32_t stride, const Fr29& fix) {
    uint32_t v[RAW_LIMBS];
#pragma unroll
    for (int i = 0; i < RAW_LIMBS; ++i) {
        v[i] = slot[i];
#pragma unroll
        for (int w = 1; w < WAVES; ++w) v[i] += slot[(uint32_t)w * stride + i];
    }
#pragma unroll
    for (int i = 0; i < RAW_LIMBS - 1; ++i) {
        v[i + 1] += v[i] >> 29;
        v[i] &= R29M;
    }
    const Fr29 top = fr29_2_522();
    const Fr29 t = fr29_redc<18>([&](int k) { return (int64_t)v[k] + (k < 9 ? (int64_t)v[18] * top.l[k < 9 ? k : 0] : 0); });
    return fr29_canon_pack<3>(fr29_mul(t, fix));
}

// ---- elements in LDS: twelve words each, so that rows of sixteen lanes read without bank conflicts ------------------------
__device__ __forceinline__ void rm_put(int32_t* slot, const Fr29& x) {
    int4* p = reinterpret_cast<int4*>(slot);
    p[0] = make_int4(x.l[0], x.l[1], x.l[2], x.l[3]);
    p[1] = make_int4(x.l[4], x.l[5], x.l[6], x.l[7]);
    slot[8] = x.l[8];
}
__device__ __forceinline__ Fr29 rm_get(const int32_t* slot) {
    const int4* p = reinterpret_cast<const int4*>(slot);
    const int4 a = p[0], b = p[1];
    Fr29 x;
    x.l[0] = a.x; x.l[1] = a.y; x.l[2] = a.z; x.l[3] = a.w;
    x.l[4] = b.x; x.l[5] = b.y; x.l[6] = b.z; x.l[7] = b.w;
    x.l[8] = slot[8];
    return x;
}
__device__ __forceinline__ Fr29 fr29_select(bool c, const Fr29& a, const Fr29& b) {
    Fr29 r;
#pragma unroll
    for (int l = 0; l < 9; ++l) r.l[l] = c ? a.l[l] : b.l[l];
    return r;
}
#endif

}  // namespace zk
