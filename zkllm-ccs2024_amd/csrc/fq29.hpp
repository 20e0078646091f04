// BLS12-381 base field in a redundant signed radix-2^29 form, for the inner loops of the G1 kernels on gfx950.
//
// A value is 14 limbs: limbs 0..12 in [0, 2^29), limb 13 signed; it stands for x * 2^406 mod p (Montgomery form with
// R' = 2^406) and may be any integer congruent to that, negative included, as long as its magnitude stays below
// about 2^11 p -- every chain of additions and subtractions in the point formulas stays below 32 p.
//
// Why: with 29-bit limbs a column of the schoolbook product (at most 28 products of 58 bits) fits a 64-bit
// accumulator, so a limb product is ONE v_mad_i64_i32 with no carry instruction behind it, the reduction needs no
// final conditional subtraction (R' is 2^24 times larger than p), and additions / subtractions are limb-wise with a
// shift-and-mask carry pass -- no carry flags, which on this chip cost wait states.  395 multiply-adds and 85
// other instructions per product, against 288 + 288 add-with-carry + about 150 in the 32-bit form (field.hpp).
//
// The same formulas as g1.hpp (dbl-2009-l, madd-2007-bl; bls12-381.cu:1361-1464), on points that carry an explicit
// infinity flag: z is not canonical here, so "z == 0" cannot be read off the limbs.
#pragma once
#include "g1.hpp"

namespace zk {

struct Fq29 { int32_t l[14]; };
static constexpr uint32_t M29 = (1u << 29) - 1u;

ZK_HD constexpr int32_t fq29_p(int i) {
    constexpr int32_t t[14] = {536849067, 267911167, 352321518, 402652514, 258097642, 156269400, 184392899, 278818978, 392460107, 303717734, 315025901, 318754100, 1121955, 13};
    return t[i];
}
static constexpr uint32_t FQ29_INV = 536674301u;       // -p^-1 mod 2^29
ZK_HD constexpr int32_t fq29_n(int i) {                // (FQ29_INV p + 1) / 2^29
    constexpr int32_t t[14] = {269986483, 288129268, 349704134, 68745122, 23551659, 302892419, 121324309, 76446693, 148975020, 469560613, 304725929, 383887694, 535436513, 12};
    return t[i];
}
ZK_HD Fq29 fq29_one() {                                // 2^406 mod p
    constexpr int32_t t[14] = {61471620, 195036816, 118655217, 257539269, 309114388, 92651318, 461745213, 486037242, 412216509, 444525573, 358254832, 121744493, 320324367, 9};
    Fq29 r;
#pragma unroll
    for (int i = 0; i < 14; ++i) r.l[i] = t[i];
    return r;
}
ZK_HD Fq29 fq29_c_in() {                               // 2^428 mod p: (x 2^384) * c_in / 2^406 = x 2^406
    constexpr int32_t t[14] = {534637501, 441406580, 43119513, 349190972, 258780460, 458009546, 361923196, 35416775, 516237956, 385703620, 211160486, 265465707, 321271185, 11};
    Fq29 r;
#pragma unroll
    for (int i = 0; i < 14; ++i) r.l[i] = t[i];
    return r;
}
ZK_HD Fq29 fq29_c_out() {                              // 2^384 mod p: (x 2^406) * c_out / 2^406 = x 2^384
    constexpr int32_t t[14] = {196605, 273154048, 50331805, 134223752, 361475775, 204188131, 487947554, 174983754, 225955416, 487765859, 385992357, 352438566, 526773311, 10};
    Fq29 r;
#pragma unroll
    for (int i = 0; i < 14; ++i) r.l[i] = t[i];
    return r;
}
ZK_HD Fq29 fq29_zero() {
    Fq29 r;
#pragma unroll
    for (int i = 0; i < 14; ++i) r.l[i] = 0;
    return r;
}

// Montgomery reduction interleaved with the product columns: col(k) is the k-th column sum of the product (k = 0..26).
// The column sums do not depend on the reduction, so they fill the latency of the m[k] computations.
// The first twelve limbs go by N = FQ29_INV p, which is -1 in its lowest limb: the multiple of N that clears a limb is the limb itself, and what it adds to
// the columns above is fq29_n.  No product stands between a column and its multiplier.  N is 2^29 times p, so the last two limbs go by p itself: what the twelve add is below
// 2^(29 * 12) N = 2^-29 R' p.  All fourteen limbs by p took k_msm_rows 9.18 ms for 45 M additions instead of 8.67, an opening of 131072 columns 6.66 instead of 6.30.
template <typename Col> ZK_HD Fq29 fq29_redc(Col col) {
    constexpr int FAST = 12;
    int32_t m[14];
    Fq29 t;
    int64_t carry = 0;
#pragma unroll
    for (int k = 0; k < 14; ++k) {
        int64_t q = carry;
#pragma unroll
        for (int i = 0; i < k; ++i) q += (int64_t)m[i] * (i < FAST ? fq29_n(k - i - 1) : fq29_p(k - i));
        q += col(k);
        if (k < FAST) m[k] = (int32_t)((uint32_t)q & M29);
        else {
            m[k] = (int32_t)(((uint32_t)q * FQ29_INV) & M29);
            q += (int64_t)m[k] * fq29_p(0);
        }
        carry = q >> 29;
    }
#pragma unroll
    for (int k = 14; k < 28; ++k) {
        int64_t q = carry;
#pragma unroll
        for (int i = k - 14; i < 14; ++i) {
            if (i < FAST) q += (int64_t)m[i] * fq29_n(k - i - 1);
            else if (i > k - 14) q += (int64_t)m[i] * fq29_p(k - i);
        }
        if (k < 27) {
            q += col(k);
            t.l[k - 14] = (int32_t)((uint32_t)q & M29);
            carry = q >> 29;
        } else {
            t.l[13] = (int32_t)q;
        }
    }
    return t;
}
// a * b / 2^406 mod p, result in (-eps, p + eps)
ZK_HD Fq29 fq29_mul_inline(const Fq29& a, const Fq29& b) {
    return fq29_redc([&](int k) {
        int64_t s = 0;
#pragma unroll
        for (int i = 0; i < 14; ++i)
            if (k - i >= 0 && k - i < 14) s += (int64_t)a.l[i] * b.l[k - i];
        return s;
    });
}
// a * a / 2^406 mod p with the symmetric products taken once (105 limb products instead of 196)
ZK_HD Fq29 fq29_sqr_inline(const Fq29& a) {
    int32_t d[14];
#pragma unroll
    for (int i = 0; i < 14; ++i) d[i] = a.l[i] * 2;
    return fq29_redc([&](int k) {
        int64_t s = 0;
#pragma unroll
        for (int i = 0; i < 14; ++i) {
            const int j = k - i;
            if (j > i && j < 14) s += (int64_t)a.l[i] * d[j];
        }
        if (!(k & 1) && (k >> 1) < 14) s += (int64_t)a.l[k >> 1] * a.l[k >> 1];
        return s;
    });
}
#if defined(__HIP_DEVICE_COMPILE__)
typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
typedef int32_t i32x2 __attribute__((ext_vector_type(2)));
// out of line, operands in vector registers (28 dwords)
static __device__ __attribute__((noinline)) Fq29 fq29_mul_regs(i32x4 a0, i32x4 a1, i32x4 a2, i32x2 a3, i32x4 b0, i32x4 b1, i32x4 b2, i32x2 b3) {
    Fq29 a, b;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        a.l[i] = a0[i]; a.l[4 + i] = a1[i]; a.l[8 + i] = a2[i];
        b.l[i] = b0[i]; b.l[4 + i] = b1[i]; b.l[8 + i] = b2[i];
    }
    a.l[12] = a3[0]; a.l[13] = a3[1];
    b.l[12] = b3[0]; b.l[13] = b3[1];
    return fq29_mul_inline(a, b);
}
static __device__ __attribute__((noinline)) Fq29 fq29_sqr_regs(Fq29 a) { return fq29_sqr_inline(a); }
__device__ __forceinline__ Fq29 fq29_mul(const Fq29& a, const Fq29& b) {
    return fq29_mul_regs(i32x4{a.l[0], a.l[1], a.l[2], a.l[3]}, i32x4{a.l[4], a.l[5], a.l[6], a.l[7]}, i32x4{a.l[8], a.l[9], a.l[10], a.l[11]}, i32x2{a.l[12], a.l[13]},
                         i32x4{b.l[0], b.l[1], b.l[2], b.l[3]}, i32x4{b.l[4], b.l[5], b.l[6], b.l[7]}, i32x4{b.l[8], b.l[9], b.l[10], b.l[11]}, i32x2{b.l[12], b.l[13]});
}
__device__ __forceinline__ Fq29 fq29_sqr(const Fq29& a) { return fq29_sqr_regs(a); }
#else
static ZK_NOINLINE_HD Fq29 fq29_mul(const Fq29& a, const Fq29& b) { return fq29_mul_inline(a, b); }
static ZK_NOINLINE_HD Fq29 fq29_sqr(const Fq29& a) { return fq29_sqr_inline(a); }
#endif

// limb-wise sum / difference with the carry pass (arithmetic shifts: intermediate limbs may be negative)
ZK_HD Fq29 fq29_add(const Fq29& a, const Fq29& b) {
    Fq29 r;
    int32_t c = 0;
#pragma unroll
    for (int i = 0; i < 13; ++i) {
        const int32_t s = a.l[i] + b.l[i] + c;
        r.l[i] = (int32_t)((uint32_t)s & M29);
        c = s >> 29;
    }
    r.l[13] = a.l[13] + b.l[13] + c;
    return r;
}
ZK_HD Fq29 fq29_sub(const Fq29& a, const Fq29& b) {
    Fq29 r;
    int32_t c = 0;
#pragma unroll
    for (int i = 0; i < 13; ++i) {
        const int32_t s = a.l[i] - b.l[i] + c;
        r.l[i] = (int32_t)((uint32_t)s & M29);
        c = s >> 29;
    }
    r.l[13] = a.l[13] - b.l[13] + c;
    return r;
}
ZK_HD Fq29 fq29_dbl(const Fq29& a) { return fq29_add(a, a); }
ZK_HD Fq29 fq29_neg(const Fq29& a) { return fq29_sub(fq29_zero(), a); }
ZK_HD bool fq29_same(const Fq29& a, const Fq29& b) {      // equal as integers (both normalised)
    int32_t o = 0;
#pragma unroll
    for (int i = 0; i < 14; ++i) o |= a.l[i] ^ b.l[i];
    return o == 0;
}
// k * p as a normalised value, |k| small
ZK_HD Fq29 fq29_kp(int k) {
    Fq29 r;
    int64_t c = 0;
#pragma unroll
    for (int i = 0; i < 13; ++i) {
        const int64_t s = (int64_t)k * fq29_p(i) + c;
        r.l[i] = (int32_t)((uint32_t)s & M29);
        c = s >> 29;
    }
    r.l[13] = (int32_t)((int64_t)k * fq29_p(13) + c);
    return r;
}
// out of line, and on the device with the value in registers: a reference parameter would make every caller keep the
// value in private memory for a call that almost never happens
#if defined(__HIP_DEVICE_COMPILE__)
static __device__ __attribute__((noinline)) bool fq29_is_kp_regs(i32x4 a0, i32x4 a1, i32x4 a2, i32x2 a3, int k) {
    Fq29 a;
    a.l[0] = a0[0]; a.l[1] = a0[1]; a.l[2] = a0[2]; a.l[3] = a0[3];
    a.l[4] = a1[0]; a.l[5] = a1[1]; a.l[6] = a1[2]; a.l[7] = a1[3];
    a.l[8] = a2[0]; a.l[9] = a2[1]; a.l[10] = a2[2]; a.l[11] = a2[3];
    a.l[12] = a3[0]; a.l[13] = a3[1];
    return fq29_same(a, fq29_kp(k));
}
__device__ __forceinline__ bool fq29_is_kp(const Fq29& a, int k) {
    return fq29_is_kp_regs(i32x4{a.l[0], a.l[1], a.l[2], a.l[3]}, i32x4{a.l[4], a.l[5], a.l[6], a.l[7]}, i32x4{a.l[8], a.l[9], a.l[10], a.l[11]}, i32x2{a.l[12], a.l[13]}, k);
}
#else
static ZK_NOINLINE_HD bool fq29_is_kp(const Fq29& a, int k) { return fq29_same(a, fq29_kp(k)); }
#endif
// a == 0 mod p, for |a| < 40 p.  A multiple k*p has top limb 13k (k >= 0) or 13k - 1 (k < 0): the top limb names the
// only candidate k, the low limb then rules it out except with probability 2^-29, and the full comparison
// runs out of line in the rare remaining case.
ZK_HD bool fq29_is_zero_mod_p(const Fq29& a) {
    const int32_t kk = a.l[13] + (a.l[13] < 0 ? 1 : 0);
    const int32_t k = (kk * 20165 + (1 << 17)) >> 18;            // kk / 13 when 13 divides kk
    if (k * 13 != kk) return false;
    if (a.l[0] != (int32_t)(((uint32_t)k * (uint32_t)fq29_p(0)) & M29)) return false;
    return fq29_is_kp(a, k);
}

// a - b, limb by limb without the carry pass: limbs within +-2^29, for operands of products alone
ZK_HD Fq29 fq29_sub_raw(const Fq29& a, const Fq29& b) {
    Fq29 r;
#pragma unroll
    for (int i = 0; i < 14; ++i) r.l[i] = a.l[i] - b.l[i];
    return r;
}
// a + p where a is negative
ZK_HD Fq29 fq29_lift(const Fq29& a) {
    const int32_t neg = a.l[13] >> 31;
    Fq29 r;
    int32_t c = 0;
#pragma unroll
    for (int i = 0; i < 13; ++i) {
        const int32_t s = a.l[i] + (fq29_p(i) & neg) + c;
        r.l[i] = (int32_t)((uint32_t)s & M29);
        c = s >> 29;
    }
    r.l[13] = a.l[13] + (fq29_p(13) & neg) + c;
    return r;
}
// a - b - 2 c in one carry pass
ZK_HD Fq29 fq29_sub2(const Fq29& a, const Fq29& b, const Fq29& c) {
    Fq29 r;
    int32_t k = 0;
#pragma unroll
    for (int i = 0; i < 13; ++i) {
        const int32_t s = a.l[i] - b.l[i] - 2 * c.l[i] + k;
        r.l[i] = (int32_t)((uint32_t)s & M29);
        k = s >> 29;
    }
    r.l[13] = a.l[13] - b.l[13] - 2 * c.l[13] + k;
    return r;
}
// (a b - c d) / 2^406 mod p with one reduction.  a, b: limbs within +-2^29; c, d: normalised (limbs 0..12 not negative).  A column
// lies within 28 * 2^58 either way: -28 when a b is at its lowest and nothing is added back, +28 with a b and the reduction's at
// their highest.
ZK_HD Fq29 fq29_mul_sub(const Fq29& a, const Fq29& b, const Fq29& c, const Fq29& d) {
    Fq29 n;
#pragma unroll
    for (int i = 0; i < 14; ++i) n.l[i] = -c.l[i];
    return fq29_redc([&](int k) {
        int64_t s = 0;
#pragma unroll
        for (int i = 0; i < 14; ++i)
            if (k - i >= 0 && k - i < 14) s += (int64_t)a.l[i] * b.l[k - i];
#pragma unroll
        for (int i = 0; i < 14; ++i)
            if (k - i >= 0 && k - i < 14) s += (int64_t)n.l[i] * d.l[k - i];
        return s;
    });
}

// ---- conversion from / to the 32-bit Montgomery form (R = 2^384, canonical) ---------------------------------------
ZK_HD Fq29 fq29_repack(const Fp& a) {                   // same integer, 29-bit limbs
    Fq29 r;
#pragma unroll
    for (int i = 0; i < 14; ++i) {
        const int off = 29 * i, w = off >> 5, sh = off & 31;
        uint32_t v = (w < 12) ? (a.v[w] >> sh) : 0u;
        if (sh > 3 && w + 1 < 12) v |= a.v[w + 1] << (32 - sh);
        r.l[i] = (int32_t)(v & M29);
    }
    return r;
}
ZK_HD Fq29 fq29_from_fp(const Fp& a) { return fq29_mul(fq29_repack(a), fq29_c_in()); }
// canonical residue in [0, p) of a value in (-p, 2p)
ZK_HD Fq29 fq29_canon(const Fq29& a) {
    Fq29 v = a;
    if (v.l[13] < 0) v = fq29_add(v, fq29_kp(1));
    const Fq29 t = fq29_sub(v, fq29_kp(1));
    if (t.l[13] >= 0) v = t;
    return v;
}
ZK_HD Fp fq29_to_fp(const Fq29& a) {
    const Fq29 c = fq29_canon(fq29_mul(a, fq29_c_out()));
    Fp r;
#pragma unroll
    for (int w = 0; w < 12; ++w) {
        // bits [32w, 32w+32) of the integer: limbs floor(32w/29) and the next one or two
        const int off = 32 * w, i = off / 29, sh = off % 29;
        uint64_t v = (uint64_t)(uint32_t)c.l[i] >> sh;
        if (i + 1 < 14) v |= (uint64_t)(uint32_t)c.l[i + 1] << (29 - sh);
        if (i + 2 < 14) v |= (uint64_t)(uint32_t)c.l[i + 2] << (58 - sh);
        r.v[w] = (uint32_t)v;
    }
    return r;
}

// ---- points -----------------------------------------------------------------------------------------------------------
// The point formulas are inlined into the kernels' loops on the device (the field products inside them stay calls with
// their operands in registers): as functions of their own they take and return points through private memory, and that
// traffic -- half a kilobyte per lane and point operation -- cost more than the arithmetic.
#if defined(__HIP_DEVICE_COMPILE__)
#define FQ29_POINT_FN ZK_HD
#else
#define FQ29_POINT_FN static ZK_NOINLINE_HD
#endif
struct A29 { Fq29 x, y; };                 // affine; all-zero limbs = infinity (as the normalised 32-bit tables mark it)
struct J29 { Fq29 x, y, z; uint32_t inf; };
ZK_HD bool a29_is_inf(const A29& p) {
    int32_t o = 0;
#pragma unroll
    for (int i = 0; i < 14; ++i) o |= p.x.l[i] | p.y.l[i];
    return o == 0;
}
ZK_HD J29 j29_infinity() { J29 r; r.x = fq29_zero(); r.y = fq29_one(); r.z = fq29_zero(); r.inf = 1u; return r; }
ZK_HD A29 a29_from_affine(const G1Affine& p) {
    A29 r;
    r.x = fq29_from_fp(p.x);          // 0 stays 0: the infinity marker survives
    r.y = fq29_from_fp(p.y);
    return r;
}
ZK_HD G1Jac j29_to_jac(const J29& p) {
    if (p.inf) return g1_infinity();
    G1Jac r;
    r.x = fq29_to_fp(p.x); r.y = fq29_to_fp(p.y); r.z = fq29_to_fp(p.z);
    return r;
}
// The flag alone says infinity: the formulas run on whatever the coordinates hold (no branch, so the result of a walk
// step is one set of registers whatever the lanes' cases are).
FQ29_POINT_FN J29 j29_double(const J29& p) {
    const Fq29 a = fq29_sqr(p.x);
    const Fq29 b = fq29_sqr(p.y);
    Fq29 c = fq29_sqr(b);
    Fq29 d = fq29_sqr(fq29_add(p.x, b));
    d = fq29_dbl(fq29_sub(fq29_sub(d, a), c));
    const Fq29 e = fq29_add(fq29_dbl(a), a);
    const Fq29 f = fq29_sqr(e);
    J29 r;
    r.inf = p.inf;
    r.z = fq29_dbl(fq29_mul(p.y, p.z));
    r.x = fq29_sub(fq29_sub(f, d), d);
    c = fq29_dbl(fq29_dbl(fq29_dbl(c)));
    r.y = fq29_sub(fq29_mul(fq29_sub(d, r.x), e), c);
    return r;
}
FQ29_POINT_FN J29 j29_add_mixed(const J29& a, const A29& b) {
    const Fq29 z1z1 = fq29_sqr(a.z);
    const Fq29 u2 = fq29_mul(b.x, z1z1);
    const Fq29 s2 = fq29_mul(fq29_mul(b.y, a.z), z1z1);
    const Fq29 h = fq29_sub(u2, a.x);
    const Fq29 rr0 = fq29_sub(s2, a.y);
    const Fq29 hh = fq29_sqr(h);
    const Fq29 i = fq29_dbl(fq29_dbl(hh));
    Fq29 j = fq29_mul(h, i);
    const Fq29 rr = fq29_dbl(rr0);
    const Fq29 v = fq29_mul(a.x, i);
    J29 r;
    r.inf = 0u;
    r.x = fq29_sub(fq29_sub(fq29_sqr(rr), j), fq29_dbl(v));
    j = fq29_dbl(fq29_mul(a.y, j));
    r.y = fq29_sub(fq29_mul(fq29_sub(v, r.x), rr), j);
    r.z = fq29_sub(fq29_sub(fq29_sqr(fq29_add(a.z, h)), z1z1), hh);
    if (a.inf) {                                       // infinity + b = b
        r.x = b.x; r.y = b.y; r.z = fq29_one();
    } else if (fq29_is_zero_mod_p(h)) {                // same abscissa: the same point (double it) or its opposite
        if (fq29_is_zero_mod_p(rr0)) r = j29_double(a);
        else r = j29_infinity();
    }
    return r;
}

// a + b, both Jacobian (add-2007-bl, bls12-381.cu:1431-1464), with the flag and the equal-abscissa cases as above
FQ29_POINT_FN J29 j29_add(const J29& a, const J29& b) {
    const Fq29 z1z1 = fq29_sqr(a.z), z2z2 = fq29_sqr(b.z);
    const Fq29 u1 = fq29_mul(a.x, z2z2), u2 = fq29_mul(b.x, z1z1);
    Fq29 s1 = fq29_mul(fq29_mul(a.y, b.z), z2z2);
    const Fq29 s2 = fq29_mul(fq29_mul(b.y, a.z), z1z1);
    const Fq29 h = fq29_sub(u2, u1), rr0 = fq29_sub(s2, s1);
    const Fq29 i = fq29_sqr(fq29_dbl(h));
    const Fq29 j = fq29_mul(h, i);
    const Fq29 rr = fq29_dbl(rr0);
    const Fq29 v = fq29_mul(u1, i);
    J29 r;
    r.inf = 0u;
    r.x = fq29_sub(fq29_sub(fq29_sqr(rr), j), fq29_dbl(v));
    s1 = fq29_dbl(fq29_mul(s1, j));
    r.y = fq29_sub(fq29_mul(fq29_sub(v, r.x), rr), s1);
    r.z = fq29_mul(fq29_sub(fq29_sub(fq29_sqr(fq29_add(a.z, b.z)), z1z1), z2z2), h);
    if (a.inf) r = b;
    else if (b.inf) r = a;
    else if (fq29_is_zero_mod_p(h)) {
        if (fq29_is_zero_mod_p(rr0)) r = j29_double(a);
        else r = j29_infinity();
    }
    return r;
}
// Points as (X / ZZ, Y / ZZZ) with ZZ^3 = ZZZ^2, for long sums of affine points: a mixed addition (madd-2008-s, dbl-2008-s-1 and
// mdbl-2008-s-1 of the explicit-formulas database) takes six products, two squares and one reduction over two products -- about 4700
// instructions against 5700 of the Jacobian one, whose squares and carry passes it does without.
struct X29 { Fq29 x, y, zz, zzz; uint32_t inf; };
ZK_HD X29 x29_infinity() { X29 r; r.x = r.y = r.zz = r.zzz = fq29_zero(); r.inf = 1u; return r; }
ZK_HD void x29_add_mixed(X29& a, const A29& b) {
    const Fq29 u2 = fq29_mul_inline(b.x, a.zz), s2 = fq29_mul_inline(b.y, a.zzz);
    const Fq29 h = fq29_sub_raw(u2, a.x), rr = fq29_sub_raw(s2, a.y);
    const Fq29 hh = fq29_sqr_inline(h), hhh = fq29_mul_inline(h, hh), q = fq29_mul_inline(a.x, hh);
    X29 r;
    r.inf = 0u;
    r.x = fq29_sub2(fq29_sqr_inline(rr), hhh, q);
    r.y = fq29_mul_sub(rr, fq29_sub_raw(q, r.x), a.y, hhh);
    r.zz = fq29_mul_inline(a.zz, hh);
    r.zzz = fq29_mul_inline(a.zzz, hhh);
    // equal abscissae: hh, a product, is 0 or p (or its neighbourhood's only other multiples of p); the low limb rules that out
    // except with probability 2^-28
    if (!a.inf && (hh.l[0] == 0 || hh.l[0] == fq29_p(0)) && fq29_is_zero_mod_p(hh)) {
        const Fq29 r0 = fq29_sub(s2, a.y);
        if (fq29_is_zero_mod_p(r0)) {                  // the same point: its double
            const Fq29 u = fq29_dbl(a.y), v = fq29_sqr(u), w = fq29_mul(u, v), s = fq29_mul(a.x, v), xx = fq29_sqr(a.x), m = fq29_add(fq29_dbl(xx), xx);
            r.x = fq29_sub(fq29_sqr(m), fq29_dbl(s));
            r.y = fq29_sub(fq29_mul(m, fq29_sub(s, r.x)), fq29_mul(w, a.y));
            r.zz = fq29_mul(v, a.zz);
            r.zzz = fq29_mul(w, a.zzz);
            if (fq29_is_zero_mod_p(u)) r.inf = 1u;     // a point of order two
        } else r.inf = 1u;
    }
    if (a.inf) { r.x = b.x; r.y = b.y; r.zz = fq29_one(); r.zzz = fq29_one(); }
    a = r;
}
// the same point in Jacobian form, with z = zzz
FQ29_POINT_FN J29 j29_from_x29(const X29& p) {
    J29 r;
    r.inf = p.inf;
    r.x = fq29_mul(p.x, fq29_sqr(p.zz));
    r.y = fq29_mul(p.y, fq29_sqr(p.zzz));
    r.z = p.zzz;
    return r;
}
// ---- Jacobian points for long walks: products inlined, differences that only products read without their carry pass, y with one
// reduction over two products ----------------------------------------------------------------------------------------------
template <int SH> ZK_HD Fq29 fq29_shl(const Fq29& a) {      // 2^SH a
    Fq29 r;
    int32_t c = 0;
#pragma unroll
    for (int i = 0; i < 13; ++i) {
        const uint32_t lo = (uint32_t)a.l[i];                // limbs 0..12 are in [0, 2^29)
        r.l[i] = (int32_t)(((lo << SH) & M29) | (uint32_t)c);
        c = (int32_t)(lo >> (29 - SH));
    }
    r.l[13] = (int32_t)((uint32_t)a.l[13] << SH) + c;
    return r;
}
// a - 8 b in one carry pass (8 b formed by shifts across the limbs)
ZK_HD Fq29 fq29_sub8(const Fq29& a, const Fq29& b) { return fq29_sub(a, fq29_shl<3>(b)); }
// x3 = (3 x^2)^2 - 8 s, y3 = 3 x^2 (4 s - x3) - 8 y^4, z3 = 2 y z with s = x y^2
ZK_HD void j29_double_walk(J29& p) {
    const Fq29 a = fq29_sqr_inline(p.x), b = fq29_sqr_inline(p.y), yz = fq29_mul_inline(p.y, p.z);
    const Fq29 s = fq29_mul_inline(p.x, b), e = fq29_add(fq29_shl<1>(a), a);
    p.x = fq29_sub8(fq29_sqr_inline(e), s);
    p.y = fq29_mul_sub(e, fq29_sub_raw(fq29_shl<2>(s), p.x), fq29_shl<3>(b), b);
    p.z = fq29_shl<1>(yz);
}
// madd-2004-hmv
ZK_HD void j29_add_mixed_walk(J29& a, const A29& b) {
    const Fq29 zz = fq29_sqr_inline(a.z), u2 = fq29_mul_inline(b.x, zz), s2 = fq29_mul_inline(fq29_mul_inline(b.y, a.z), zz);
    const Fq29 h = fq29_sub_raw(u2, a.x), rr = fq29_sub_raw(s2, a.y);
    const Fq29 hh = fq29_sqr_inline(h), hhh = fq29_mul_inline(h, hh), v = fq29_mul_inline(a.x, hh);
    J29 r;
    r.inf = 0u;
    r.z = fq29_mul_inline(a.z, h);
    r.x = fq29_sub2(fq29_sqr_inline(rr), hhh, v);
    r.y = fq29_mul_sub(rr, fq29_sub_raw(v, r.x), a.y, hhh);
    if (!a.inf && (hh.l[0] == 0 || hh.l[0] == fq29_p(0)) && fq29_is_zero_mod_p(hh)) {      // the same point or its opposite
        if (fq29_is_zero_mod_p(fq29_sub(s2, a.y))) r = j29_double(a);
        else r.inf = 1u;
    }
    if (a.inf) { r.x = b.x; r.y = b.y; r.z = fq29_one(); }
    a = r;
}
// ---- homogeneous projective points ----------------------------------------------------------------------------------------------
// (X / Z, Y / Z), infinity (0 : y : 0).  The complete formulas of Renes, Costello and Batina (2016, algorithms 7 and 9, a = 0, b = 4) hold for
// every pair of points of a curve without a point of order two, which this one is: its group has odd order.  So there are no cases, and
// nothing to keep beside the coordinates.  An addition takes six products and three reductions over two products each, 4116 limb products
// against 5817 of the Jacobian one, and is three products deep where that is five; a doubling is two deep instead of three.
struct P29 { Fq29 x, y, z; };
ZK_HD P29 p29_infinity() { P29 r; r.x = r.z = fq29_zero(); r.y = fq29_one(); return r; }
ZK_HD P29 p29_from_x29(const X29& p) {
    P29 r;
    r.x = fq29_mul(p.x, p.zzz);
    r.y = fq29_mul(p.y, p.zz);
    r.z = fq29_mul(p.zz, p.zzz);
    if (p.inf) r = p29_infinity();
    return r;
}
ZK_HD P29 p29_from_j29(const J29& p) {
    P29 r;
    r.x = fq29_mul(p.x, p.z);
    r.y = p.y;
    r.z = fq29_mul(fq29_sqr(p.z), p.z);
    if (p.inf) r = p29_infinity();
    return r;
}
ZK_HD G1Jac p29_to_jac(const P29& p) {
    if (fq29_is_zero_mod_p(p.z)) return g1_infinity();
    G1Jac r;
    r.x = fq29_to_fp(fq29_mul(p.x, p.z));
    r.y = fq29_to_fp(fq29_mul(p.y, fq29_sqr(p.z)));
    r.z = fq29_to_fp(p.z);
    return r;
}
// ka a + kb b for small factors, in one carry pass
ZK_HD Fq29 fq29_lin(const Fq29& a, int32_t ka, const Fq29& b, int32_t kb) {
    Fq29 r;
    int64_t c = 0;
#pragma unroll
    for (int i = 0; i < 13; ++i) {
        c += (int64_t)a.l[i] * ka + (int64_t)b.l[i] * kb;
        r.l[i] = (int32_t)((uint32_t)c & M29);
        c >>= 29;
    }
    r.l[13] = a.l[13] * ka + b.l[13] * kb + (int32_t)c;
    return r;
}
// a - b - c in one carry pass
ZK_HD Fq29 fq29_sub_both(const Fq29& a, const Fq29& b, const Fq29& c) {
    Fq29 r;
    int32_t k = 0;
#pragma unroll
    for (int i = 0; i < 13; ++i) {
        const int32_t s = a.l[i] - b.l[i] - c.l[i] + k;
        r.l[i] = (int32_t)((uint32_t)s & M29);
        k = s >> 29;
    }
    r.l[13] = a.l[13] - b.l[13] - c.l[13] + k;
    return r;
}
// a + b on one lane.  INL: everything inlined, for kernels that do little else; otherwise products by calls
template <bool INL> ZK_HD P29 p29_add(const P29& a, const P29& b) {
    auto mul = [](const Fq29& x, const Fq29& y) { if constexpr (INL) return fq29_mul_inline(x, y); else return fq29_mul(x, y); };
    auto mul_sub = [](const Fq29& x, const Fq29& y, const Fq29& z, const Fq29& w) { if constexpr (INL) return fq29_mul_sub(x, y, z, w); else return fq29_sub(fq29_mul(x, y), fq29_mul(z, w)); };
    const Fq29 t0 = mul(a.x, b.x), t1 = mul(a.y, b.y), t2 = mul(a.z, b.z);
    const Fq29 xy = fq29_sub_both(mul(fq29_add(a.x, a.y), fq29_add(b.x, b.y)), t0, t1);
    const Fq29 yz = fq29_sub_both(mul(fq29_add(a.y, a.z), fq29_add(b.y, b.z)), t1, t2);
    const Fq29 xz = fq29_sub_both(mul(fq29_add(a.x, a.z), fq29_add(b.x, b.z)), t0, t2);
    const Fq29 u = fq29_lin(t1, 1, t2, 12), v = fq29_lin(t1, 1, t2, -12), w = fq29_lin(t0, -3, t0, 0), g = fq29_lin(xz, 12, xz, 0);
    P29 r;
    r.x = mul_sub(xy, v, yz, g);
    r.y = mul_sub(u, v, w, g);
    r.z = mul_sub(yz, u, w, xy);
    return r;
}
#if defined(__HIPCC__)
// ---- one point on four lanes -------------------------------------------------------------------------------------------------
// Every lane of four holds the whole point; the independent products of a formula's step go one to a lane and come back by quad
// permutations: two products one after the other for a doubling, three for an addition.  For chains that a launch waits for while the
// chip is empty: a wave alone issues one instruction every six to seven cycles, so the instructions of one lane are what takes the time.
template <int CTRL> __device__ __forceinline__ Fq29 quad_perm(const Fq29& a) {
    Fq29 r;
#pragma unroll
    for (int i = 0; i < 14; ++i) r.l[i] = __builtin_amdgcn_mov_dpp(a.l[i], CTRL, 0xF, 0xF, true);      // every lane of a quad is there: no old value to keep
    return r;
}
template <int FROM> __device__ __forceinline__ Fq29 quad_get(const Fq29& a) { return quad_perm<FROM * 0x55>(a); }
__device__ __forceinline__ Fq29 fq29_select(bool c, const Fq29& a, const Fq29& b) {
    Fq29 r;
#pragma unroll
    for (int i = 0; i < 14; ++i) r.l[i] = c ? a.l[i] : b.l[i];
    return r;
}
// with A = y^2, B = z^2: x3 = 2 xy (A - 36 B), y3 = (A + 12 B)(A - 36 B) + 96 A B, z3 = 8 A yz
__device__ __forceinline__ void p29_quad_double(P29& p, uint32_t q) {
    const Fq29 m1 = fq29_mul_inline(fq29_select(q == 1, p.z, fq29_select(q == 2, p.x, p.y)), fq29_select((q & 1u) != 0, p.z, p.y));      // A | B | x y | y z
    const Fq29 a = quad_get<0>(m1), b = quad_get<1>(m1), own = quad_perm<0xD2>(m1);                                                       // own: x y | A | B | y z
    const int32_t k = q == 0 ? 2 : (q == 1 ? 1 : (q == 2 ? 96 : 8)), kb = q == 1 ? 12 : 0, kr = q < 2 ? -36 : 0;
    const Fq29 m2 = fq29_mul_inline(fq29_lin(own, k, b, kb), fq29_lin(a, 1, b, kr));
    p.x = quad_get<0>(m2);
    p.y = fq29_add(quad_get<1>(m2), quad_get<2>(m2));
    p.z = quad_get<3>(m2);
}
__device__ __forceinline__ void p29_quad_add(P29& a, const P29& b, uint32_t q) {
    const Fq29 m1 = fq29_mul_inline(fq29_select(q == 0, a.x, fq29_select(q == 1, a.y, fq29_select(q == 2, a.z, fq29_add(a.x, a.y)))),
                                    fq29_select(q == 0, b.x, fq29_select(q == 1, b.y, fq29_select(q == 2, b.z, fq29_add(b.x, b.y)))));    // t0 | t1 | t2 | (x + y)(x + y)
    const Fq29 m2 = fq29_mul_inline(fq29_add(fq29_select(q == 0, a.y, a.x), a.z), fq29_add(fq29_select(q == 0, b.y, b.x), b.z));          // (y + z)(y + z) | (x + z)(x + z) | -- | --
    const Fq29 t0 = quad_get<0>(m1), t1 = quad_get<1>(m1), t2 = quad_get<2>(m1);
    const Fq29 xy = fq29_sub_both(quad_get<3>(m1), t0, t1), yz = fq29_sub_both(quad_get<0>(m2), t1, t2), xz = fq29_sub_both(quad_get<1>(m2), t0, t2);
    const Fq29 w = fq29_lin(t0, -3, t0, 0), g = fq29_lin(xz, 12, xz, 0);
    const Fq29 m3 = fq29_mul_sub(fq29_select(q == 0, xy, fq29_select(q == 1, fq29_lin(t1, 1, t2, 12), yz)), fq29_lin(t1, 1, t2, q == 2 ? 12 : -12),
                                 fq29_select(q == 0, yz, w), fq29_select(q == 2, xy, g));                                                 // x3 | y3 | z3 | --
    a.x = quad_get<0>(m3);
    a.y = quad_get<1>(m3);
    a.z = quad_get<2>(m3);
}
#endif
ZK_HD J29 j29_from_jac(const G1Jac& p) {
    if (is_zero(p.z)) return j29_infinity();
    J29 r;
    r.inf = 0u;
    r.x = fq29_from_fp(p.x); r.y = fq29_from_fp(p.y); r.z = fq29_from_fp(p.z);
    return r;
}

}  // namespace zk
