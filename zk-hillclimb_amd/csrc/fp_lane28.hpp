// fp_lane28.hpp -- BLS12-381 Fp and G1 with one element per lane as 14 signed limbs of 28 bits.
//
// The throughput form of the row arithmetic (fp_row.hpp): the same residues with the Montgomery
// radix R' = 2^392, one whole element per lane.  With 12 limbs of 32 bits (fp_dev.hpp) every
// 32 x 32 product needs an add-with-carry beside it and every sum a canonical reduction; 28-bit
// limbs leave a column of 28 products inside 64 bits, so a product is 392 multiply-adds and
// ~100 other instructions, and sums and differences are taken limb by limb, signed, without
// carries.  Values lie within a few p of zero on either side; canonical values exist only at
// f28_canon.  Bounds (in units of 2^28 for limbs, of p for values) are written at each use: a
// product's operands need (limb bound a) x (limb bound b), summed over the products it adds, of
// at most 8 - 1 (14 x 2^56 x 8 < 2^63, the reduction adding one unit), and leaves limbs in [0, 1],
// the top limb signed, and a value in (-v, 2 + v) for v = sum of alpha beta / 2520.
#pragma once
#include "fp_row.hpp"

struct f28_t {
    int32_t v[14];
};
__device__ constexpr int32_t k_f28_p[16] = {FPR_P_LIMBS};
__device__ constexpr int32_t k_f28_m[16] = {FPR_M_LIMBS};

FDEV f28_t f28_add(const f28_t& a, const f28_t& b) {
    f28_t r;
#pragma unroll
    for (int i = 0; i < 14; i++) r.v[i] = a.v[i] + b.v[i];
    return r;
}
FDEV f28_t f28_sub(const f28_t& a, const f28_t& b) {
    f28_t r;
#pragma unroll
    for (int i = 0; i < 14; i++) r.v[i] = a.v[i] - b.v[i];
    return r;
}
FDEV f28_t f28_twice(const f28_t& a) {
    f28_t r;
#pragma unroll
    for (int i = 0; i < 14; i++) r.v[i] = 2 * a.v[i];
    return r;
}
// limbs back to [0, 2^28) plus a carry of a few units (one pass), the top limb signed
FDEV f28_t f28_carry(const f28_t& a) {
    f28_t r;
    int32_t c = 0;
#pragma unroll
    for (int i = 0; i < 14; i++) {
        const int32_t t = a.v[i] + c;
        r.v[i] = i < 13 ? t & (int32_t)FPR_MASK : t;
        c = t >> 28;
    }
    return r;
}
// the sum of the PRODUCTS products a_k b_k (b_k = a_k, its cross products taken once, when SQR)
// times R'^-1, column by column; the reduction is fp_row.hpp's: columns 0 .. 12 drop their low
// 28 bits m and add m M one column up, column 13 takes m = acc n0 and adds m p
template <int PRODUCTS, bool SQR>
FDEV f28_t f28_dot(const f28_t& a0, const f28_t& b0, const f28_t& a1, const f28_t& b1) {
    int32_t m[14];
    int64_t acc = 0;
    f28_t r;
    f28_t d;
    if (SQR) d = f28_twice(a0);
#pragma unroll
    for (int k = 0; k < 27; k++) {
#pragma unroll
        for (int i = 0; i < 14; i++) {
            const int j = k - i;
            if (j < 0 || j > 13) continue;
            if (SQR) {
                if (i < j) acc += (int64_t)d.v[i] * a0.v[j];
                if (i == j) acc += (int64_t)a0.v[i] * a0.v[i];
            } else {
                acc += (int64_t)a0.v[i] * b0.v[j];
                if (PRODUCTS == 2) acc += (int64_t)a1.v[i] * b1.v[j];
            }
        }
#pragma unroll
        for (int i = 0; i < 13; i++) {
            const int j = k - 1 - i;
            if (j >= 0 && j <= 13) acc += (int64_t)m[i] * k_f28_m[j];
        }
        if (k > 13) acc += (int64_t)m[13] * k_f28_p[k - 13];
        if (k < 13) {
            m[k] = (int32_t)((uint32_t)acc & FPR_MASK);
        } else if (k == 13) {
            m[13] = (int32_t)(((uint32_t)acc * FPR_N0) & FPR_MASK);
            acc += (int64_t)m[13] * k_f28_p[0];
        } else {
            r.v[k - 14] = (int32_t)((uint32_t)acc & FPR_MASK);
        }
        acc >>= 28;
    }
    r.v[13] = (int32_t)acc;
    return r;
}
FDEV f28_t f28_mul(const f28_t& a, const f28_t& b) { return f28_dot<1, false>(a, b, a, b); }
FDEV f28_t f28_sqr(const f28_t& a) { return f28_dot<1, true>(a, a, a, a); }

struct g28_t {
    f28_t x, y, z;
};
// a second operand with its Z^2 and Z^3, taken once for all the additions it enters
struct g28b_t {
    f28_t x, y, z, zz, zzz;
};

// add-2007-bl of a and b, neither at infinity, without the equal-point branch: h and r are left
// to the caller's test.  Coordinates: limbs [0, 1], values within 3.
FDEV g28_t g28_add_core(const g28_t& a, const g28b_t& b, f28_t& h, f28_t& r) {
    const f28_t z1z1 = f28_sqr(a.z);
    const f28_t u1 = f28_mul(a.x, b.zz);
    h = f28_sub(f28_mul(b.x, z1z1), u1);
    const f28_t s1 = f28_mul(a.y, b.zzz);
    r = f28_sub(f28_mul(b.y, f28_mul(a.z, z1z1)), s1);
    g28_t o;
    const f28_t h2 = f28_twice(h), r2 = f28_twice(r);
    o.z = f28_mul(f28_mul(a.z, b.z), h2);
    const f28_t i = f28_sqr(h2);  // limbs 2 x 2 = 4
    const f28_t j = f28_mul(h, i), v = f28_mul(u1, i);
    o.x = f28_carry(f28_sub(f28_sub(f28_sqr(r2), j), f28_twice(v)));
    // r (V - X3) - 2 S1 J: limbs 2 x 1 + 2 x 1 = 4
    f28_t nj;
#pragma unroll
    for (int k = 0; k < 14; k++) nj.v[k] = -2 * j.v[k];
    o.y = f28_dot<2, false>(r2, f28_sub(v, o.x), s1, nj);
    return o;
}
