// fp_lane28.hpp -- BLS12-381 Fp and G1 with one element per lane as 14 signed limbs of 28 bits.
//
// The throughput form of the row arithmetic (fp_row.hpp): the same residues with the Montgomery
// radix R' = 2^392, one whole element per lane.  With 12 limbs of 32 bits every 32 x 32 product
// needs an add-with-carry beside it and every sum a canonical reduction; 28-bit limbs leave a
// column of 28 products inside 64 bits, so a product is 392 multiply-adds and ~100 other
// instructions, and sums and differences are taken limb by limb, signed, without carries: an
// addition 0.19 us of a SIMD's time instead of 0.34 (12 us with a SIMD to itself instead of 29).
// Values lie within a few p of zero on either side.  Bounds (in units of 2^28 for limbs, of p for values) are written at each use: a
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
__device__ constexpr int32_t k_f28_kb[16] = {FPR_KB_LIMBS};  // 32 p, limbs raised by 2^30

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

// whether x (in (-32 p, 64 p)) is a multiple of p: a multiple j p has limb 0 = j p_0 mod 2^28, so
// all but 2^-21 of the other values stop at the first test
FDEV bool f28_maybe_zero(const f28_t& x) { return (((uint32_t)x.v[0] * FPR_PINV + 32) & FPR_MASK) <= 96; }
FDEV bool f28_zero(const f28_t& x) {
    if (!f28_maybe_zero(x)) return false;
    f28_t t = x;
#pragma unroll
    for (int i = 0; i < 14; i++) t.v[i] += k_f28_kb[i];
#pragma unroll 1
    for (int j = 0; j <= 96; j++) {
        t = f28_carry(t);
        int32_t o = 0;
#pragma unroll
        for (int i = 0; i < 14; i++) o |= t.v[i];
        if (o == 0) return true;
#pragma unroll
        for (int i = 0; i < 14; i++) t.v[i] -= k_f28_p[i];
    }
    return false;
}

struct g28_t {
    f28_t x, y, z;
};
FDEV g28_t g28_zero() {
    constexpr int32_t one[16] = {FPR_ONE_LIMBS};
    g28_t o;
#pragma unroll
    for (int i = 0; i < 14; i++) o.x.v[i] = o.z.v[i] = 0, o.y.v[i] = one[i];
    return o;
}
// limbs of a row-form point's coordinate (16 words, 14 limbs)
FDEV f28_t f28_load(const uint32_t* p) {
    const uint4* q = (const uint4*)p;
    f28_t r;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const uint4 t = q[k];
        r.v[4 * k] = (int32_t)t.x, r.v[4 * k + 1] = (int32_t)t.y;
        r.v[4 * k + 2] = (int32_t)t.z, r.v[4 * k + 3] = (int32_t)t.w;
    }
    const uint2 t = ((const uint2*)p)[6];
    r.v[12] = (int32_t)t.x, r.v[13] = (int32_t)t.y;
    return r;
}
FDEV void f28_put(uint32_t* p, const f28_t& t, uint32_t extra) {  // limbs as they are; word 14 = extra
    uint4* q = (uint4*)p;
#pragma unroll
    for (int k = 0; k < 3; k++)
        q[k] = make_uint4((uint32_t)t.v[4 * k], (uint32_t)t.v[4 * k + 1], (uint32_t)t.v[4 * k + 2], (uint32_t)t.v[4 * k + 3]);
    q[3] = make_uint4((uint32_t)t.v[12], (uint32_t)t.v[13], extra, 0);
}
// as a nonnegative value with carried limbs: a negative x (above -32 p; its top limb is negative)
// plus 32 p, any other as it is, so that a value that was loaded and only copied stays within
// its bound however often it is stored
FDEV void f28_store(uint32_t* p, const f28_t& x, uint32_t extra) {
    f28_t t;
#pragma unroll
    for (int i = 0; i < 14; i++) t.v[i] = x.v[i] + (x.v[13] < 0 ? k_f28_kb[i] : 0);
    f28_put(p, f28_carry(t), extra);
}
// a row-form point (fp_row.hpp; G1R_WORDS) as loaded, taken apart where it is used.  The words
// past the limbs are zero but for the flag, and all of them are read: destinations whose ends
// are dead get reused by the next load, which then waits for the one before.
struct g28_raw {
    uint4 q[12];
};
FDEV g28_raw g28_fetch(const uint32_t* p) {
    g28_raw r;
#pragma unroll
    for (int k = 0; k < 12; k++) r.q[k] = ((const uint4*)p)[k];
    return r;
}
FDEV f28_t f28_limbs(const uint4* q) {
    f28_t r;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        r.v[4 * k] = (int32_t)q[k].x, r.v[4 * k + 1] = (int32_t)q[k].y;
        r.v[4 * k + 2] = (int32_t)q[k].z, r.v[4 * k + 3] = (int32_t)q[k].w;
    }
    r.v[12] = (int32_t)q[3].x, r.v[13] = (int32_t)q[3].y;
    return r;
}
FDEV g28_t g28_take(const g28_raw& w, bool& inf) {
    inf = (w.q[3].z | w.q[3].w | w.q[7].z | w.q[7].w | w.q[11].z | w.q[11].w) != 0;
    return {f28_limbs(w.q), f28_limbs(w.q + 4), f28_limbs(w.q + 8)};
}
FDEV g28_t g28_load(const uint32_t* p, bool& inf) { return g28_take(g28_fetch(p), inf); }
FDEV void g28_store(uint32_t* p, const g28_t& a, bool inf) {
    f28_store(p, a.x, inf ? 1u : 0u);
    f28_store(p + 16, a.y, 0);
    f28_store(p + 32, a.z, 0);
}

// a coordinate of a 144-byte point (fp_row.hpp) in R' form, below 3 p; any: its words or-ed
FDEV f28_t f28_from_words(const uint32_t* p, uint32_t& any) {
    constexpr int32_t in[16] = {FPR_IN_LIMBS};
    uint32_t w[12];
    f28_t r, k;
    any = 0;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const uint4 t = ((const uint4*)p)[i];
        w[4 * i] = t.x, w[4 * i + 1] = t.y, w[4 * i + 2] = t.z, w[4 * i + 3] = t.w;
        any |= t.x | t.y | t.z | t.w;
    }
#pragma unroll
    for (int i = 0; i < 14; i++) {
        const int j = 28 * i / 32, off = 28 * i % 32;
        uint32_t x = w[j] >> off;
        if (off > 4 && j < 11) x |= w[j + 1] << (32 - off);
        r.v[i] = (int32_t)(x & FPR_MASK);
        k.v[i] = in[i];
    }
    return f28_mul(r, k);
}
// and back: canonical words of x (in (-45 p, 45 p))
FDEV void f28_to_words(uint32_t* p, const f28_t& x) {
    constexpr int32_t out[16] = {FPR_OUT_LIMBS};
    f28_t k;
#pragma unroll
    for (int i = 0; i < 14; i++) k.v[i] = out[i];
    f28_t t = f28_mul(x, k);  // in (-1, 3)
#pragma unroll
    for (int i = 0; i < 14; i++) t.v[i] += k_f28_p[i];
    t = f28_carry(t);
#pragma unroll 1
    for (int n = 0; n < 3; n++) {  // less p where that is not negative
        f28_t d;
#pragma unroll
        for (int i = 0; i < 14; i++) d.v[i] = t.v[i] - k_f28_p[i];
        d = f28_carry(d);
        if (d.v[13] >= 0) t = d;
    }
    uint32_t w[12];
#pragma unroll
    for (int j = 0; j < 12; j++) {
        const int l = 32 * j / 28, off = 32 * j % 28;
        w[j] = (uint32_t)t.v[l] >> off | (uint32_t)t.v[l + 1] << (28 - off);
        if (off > 24) w[j] |= (uint32_t)t.v[l + 2] << (56 - off);
    }
#pragma unroll
    for (int i = 0; i < 3; i++) ((uint4*)p)[i] = make_uint4(w[4 * i], w[4 * i + 1], w[4 * i + 2], w[4 * i + 3]);
}

// dbl-2009-l as g1r_dbl, for a point not at infinity.  Coordinates between operations: limbs
// [0, 1] (z from the row form: [0, 2]) with a signed top limb, x and y in (-17, 45), z in
// (-1, 36): loaded ones up to the row form's bounds, computed ones below 9.
FDEV g28_t g28_dbl(const g28_t& a) {
    const f28_t A = f28_sqr(a.x), B = f28_sqr(a.y), C = f28_sqr(B), XB = f28_mul(a.x, B);
    g28_t o;
    o.z = f28_mul(a.y, f28_twice(a.z));
    f28_t E, t;
#pragma unroll
    for (int i = 0; i < 14; i++) E.v[i] = 3 * A.v[i];
    const f28_t F = f28_sqr(f28_carry(E));
#pragma unroll
    for (int i = 0; i < 14; i++) t.v[i] = F.v[i] - 8 * XB.v[i];
    o.x = f28_carry(t);
    // E (D - X3): limbs 3 x 1
#pragma unroll
    for (int i = 0; i < 14; i++) t.v[i] = 4 * XB.v[i] - o.x.v[i];
    const f28_t y = f28_mul(E, f28_carry(t));
#pragma unroll
    for (int i = 0; i < 14; i++) t.v[i] = y.v[i] - 8 * C.v[i];
    o.y = f28_carry(t);
    return o;
}

// add-2007-bl as g1r_add, of a (inf: its flag, updated) and a point b not at infinity with its
// Z^2 and Z^3: the equal-point branch doubles a, U1 = U2 with S1 != S2 leaves Z3 = 0.
FDEV void g28_add(g28_t& a, bool& inf, const g28_t& b, const f28_t& zz2, const f28_t& zzz2) {
    if (inf) {
        a = b;
        inf = false;
        return;
    }
    const f28_t z1z1 = f28_sqr(a.z);
    const f28_t u1 = f28_mul(a.x, zz2);
    const f28_t h = f28_sub(f28_mul(b.x, z1z1), u1);
    const f28_t s1 = f28_mul(a.y, zzz2);
    const f28_t r = f28_sub(f28_mul(b.y, f28_mul(a.z, z1z1)), s1);
    const bool h0 = f28_zero(h);
    if (h0 && f28_zero(r)) {
        inf = f28_zero(a.y);  // Z3 = 2 Y Z
        a = g28_dbl(a);
        return;
    }
    inf = h0;
    const f28_t h2 = f28_twice(h), r2 = f28_twice(r);
    a.z = f28_mul(f28_mul(a.z, b.z), h2);
    const f28_t i = f28_sqr(h2);  // limbs 2 x 2
    const f28_t j = f28_mul(h, i), v = f28_mul(u1, i);
    a.x = f28_carry(f28_sub(f28_sub(f28_sqr(r2), j), f28_twice(v)));
    // r (V - X3) - 2 S1 J: limbs 2 x 1 + 1 x 2
    f28_t nj;
#pragma unroll
    for (int k = 0; k < 14; k++) nj.v[k] = -2 * j.v[k];
    a.y = f28_dot<2, false>(r2, f28_sub(v, a.x), s1, nj);
}

// ---- a point on a lane quad: the four lanes hold the same point and share each operation, one
// product per lane and level (three levels a doubling, four an addition, fp_row.hpp's
// schedules), results moving by DPP quad permutations.  Between the row form (a wave per point)
// and the lane form in latency and in work: on an idle SIMD a doubling takes 3.5 us and an
// addition 6.5, for sixteen points at once.
// (the empty asm keeps the permutation a move of its own: folded into a reversed subtraction,
// v_subrev_u32_dpp, the lane's own value was read instead of the permuted one)
template <int P0, int P1, int P2, int P3>
FDEV f28_t f28_perm(const f28_t& x) {
    f28_t r;
#pragma unroll
    for (int i = 0; i < 14; i++) {
        r.v[i] = __builtin_amdgcn_update_dpp(0, x.v[i], P0 | P1 << 2 | P2 << 4 | P3 << 6, 0xf, 0xf, true);
        asm("" : "+v"(r.v[i]));
    }
    return r;
}
template <int K>
FDEV f28_t f28_quad(const f28_t& x) {  // lane K's
    return f28_perm<K, K, K, K>(x);
}
FDEV f28_t f28_sel(bool c, const f28_t& a, const f28_t& b) {
    f28_t r;
#pragma unroll
    for (int i = 0; i < 14; i++) r.v[i] = c ? a.v[i] : b.v[i];
    return r;
}
FDEV f28_t f28_sel4(int q, const f28_t& a, const f28_t& b, const f28_t& c, const f28_t& d) {
    return f28_sel(q == 0, a, f28_sel(q == 1, b, f28_sel(q == 2, c, d)));
}
// a 144-byte point to and from a quad, lane q < 3 converting coordinate q
FDEV g28_t g28q_load(const uint32_t* p, int q, bool& inf) {
    uint32_t any;
    const f28_t t = f28_from_words(p + 12 * (q < 3 ? q : 2), any);
    inf = __builtin_amdgcn_update_dpp(0, (int)any, 0xaa, 0xf, 0xf, true) == 0;  // lane 2's: z = 0
    return {f28_quad<0>(t), f28_quad<1>(t), f28_quad<2>(t)};
}
FDEV void g28q_store(uint32_t* p, const g28_t& a, int q) {
    if (q < 3) f28_to_words(p + 12 * q, f28_sel4(q, a.x, a.y, a.z, a.z));
}
// q: the lane in its quad; a not at infinity.  zz, zzz: lane 3's are a's Z^2 and Z^3
FDEV g28_t g28q_dbl(const g28_t& a, int q, f28_t& zz, f28_t& zzz) {
    // X X, Y Y, Y Z, Z Z
    f28_t t = f28_mul(f28_sel4(q, a.x, a.y, a.y, a.z), f28_sel4(q, a.x, a.y, a.z, a.z));
    const f28_t A = f28_quad<0>(t), B = f28_quad<1>(t);
    g28_t o;
    o.z = f28_twice(f28_quad<2>(t));
    zz = t;
    f28_t E, u;
#pragma unroll
    for (int i = 0; i < 14; i++) E.v[i] = 3 * A.v[i];
    E = f28_carry(E);
    // B B, X B, E E, Z^2 Z
    t = f28_mul(f28_sel4(q, B, a.x, E, t), f28_sel4(q, B, B, E, a.z));
    zzz = t;
    const f28_t C = f28_quad<0>(t), XB = f28_quad<1>(t), F = f28_quad<2>(t);
#pragma unroll
    for (int i = 0; i < 14; i++) u.v[i] = F.v[i] - 8 * XB.v[i];
    o.x = f28_carry(u);
#pragma unroll
    for (int i = 0; i < 14; i++) u.v[i] = 4 * XB.v[i] - o.x.v[i];
    t = f28_mul(E, f28_carry(u));
#pragma unroll
    for (int i = 0; i < 14; i++) u.v[i] = t.v[i] - 8 * C.v[i];
    o.y = f28_carry(u);
    return o;
}
// a += b (b not at infinity) in g1z_add's four levels; inf: a's flag.  next() is called once b
// has been read (its registers are free for what is loaded ahead)
template <typename Next>
FDEV void g28q_add(g28_t& a, bool& inf, const g28_t& b, const f28_t& zz2, const f28_t& zzz2, int q, Next next) {
    if (inf) {
        a = b;
        inf = false;
        next();
        return;
    }
    // Z1^2, S1 = Y1 Z2^3, Y2 Z1, Z1 Z2
    f28_t t = f28_mul(f28_sel4(q, a.z, a.y, b.y, a.z), f28_sel4(q, a.z, zzz2, a.z, b.z));
    const f28_t S1 = f28_quad<1>(t), ZZ = f28_quad<3>(t);
    // U2 = X2 Z1^2, U1 = X1 Z2^2, S2 = Y2 Z1 Z1^2
    t = f28_mul(f28_sel(q == 0, b.x, f28_sel(q == 1, a.x, t)), f28_sel(q == 1, zz2, f28_quad<0>(t)));
    next();
    const f28_t U1 = f28_quad<1>(t);
    const f28_t H = f28_sub(f28_quad<0>(t), U1), R = f28_sub(f28_quad<2>(t), S1);
    const bool hz = f28_zero(H);
    if (hz && f28_zero(R)) {
        f28_t zz, zzz;
        inf = f28_zero(a.y);  // Z3 = 2 Y Z
        a = g28q_dbl(a, q, zz, zzz);
        return;
    }
    inf = hz;
    f28_t u;
#pragma unroll
    for (int i = 0; i < 14; i++) u.v[i] = 3 * U1.v[i] + H.v[i];
    // H H, R (3 U1 + H), R R, S1 H: limbs 1 x 4 at most
    t = f28_mul(f28_sel(q == 1 || q == 2, R, H), f28_sel4(q, H, u, R, S1));
    const f28_t HH2 = f28_twice(f28_quad<0>(t)), RR2 = f28_twice(f28_quad<2>(t));
    const f28_t P2 = f28_twice(f28_sub(f28_quad<1>(t), f28_quad<3>(t)));
#pragma unroll
    for (int i = 0; i < 14; i++) u.v[i] = H.v[i] + 2 * U1.v[i];
    // (H + 2 U1) 2 HH, Z1 Z2 2 H, 2 P 2 HH, 2 R 2 RR: limbs 3 x 2 at most
    t = f28_mul(f28_sel4(q, u, ZZ, P2, f28_twice(R)), f28_sel(q == 1, f28_twice(H), f28_sel(q == 3, RR2, HH2)));
    a.x = f28_carry(f28_twice(f28_sub(RR2, f28_quad<0>(t))));
    a.z = f28_quad<1>(t);
    a.y = f28_carry(f28_twice(f28_sub(f28_quad<2>(t), f28_quad<3>(t))));
}
