// fp_row.hpp -- BLS12-381 Fp and G1 with every element spread over the 16 lanes of a DPP row.
//
// A G1 point in memory is {x, y, z} Jacobian, 144 bytes, the reference's G1Jacobian_t: each
// coordinate 12 x 32-bit limbs, little-endian, canonical in [0, p), in Montgomery form with R =
// 2^384 (bls12-381.cuh:220-229, g1-tensor.cuh:26-63); {0, ONE, 0} is the point at infinity
// (bls12-381.cuh:422).  The representative of a group operation depends on the formula, and
// the bytes of a commitment are absorbed by the transcript: doubling is dbl-2009-l and addition
// add-2007-bl with the reference's infinity and equal-point branches (bls12-381.cu:1359-1465).
// Any computation of the same field elements gives the same bytes.
//
// A scalar multiply (G1Jacobian_mul, g1-tensor.cu:445-454) is one chain of dependent point
// operations, and its length is the latency of a field product times the chain's depth.  With
// a whole element of 32-bit limbs per lane a product is ~750 instructions in sequence; here
// lane k of a row holds limb k (14 limbs of 28 bits), a product is ~107 instructions, and the
// four rows of a wave run the up to four independent products of a point operation's level
// side by side: one wave per point, a doubling is three levels and an addition five.  On an
// idle SIMD a doubling takes 0.77 us and an addition 1.28 (32-bit limbs on a lane quad per
// point: 6.9 and 13.5); with the SIMD full, 0.64 and 1.06 us of its time per point (0.30 and
// 0.59), so this form is for chains whose latency counts.
//
// Form: Montgomery with R' = 2^392, residues not canonical: a product is below 3 p with limbs
// below 2^28 + 16, sums are taken limb by limb and renormalised by one carry pass where the next
// use needs it.  The bound on every value is written beside it; canonical values exist only at
// g1r_store and in the exact tests.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#ifndef FDEV
#define FDEV __device__ __forceinline__
#endif
#include "fp_row_consts.inc"

#define FPR_MASK 0x0fffffffu

// the constants of this lane's limb
struct fpr_k {
    uint32_t p, m, ka, kb;
    uint32_t lane;  // lane in the row
    uint32_t row;
};
__device__ const uint32_t k_fpr_tab[7][16] = {{FPR_P_LIMBS},  {FPR_M_LIMBS},   {FPR_KA_LIMBS}, {FPR_KB_LIMBS},
                                              {FPR_IN_LIMBS}, {FPR_OUT_LIMBS}, {FPR_ONE_LIMBS}};
FDEV fpr_k fpr_consts() {
    fpr_k c;
    c.lane = threadIdx.x & 15;
    c.row = (threadIdx.x >> 4) & 3;
    c.p = k_fpr_tab[0][c.lane];
    c.m = k_fpr_tab[1][c.lane];
    c.ka = k_fpr_tab[2][c.lane];
    c.kb = k_fpr_tab[3][c.lane];
    return c;
}

// ---- movement inside a row (DPP) and between rows (permlane swaps) ----
// The compiler folds these moves into the additions that use them.  None feeds a subtraction:
// folded into v_subrev_u32_dpp such a move gave wrong results in f28_perm (fp_lane28.hpp, whose
// guard a subtraction here would need too).
template <int I>
FDEV uint32_t row_bcast(uint32_t x) {  // lane I of the row to all its lanes
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x150 + I, 0xf, 0xf, true);
}
FDEV uint32_t row_up(uint32_t x) {  // lane k takes lane k - 1's (lane 0: 0)
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, true);
}
// rows (r0, r1, r2, r3) of x: lo = (r0, r1, r0, r1), hi = (r2, r3, r2, r3)
FDEV void rows_halves(uint32_t x, uint32_t& lo, uint32_t& hi) {
    const auto s = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    lo = s[0];
    hi = s[1];
}
// rows (r0, r1, r2, r3) of x: even = (r0, r0, r2, r2), odd = (r1, r1, r3, r3)
FDEV void rows_pairs(uint32_t x, uint32_t& even, uint32_t& odd) {
    const auto s = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    even = s[0];
    odd = s[1];
}

// ---- field ----
// one carry pass: limbs below 2^32 to limbs below 2^28 + 16 (the top limb keeps its value's
// high part: every value here is below 2^392)
FDEV uint32_t fpr_norm(uint32_t x) { return (x & FPR_MASK) + row_up(x >> 28); }

// a b / R' mod p, below (alpha beta / 2520 + 2) p for operands below alpha p and beta p (p =
// 2^392 / 2520): every use here keeps it below 2.96 p, or 4 p where that is written; limbs
// below 2^28 + 16.  Limbs of a and b: their products below 13 x 2^56 (the largest here are 9 x
// 2^56), so that with m M's 2^56 and a carry the sum stays below 15 x 2^56 and its carry, plus the
// 28-bit limb that moves in beside it, below 2^32.
//
// Lane k's v[4:5] holds the sum's limb k.  A step I drops the cleared limb 0 (its low 28 bits m
// go to every lane), moves the limbs down one lane with their carries, and adds a_I b and the
// multiple of p that cleared limb 0: that is m M after the shift (gen_fp_row.py), with m the
// limb itself instead of a product.  The last step takes m = acc_0 n0 and adds m p before
// the shift: the steps before it leave a multiple of 2^28 p above the residue that only this
// form brings below 2 p.  Straight-line code with its own registers, ordered so that two
// instructions lie between a register's write and its DPP read; as separate statements the
// compiler adds a 64-bit add and two wait states per step (0.90 against 0.77 us per
// doubling).  Nearly all of it is 8-byte instructions, aligned so by a no-op where the code
// before it is not: four bytes off, a wave alone on its SIMD takes 3 to 6 % longer (a 16384-term
// row's commitment 11.4 and 10.5 ms, an opening of 64 points 2.61 and 2.44), and which way it
// lies changed with every edit of the file; on full SIMDs the no-ops cost 1 to 3 %.
#define FPR_SHIFT                                                               \
    "v_and_b32_e32 v8, 0xfffffff, v4\n\t"                                     \
    "v_alignbit_b32 v9, v5, v4, 28\n\t"
#define FPR_STEP(I)                                                             \
    FPR_SHIFT                                                                   \
    "v_mov_b32_dpp v6, %1 row_newbcast:" #I " row_mask:0xf bank_mask:0xf\n\t"  \
    "v_mov_b32_dpp v7, v8 row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"       \
    "v_add_u32_dpp v2, v8, v9 row_shl:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t" \
    "v_mad_u64_u32 v[4:5], vcc, v6, %2, v[2:3]\n\t"                           \
    "v_mad_u64_u32 v[4:5], vcc, v7, %3, v[4:5]\n\t"
FDEV uint32_t fpr_mul(uint32_t a, uint32_t b, const fpr_k& c) {
    uint32_t r;
    asm(".p2align 3\n\t"
        "v_mov_b32_e32 v3, 0\n\t"
        "s_nop 0\n\t"
        "v_mov_b32_dpp v6, %1 row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
        "v_mad_u64_u32 v[4:5], vcc, v6, %2, 0\n\t"
        FPR_STEP(1) FPR_STEP(2) FPR_STEP(3) FPR_STEP(4) FPR_STEP(5) FPR_STEP(6) FPR_STEP(7)
        FPR_STEP(8) FPR_STEP(9) FPR_STEP(10) FPR_STEP(11) FPR_STEP(12) FPR_STEP(13)
        "v_mul_lo_u32 v6, v4, %5\n\t"
        "s_nop 1\n\t"
        "v_mov_b32_dpp v7, v6 row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
        "v_and_b32_e32 v7, 0xfffffff, v7\n\t"
        "v_mad_u64_u32 v[4:5], vcc, v7, %4, v[4:5]\n\t"
        FPR_SHIFT
        "s_nop 0\n\t"
        "v_add_u32_dpp v8, v8, v9 row_shl:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
        "v_lshrrev_b32_e32 v9, 28, v8\n\t"
        "v_and_b32_e32 v8, 0xfffffff, v8\n\t"
        "s_nop 0\n\t"
        "v_add_u32_dpp %0, v9, v8 row_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
        "s_nop 1"  // the next instruction may read the result by DPP or a permlane swap
        : "=v"(r)
        : "v"(a), "v"(b), "v"(c.m), "v"(c.p), "s"(FPR_N0)
        : "v2", "v3", "v4", "v5", "v6", "v7", "v8", "v9", "vcc");
    return r;
}

// ---- exact values (stores and rare branches) ----
// signed carries to limbs in [0, 2^28), the top limb (lane 13) keeping the sign
FDEV int32_t fpr_ripple(int32_t x, const fpr_k& c) {
    for (;;) {
        const int32_t h = c.lane >= 13 ? 0 : x >> 28;
        if (!__any(h != 0)) return x;
        x = x - (int32_t)((uint32_t)h << 28) + (int32_t)row_up((uint32_t)h);
    }
}
// the canonical residue of x (limbs below 2^31, value below 2^(TOP + 1) p)
template <int TOP>
FDEV uint32_t fpr_canon(uint32_t x, const fpr_k& c) {
    int32_t v = fpr_ripple((int32_t)x, c);
#pragma unroll 1
    for (int sh = TOP; sh >= 0; sh--) {  // v - 2^sh p where that is not negative
        int32_t d = v;
#pragma unroll 1
        for (int k = 0; k < (1 << (sh > 2 ? sh - 2 : 0)); k++)  // p's limbs times at most 4: below 2^30
            d = fpr_ripple(d - (int32_t)(c.p << (sh > 2 ? 2 : sh)), c);
        v = (int32_t)row_bcast<13>((uint32_t)d) < 0 ? v : d;
    }
    return (uint32_t)v;
}
// whether x, equal in the wave's four rows and below 64 p (limbs below 2^32), is a multiple of
// p: a multiple j p has limb 0 = j p_0 mod 2^28, so all but 2^-22 of the other values stop here
FDEV bool fpr_zero(uint32_t x, const fpr_k& c) {
    const uint32_t j = ((uint32_t)__builtin_amdgcn_readfirstlane((int)x) * FPR_PINV) & FPR_MASK;
    if (j >= 64) return false;
    return !__any(fpr_canon<5>(fpr_norm(x), c) != 0);
}

// ---- points: x, y, z replicated in the wave's four rows ----
struct g1r_t {
    uint32_t x, y, z;
    bool inf;  // z = 0 mod p (wave-uniform)
};
FDEV uint32_t row_sel(const fpr_k& c, uint32_t r0, uint32_t r1, uint32_t r2, uint32_t r3) {
    uint32_t v = c.row == 1 ? r1 : r0;
    v = c.row == 2 ? r2 : v;
    return c.row == 3 ? r3 : v;
}
FDEV g1r_t g1r_zero(const fpr_k& c) {
    g1r_t o;
    o.x = o.z = 0;
    o.y = k_fpr_tab[6][c.lane];
    o.inf = true;
    return o;
}
// limb `lane` of a canonical 12-word value at w (28 bits from bit 28 lane on)
FDEV uint32_t fpr_unpack(const uint32_t* w, const fpr_k& c) {
    const uint32_t bit = 28 * c.lane, i = bit >> 5, off = bit & 31;
    if (c.lane > 13) return 0;
    uint32_t v = w[i] >> off;
    if (off > 4 && i < 11) v |= w[i + 1] << (32 - off);
    return v & FPR_MASK;
}
// a point in memory or LDS in row form: 16 words each for x, y, z (14 limbs), word 14 the flag
#define G1R_WORDS 48
FDEV uint32_t g1r_word(const g1r_t& a, const fpr_k& c) {  // this lane's word (row 3: unused)
    return c.row == 0 && c.lane == 14 ? (a.inf ? 1u : 0u) : row_sel(c, a.x, a.y, a.z, a.z);
}
FDEV void g1r_put(uint32_t* p, const g1r_t& a, const fpr_k& c) {
    const uint32_t v = g1r_word(a, c);
    if (c.row < 3) p[threadIdx.x & 63] = v;
}
// the words of a point as loaded: taken apart only where the point is used, so that a load made
// ahead does not wait
struct g1r_raw {
    uint32_t x, y, z;
};
FDEV g1r_raw g1r_fetch(const uint32_t* p, const fpr_k& c) { return {p[c.lane], p[16 + c.lane], p[32 + c.lane]}; }
FDEV g1r_t g1r_take(const g1r_raw& w, const fpr_k& c) {
    g1r_t o;
    o.x = c.lane < 14 ? w.x : 0;
    o.y = w.y;
    o.z = w.z;
    o.inf = __builtin_amdgcn_readfirstlane((int)row_bcast<14>(w.x)) != 0;
    return o;
}
FDEV g1r_t g1r_get(const uint32_t* p, const fpr_k& c) { return g1r_take(g1r_fetch(p, c), c); }
// a second operand with its Z^2 and Z^3 (known ahead, they take a level off an addition), in
// memory as the point and 16 words each behind it
#define G1Z_WORDS 80
struct g1z_t {
    g1r_t p;
    uint32_t zz, zzz;
};
struct g1z_raw {
    g1r_raw p;
    uint32_t zz, zzz;
};
FDEV g1z_raw g1z_fetch(const uint32_t* p, const fpr_k& c) {
    return {g1r_fetch(p, c), p[G1R_WORDS + c.lane], p[G1R_WORDS + 16 + c.lane]};
}
FDEV g1z_t g1z_take(const g1z_raw& w, const fpr_k& c) { return {g1r_take(w.p, c), w.zz, w.zzz}; }
// this lane's words of an entry: word tid, and word 64 + tid for the lanes of row 0
FDEV uint32_t g1z_word(const g1z_t& a, const fpr_k& c) {
    return c.row == 0 && c.lane == 14 ? (a.p.inf ? 1u : 0u) : row_sel(c, a.p.x, a.p.y, a.p.z, a.zz);
}
FDEV void g1z_put(uint32_t* p, uint32_t word, const g1z_t& a, const fpr_k& c) {
    p[threadIdx.x & 63] = word;
    if (c.row == 0) p[64 + c.lane] = a.zzz;
}
// 144-byte point: row r converts coordinate r
FDEV g1r_t g1r_load(const uint32_t* p, const fpr_k& c) {
    const uint32_t raw = fpr_unpack(p + 12 * (c.row < 3 ? c.row : 2), c);
    const uint32_t v = fpr_mul(raw, k_fpr_tab[4][c.lane], c);
    g1r_t o;
    uint32_t lo, hi, d;
    rows_halves(v, lo, hi);
    rows_pairs(lo, o.x, o.y);
    rows_pairs(hi, o.z, d);
    o.inf = !__any(c.row == 2 && raw != 0);
    return o;
}
FDEV void g1r_store(uint32_t* p, const g1r_t& a, const fpr_k& c) {
    const uint32_t v = fpr_canon<1>(fpr_mul(row_sel(c, a.x, a.y, a.z, a.z), k_fpr_tab[5][c.lane], c), c);
    // word j = bits 32 j .. 32 j + 31: limbs l, l + 1 and, from offset 25 on, l + 2
    const uint32_t bit = 32 * c.lane, l = bit / 28, off = bit % 28;
    const uint32_t base = threadIdx.x & 0x30;
    const uint32_t w0 = (uint32_t)__shfl((int)v, (int)(base + (l & 15)));
    const uint32_t w1 = (uint32_t)__shfl((int)v, (int)(base + ((l + 1) & 15)));
    const uint32_t w2 = (uint32_t)__shfl((int)v, (int)(base + ((l + 2) & 15)));
    uint32_t w = (w0 >> off) | (w1 << (28 - off));
    if (off > 24) w |= w2 << (56 - off);
    if (c.lane < 12 && c.row < 3) p[12 * c.row + c.lane] = w;
}

// Coordinates between operations: x, y below 45 p with limbs below 2^28 + 16, z below 36 p with
// limbs below 2^29 + 32 (z below 6 p from the operations here, up to 36 p from fp_lane28.hpp's
// stores); Z^2, Z^3 below 3 p.
//
// dbl-2009-l with D = 4 X B for 2 ((X + B)^2 - A - C): A = X^2, B = Y^2, C = B^2, E = 3 A,
// F = E^2, X3 = F - 2 D, Y3 = E (D - X3) - 8 C, Z3 = 2 Y Z; Z = 0 returns the point unchanged
// (a.zz, a.zzz: its own Z^2 and Z^3 on the way, in the rows the formula leaves free)
FDEV g1r_t g1z_dbl(g1z_t& az, const fpr_k& c) {
    const g1r_t& a = az.p;
    if (a.inf) return a;
    uint32_t lo, hi, A, B, C, XB, YZ, F;
    // rows: X X, Y Y, Y Z, Z Z
    uint32_t t = fpr_mul(row_sel(c, a.x, a.y, a.y, a.z), row_sel(c, a.x, a.y, a.z, a.z), c);
    rows_halves(t, lo, hi);
    rows_pairs(lo, A, B);
    rows_pairs(hi, YZ, az.zz);
    g1r_t o;
    o.z = 2 * YZ;
    const uint32_t E = 3 * A;  // below 9 p, limbs below 2^29.6
    // rows: B B, X B, E E, Z^2 Z
    t = fpr_mul(row_sel(c, B, a.x, E, t), row_sel(c, B, B, E, a.z), c);
    rows_halves(t, lo, hi);
    rows_pairs(lo, C, XB);
    rows_pairs(hi, F, az.zzz);
    o.x = fpr_norm(F + (c.ka - 8 * XB));                  // below 27 p
    t = fpr_mul(E, fpr_norm(4 * XB + (c.kb - o.x)), c);  // D - X3 below 44 p
    o.y = fpr_norm(t + (c.ka - 8 * C));                   // below 27 p
    o.inf = fpr_zero(a.y, c);                             // Z3 = 2 Y Z with Z not 0
    return o;
}
FDEV g1r_t g1r_dbl(const g1r_t& a, const fpr_k& c) {
    g1z_t z{a, 0, 0};
    return g1z_dbl(z, c);
}

// add-2007-bl with Z3 = 2 Z1 Z2 H for ((Z1 + Z2)^2 - Z1Z1 - Z2Z2) H: an operand at infinity returns
// the other unchanged, U1 = U2 and S1 = S2 doubles the first operand, and U1 = U2 with S1 != S2
// runs the general formula (Z3 = 0)
FDEV g1r_t g1r_add(const g1r_t& a, const g1r_t& b, const fpr_k& c) {
    if (a.inf) return b;
    if (b.inf) return a;
    uint32_t lo, hi, ev, od, H, R, I, ZZ, J, V;
    const bool odd = c.row & 1, low = c.row < 2;
    // rows: Z2^2, Z1^2, Y1 Z2, Y2 Z1
    uint32_t t = fpr_mul(low ? (odd ? a.z : b.z) : (odd ? b.y : a.y), odd ? a.z : b.z, c);
    rows_halves(t, lo, hi);
    // rows: U1 = X1 Z2Z2, U2 = X2 Z1Z1, S1 = Y1 Z2 Z2Z2, S2 = Y2 Z1 Z1Z1
    t = fpr_mul(low ? (odd ? b.x : a.x) : t, lo, c);
    rows_pairs(t, ev, od);                       // (U1, S1), (U2, S2)
    const uint32_t d = fpr_norm(od + (c.kb - ev));  // (H, S2 - S1): below 35 p
    rows_halves(d, H, R);
    g1r_t o;
    o.inf = fpr_zero(H, c);
    if (o.inf && fpr_zero(R, c)) return g1r_dbl(a, c);
    // rows: I = (2 H)^2, Z1 Z2, r^2, r^2 with r = 2 (S2 - S1): below 4 p
    t = fpr_mul(c.row == 1 ? a.z : 2 * d, c.row == 1 ? b.z : 2 * d, c);
    uint32_t rr;
    rows_halves(t, lo, rr);
    rows_pairs(lo, I, ZZ);
    // rows: J = H I, V = U1 I, Z1 Z2 H, Z1 Z2 H
    t = fpr_mul(c.row == 1 ? ev : H, low ? I : ZZ, c);
    rows_halves(t, lo, hi);
    rows_pairs(lo, J, V);
    o.z = 2 * hi;
    o.x = fpr_norm(rr + (c.ka - J - 2 * V));  // below 28 p
    // rows: r (V - X3) twice, S1 J twice
    t = fpr_mul(low ? 2 * R : ev, low ? fpr_norm(V + (c.kb - o.x)) : J, c);
    rows_halves(t, lo, hi);
    o.y = fpr_norm(lo + (c.ka - 2 * hi));  // below 27 p
    return o;
}

// The same with Z2^2 and Z2^3 at hand, in four levels.  With H = U2 - U1, R = S2 - S1 the
// formula's I = 4 H^2, J = H I, V = U1 I, r = 2 R give
//   X3 = r^2 - J - 2 V            = 4 R^2 - 4 (H + 2 U1) H^2
//   Y3 = r (V - X3) - 2 S1 J      = 8 [(R (3 U1 + H) - S1 H) H^2 - R R^2]
//   Z3 = 2 Z1 Z2 H
// so that no product waits for X3 (five levels in g1r_add: 1.28 us on an idle SIMD, 1.05 here).
FDEV g1r_t g1z_add(const g1r_t& a, const g1z_t& bz, const fpr_k& c) {
    const g1r_t& b = bz.p;
    if (a.inf) return b;
    if (b.inf) return a;
    uint32_t lo, hi, ev, od, H, R, U1, S1, x;
    const bool low = c.row < 2;
    // rows: Z1^2, S1 = Y1 Z2^3, Y2 Z1, Z1 Z2
    uint32_t t = fpr_mul(row_sel(c, a.z, a.y, b.y, a.z), row_sel(c, a.z, bz.zzz, a.z, b.z), c);
    rows_halves(t, lo, hi);
    const uint32_t ZZ = hi;  // (row 1)
    rows_pairs(lo, x, S1);
    // rows: U2 = X2 Z1^2, U1 = X1 Z2^2, S2 = Y2 Z1 Z1^2, -
    t = fpr_mul(row_sel(c, b.x, a.x, t, t), c.row == 1 ? bz.zz : lo, c);
    rows_pairs(t, ev, od);
    rows_halves(od, U1, x);
    const uint32_t d = fpr_norm(ev + (c.kb - (low ? od : S1)));  // (H, R): below 35 p
    rows_halves(d, H, R);
    g1r_t o;
    o.inf = fpr_zero(H, c);
    if (o.inf && fpr_zero(R, c)) return g1r_dbl(a, c);
    // rows: H H, R (3 U1 + H), R R, S1 H
    t = fpr_mul(c.row == 1 || c.row == 2 ? R : H, row_sel(c, H, 3 * U1 + H, R, S1), c);
    uint32_t HH, RR, P1, P2;
    rows_pairs(t, ev, od);
    rows_halves(ev, HH, RR);
    rows_halves(od, P1, P2);
    const uint32_t q = fpr_norm(P1 + (c.kb - P2));  // below 35 p
    // rows: (H + 2 U1) 2 HH, Z1 Z2 2 H, 4 q 2 HH, 4 R 2 RR: limbs below 2^29.6 x 2^29 and 2^30 x 2^29
    t = fpr_mul(row_sel(c, H + 2 * U1, ZZ, 4 * q, 4 * R), 2 * row_sel(c, HH, H, HH, RR), c);
    uint32_t X, Y8, R8;
    rows_halves(t, lo, hi);
    rows_pairs(lo, X, o.z);
    rows_pairs(hi, Y8, R8);
    o.x = fpr_norm(4 * RR + (c.kb - 2 * X));  // below 44 p
    o.y = fpr_norm(Y8 + (c.kb - R8));         // below 35 p
    return o;
}
