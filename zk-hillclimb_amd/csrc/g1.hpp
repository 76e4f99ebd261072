// g1.hpp -- host launchers of the G1 commitment kernels (g1.hip).
//
// Pedersen commitment by the bucket method, producing the reference's commit_pippenger
// result byte for byte (commitment.cu:47-103): for every row of a [m][n] scalar table,
// out[row] = sum_i s[row][i] * gens[i] over 4-bit windows of the scalar's raw limbs.
// Points are 144-byte G1Jacobian_t in Montgomery form, array-of-structures.
//
// The reference runs one thread per (row, window) that walks all n generators adding
// each into one of 16 buckets.  Here the work is split where the Jacobian result allows
// it -- each bucket's additions form an independent chain (its generators in ascending
// index order) -- after the chains' generator indices have been listed:
//   pip_gens    generators in row form with Z^2, Z^3; the plan's counters cleared
//   pip_sort    a block per row, lane w = window w: per-digit counts, then the index
//               lists (uint16, generators in ascending order) and their offsets
//   pip_alias   a block per row: chains whose index lists are equal (the usual case for
//               small signed scalars, where every window above the witness width holds
//               the list of negative entries) are computed once; lists are matched by a
//               fingerprint and confirmed entry by entry.  Windows whose digits share
//               their buckets are summed once
//   pip_bucket  plan and sort of the distinct nonempty chains by length, then each once: the
//               long ones on a wave each (latency), the others on a lane each (throughput)
//   pip_window  each distinct window once: the running sum over digits 15..1
//   pip_combine one wave per row: Horner over windows 63..0 (four doublings, one add)
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define ZKH_PIP_MAX_GENS 65536u  // generator indices are stored as uint16

// scalars: FR limb planes (lo: limbs 0-3, hi: limbs 4-7 as uint4 per element), m*n entries
void launch_pip_sort(hipStream_t s, const uint32_t* lo, const uint32_t* hi, uint32_t m, uint32_t n,
                     uint16_t* lists, uint32_t* offs);
#define ZKH_ROW_WORDS 48       // a point in row form (fp_row.hpp)
#define ZKH_POINTZ_WORDS 80    // and with Z^2 and Z^3 behind it
#define PIP_BINS 288           // chain length classes
struct PipPlan {
    uint32_t total[PIP_BINS];   // distinct chains per length class
    uint32_t cursor[PIP_BINS];  // the class's next place in the sorted list
    uint32_t items, waves;      // chains, and how many of the longest go to waves
    uint32_t nwin;              // distinct windows
    uint32_t taken[2];          // queues of the bucket launch: wave chains, lane groups
    uint32_t pad[3];
};
void launch_pip_gens(hipStream_t s, const uint32_t* gens, uint32_t n, uint32_t* tab, PipPlan* plan);
void launch_pip_alias(hipStream_t s, const uint16_t* lists, const uint32_t* offs, uint32_t m, uint32_t n,
                      uint16_t* alias, uint16_t* walias, PipPlan* plan, uint32_t* wins);
void launch_pip_bucket(hipStream_t s, const uint32_t* tab, const uint16_t* lists, const uint32_t* offs,
                       const uint16_t* alias, uint32_t m, uint32_t n, PipPlan* plan, uint32_t* items,
                       uint32_t* buckets);
void launch_pip_window(hipStream_t s, const uint32_t* buckets, const uint32_t* offs, const uint16_t* alias,
                       uint32_t m, const PipPlan* plan, const uint32_t* wins, uint32_t* partials);
void launch_pip_combine(hipStream_t s, const uint32_t* partials, const uint16_t* walias, uint32_t m, uint32_t* out);
// inner-product argument rounds (ipa_prove) of up to ZKH_IPA_MAX_JOBS openings per launch
// (blockIdx.y = job); a, b plain Fr 8 words per entry.  g, g2, Qr, P: points in row form
// (fp_row.hpp, ZKH_ROW_WORDS each); g_in, Q: 144-byte points; LR: two 144-byte points (host).
// A job with h = 0 has finished its rounds and is skipped.  x, xi plain; xm, xim in
// Montgomery form.
#define ZKH_IPA_MAX_JOBS 8
struct IpaJobDev {
    const uint32_t *g_in, *Q, *g, *a, *b, *Qr;
    uint32_t *g0, *P, *LR, *g2, *a2, *b2;
    uint32_t h, scale0, fold0, pt0;  // the job's first block of a scale and fold launch, first point
    uint32_t x[8], xi[8], xm[8], xim[8];
};
// D: the points' tables (2^i g, i < 255), cap of them: of points [slice0, slice0 + cap) where
// there are more (the points of all jobs in order, ipa_table; cap is even then)
#define ZKH_IPA_TABLES 24576u
#define ZKH_TABLE_WORDS (255u * ZKH_POINTZ_WORDS)
struct IpaBatchDev {
    IpaJobDev j[ZKH_IPA_MAX_JOBS];
    uint32_t* D;
    uint32_t slice0, slice;  // the first point whose table is at hand, and how many are
    uint32_t cap, pad_;
};
// g0[0, 2h] = row forms of g_in[0, 2h) and Q
void launch_ipa_points(hipStream_t s, const IpaBatchDev& B, uint32_t nj, uint32_t hmax);
void launch_ipa_scale(hipStream_t s, IpaBatchDev& B, uint32_t nj, const uint32_t r2[8]);
// every tree level and L, R (hmax the largest h)
void launch_ipa_tree(hipStream_t s, const IpaBatchDev& B, uint32_t nj, uint32_t hmax);
void launch_ipa_fold(hipStream_t s, IpaBatchDev& B, uint32_t nj);
void launch_planes_to_aos(hipStream_t s, const uint32_t* lo, const uint32_t* hi, uint32_t n, uint32_t* out);
// out[i] = base[i % nb] * s[i] (G1Jacobian_mul, raw scalar bits)
// a scalar passed by value to a kernel: 8 plain little-endian words
struct G1Scalar {
    uint32_t v[8];
};
// out[i] = b[i] + a[i] * sc (hb_addmul, mul_first = false)
void launch_g1_addmul(hipStream_t s, const uint32_t* a, const G1Scalar& sc, const uint32_t* b, uint32_t n,
                      uint32_t* out);
void launch_g1_mul(hipStream_t s, const uint32_t* base, uint32_t nb, const uint32_t* lo, const uint32_t* hi,
                   uint32_t n, uint32_t* out, uint32_t* tab, uint32_t nt, uint32_t* tops);
// its scratch: tab, tables of nt bases (ZKH_TABLE_WORDS each; want of them, fewer down to least,
// or none), and tops, ZKH_G1_TOPS words beside tables
#define ZKH_G1_TOPS 256u
void g1_mul_tables(uint32_t nb, uint32_t n, uint32_t* want, uint32_t* least);
