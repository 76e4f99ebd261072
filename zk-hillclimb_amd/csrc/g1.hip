// g1.hip -- G1 Pedersen commitment kernels (bucket method, commitment.cu:47-103).
#include "fp_lane28.hpp"
#include "fp_row.hpp"
#include "fr_dev.hpp"
#include "g1.hpp"

// A block per row, lane w of every wave owning window w (bits 4w..4w+3 of the raw scalar,
// commitment.cu:50-55): a wave reads limb w/8 of its eighth of the elements and counts the
// digits in its LDS row; one wave turns the counts into offsets, per digit and eighth; then
// every wave lists its elements with a nonzero digit under that digit (ascending: eighths in
// order).  Lists hold at most n entries per (row, window); offs[.][0] is the total, offs[.][d]
// the start of digit d.  One wave per row walked the elements through one chain of LDS updates:
// 0.61 ms at 512 x 2048 against 0.38 (the 2-byte stores into 64 lists are most of that).
#define PIP_SEG 8
__global__ __launch_bounds__(64 * PIP_SEG) void k_pip_sort(const uint32_t* __restrict__ lo,
                                                           const uint32_t* __restrict__ hi, uint32_t n,
                                                           uint16_t* __restrict__ lists,
                                                           uint32_t* __restrict__ offs) {
    __shared__ uint32_t cnt[PIP_SEG][64][17];
    const uint32_t row = blockIdx.x, w = threadIdx.x & 63, seg = threadIdx.x >> 6;
    const uint32_t limb = w >> 3, sh = 4 * (w & 7);
    const uint32_t* src = (limb < 4 ? lo : hi) + (limb & 3) + 4 * (size_t)row * n;
    const uint32_t i0 = (uint32_t)((uint64_t)n * seg / PIP_SEG), i1 = (uint32_t)((uint64_t)n * (seg + 1) / PIP_SEG);
    uint32_t* my = cnt[seg][w];
#pragma unroll
    for (int d = 0; d < 16; d++) my[d] = 0;
#pragma unroll 8
    for (uint32_t i = i0; i < i1; i++) my[(src[4 * (size_t)i] >> sh) & 15u] += 1;
    __syncthreads();
    const size_t rw = (size_t)row * 64 + w;
    if (seg == 0) {
        uint32_t* o = offs + rw * 16;
        uint32_t run = 0;
        for (int d = 1; d < 16; d++) {
            o[d] = run;
            for (int s = 0; s < PIP_SEG; s++) {
                const uint32_t k = cnt[s][w][d];
                cnt[s][w][d] = run;
                run += k;
            }
        }
        o[0] = run;
    }
    __syncthreads();
    uint16_t* L = lists + rw * n;
#pragma unroll 8
    for (uint32_t i = i0; i < i1; i++) {
        const uint32_t d = (src[4 * (size_t)i] >> sh) & 15u;
        if (d) {
            const uint32_t pos = my[d];
            my[d] = pos + 1;
            L[pos] = (uint16_t)i;
        }
    }
}

// 64-bit mix of a generator index (the splitmix64 finaliser); a list's fingerprint is the
// sum over its entries, so equal sets give equal fingerprints in any order
__device__ __forceinline__ uint64_t pip_mix(uint64_t z) {
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// Identical chains.  A bucket is a fixed sequence of additions over its list, so two
// (window, digit) chains of a row with the same list produce the same bytes.  For small
// signed scalars this is the common case: a negative v is r - |v|, whose digits above
// |v|'s top window are those of r - 2^k for every such element, so the windows above
// the witness width all hold the list of negative entries under one digit each.  A block
// per row, its sixteen waves taking the chains in turn: each nonempty list is fingerprinted
// (count, sum of mixed indices; coalesced reads), then looked up among the earlier windows'
// chains, and the first one with an equal fingerprint confirmed entry by entry.  alias holds
// the (window * 16 + digit) whose bucket stands in, itself when there is none;
// representatives are always first occurrences.  One wave per row took 1.9 ms at 512 rows of
// 1024 field elements, sixteen 0.26.
__device__ __forceinline__ uint64_t wave_sum_u64(uint64_t v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
    return v;
}
// length class: exact below 128, then 16 per factor of two (n <= 65536)
__device__ __forceinline__ uint32_t pip_bin(uint32_t len) {
    if (len < 128) return len;
    const uint32_t l2 = 31 - __builtin_clz(len);
    return 128 + 16 * (l2 - 7) + ((len >> (l2 - 4)) & 15);
}
// the longest length of a class
__device__ __forceinline__ uint32_t pip_bin_len(uint32_t b) {
    if (b < 128) return b;
    const uint32_t l2 = 7 + (b - 128) / 16;
    return (1u << l2) + (((b - 128) % 16 + 1) << (l2 - 4)) - 1;
}

__global__ __launch_bounds__(1024) void k_pip_alias(const uint16_t* __restrict__ lists,
                                                    const uint32_t* __restrict__ offs, uint32_t n,
                                                    uint16_t* __restrict__ alias, uint16_t* __restrict__ walias,
                                                    PipPlan* __restrict__ plan, uint32_t* __restrict__ wins) {
    __shared__ uint32_t beg_s[1024], cnt_s[1024], hist[PIP_BINS];
    __shared__ uint64_t fp_s[1024];
    __shared__ uint16_t sig[1024];
    __shared__ uint32_t nwin, wbase;
    const uint32_t row = blockIdx.x, lane = threadIdx.x & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint16_t* Lrow = lists + (size_t)row * 64 * n;
    {
        const uint32_t c = threadIdx.x, d = c & 15;
        const uint32_t* o = offs + (size_t)row * 1024 + (c & ~15u);
        const uint32_t b = d ? o[d] : 0, e = d == 15 ? o[0] : d ? o[d + 1] : 0;
        beg_s[c] = b;
        cnt_s[c] = e - b;
        if (c < PIP_BINS) hist[c] = 0;
        if (c == 0) nwin = 0;
    }
    __syncthreads();
    for (uint32_t c = wave; c < 1024; c += 16) {
        const uint32_t cnt = cnt_s[c];
        uint64_t h = 0;
        if (cnt) {
            const uint16_t* L = Lrow + (size_t)(c >> 4) * n + beg_s[c];
            for (uint32_t k = lane; k < cnt; k += 64) h += pip_mix(L[k]);
            h = wave_sum_u64(h);
        }
        if (lane == 0) fp_s[c] = h;
    }
    __syncthreads();
    uint16_t* out = alias + (size_t)row * 1024;
    for (uint32_t c = wave; c < 1024; c += 16) {
        const uint32_t cnt = cnt_s[c];
        uint32_t target = c;
        if (cnt && c >= 16) {
            const uint64_t h = fp_s[c];
            const uint16_t* A = Lrow + (size_t)(c >> 4) * n + beg_s[c];
            // candidates in earlier windows, 64 at a time, lowest first (digit 0 has no list)
            for (uint32_t base = 0; base < (c & ~15u) && target == c; base += 64) {
                const uint32_t cc = base + lane;
                const bool hit = cc < (c & ~15u) && cnt_s[cc] == cnt && fp_s[cc] == h;
                uint64_t hits = __ballot(hit);
                while (hits && target == c) {
                    const uint32_t cand = base + __builtin_ctzll(hits);
                    hits &= hits - 1;
                    const uint16_t* B = Lrow + (size_t)(cand >> 4) * n + beg_s[cand];
                    bool diff = false;
                    for (uint32_t k = lane; k < cnt; k += 64) diff |= A[k] != B[k];
                    if (!__any(diff)) target = cand;
                }
            }
        }
        if (lane == 0) {
            out[c] = (uint16_t)target;
            sig[c] = cnt ? (uint16_t)target : 0xffff;  // the digit's bucket; none
            if (cnt && target == c) atomicAdd(&hist[pip_bin(cnt)], 1u);
        }
    }
    __syncthreads();
    // windows whose digits share their buckets share their sum: the first of them stands in
    // (small signed scalars: the windows above the witness width have r's digits, 15 at most)
    uint32_t first = 64, slot = 0;
    if (threadIdx.x < 64) {
        first = lane;
        for (uint32_t v = 0; v < lane && first == lane; v++) {
            bool same = true;
            for (uint32_t d = 15; d >= 1 && same; d--) same = sig[v * 16 + d] == sig[lane * 16 + d];
            if (same) first = v;
        }
        walias[(size_t)row * 64 + lane] = (uint16_t)first;
        if (first == lane) slot = atomicAdd(&nwin, 1u);
    }
    __syncthreads();
    if (threadIdx.x == 0) wbase = atomicAdd(&plan->nwin, nwin);
    for (uint32_t b = threadIdx.x; b < PIP_BINS; b += 1024)
        if (hist[b]) atomicAdd(&plan->total[b], hist[b]);
    __syncthreads();
    if (first == lane && threadIdx.x < 64) wins[wbase + slot] = row * 64 + lane;
}

// ---- bucket chains.  A chain starts from the point at infinity, so its first addition returns
// the generator itself (bls12-381.cu:1432), as the reference's bucket does.  Two ways to run
// one: in row form a wave takes one chain, 1.1 us per addition and 0.9 us of a SIMD's time; a
// lane takes one chain (fp_lane28.hpp), 15 us per addition here (two waves on a SIMD, operands
// from the table) and 0.2 us of a SIMD's time.  With
// small signed scalars the row's shared list of negative entries is a chain of n/2 additions,
// with full-size scalars every chain has about n/16: so the chains are sorted by length, the
// ones from a length on go to waves and the others, 64 of about one length together, to lanes.
// 512 rows of 2048 int16: 17.7 ms with long chains on lane quads and short ones on lanes of
// 32-bit limbs, 2.5 so; 512 rows of 1000 field elements 15.3 and 6.0 (0.2 us x 31M additions
// over 1024 SIMDs).

// the generators in row form with Z^2 and Z^3 behind them (they enter every addition), one
// wave per point; the plan's counters start at zero
__global__ __launch_bounds__(256) void k_pip_gens(const uint32_t* __restrict__ gens, uint32_t n,
                                                  uint32_t* __restrict__ tab, PipPlan* __restrict__ plan) {
    const uint32_t i = blockIdx.x * 4 + threadIdx.x / 64;
    if (blockIdx.x == 0)
        for (uint32_t k = threadIdx.x; k < sizeof(PipPlan) / 4; k += 256) ((uint32_t*)plan)[k] = 0;
    if (i >= n) return;
    const fpr_k c = fpr_consts();
    const g1r_t g = g1r_load(gens + 36 * (size_t)i, c);
    uint32_t* o = tab + G1Z_WORDS * (size_t)i;
    g1r_put(o, g, c);
    const uint32_t zz = fpr_mul(g.z, g.z, c), zzz = fpr_mul(zz, g.z, c);
    if (c.row < 2) o[G1R_WORDS + 16 * c.row + c.lane] = c.row ? zzz : zz;
}
// Where each length class starts in the sorted list (longest first) and from which class on
// chains go to waves.  The cost of a choice, in us: the busiest of (the SIMDs' total work, the
// longest lane chain, the longest wave chain), with the total again at a tenth to break ties.
__global__ __launch_bounds__(512) void k_pip_plan(PipPlan* __restrict__ plan) {
    static_assert(PIP_BINS <= 512, "one thread per class");
    __shared__ uint32_t cnt[512], lmax[512];
    __shared__ float work[512], best[512];
    __shared__ uint32_t arg[512];
    const uint32_t b = threadIdx.x;
    const uint32_t t = b < PIP_BINS ? plan->total[b] : 0;
    const float len = (float)pip_bin_len(b);
    cnt[b] = t;
    work[b] = t * len;
    lmax[b] = t ? pip_bin_len(b) : 0;
    __syncthreads();
    // inclusive sums over the classes from b on; the longest length up to b
    for (uint32_t o = 1; o < 512; o <<= 1) {
        const uint32_t ca = b + o < 512 ? cnt[b + o] : 0, la = b >= o ? lmax[b - o] : 0;
        const float wa = b + o < 512 ? work[b + o] : 0;
        __syncthreads();
        cnt[b] += ca;
        work[b] += wa;
        lmax[b] = lmax[b] > la ? lmax[b] : la;
        __syncthreads();
    }
    // the choice b: classes from b on to waves
    const float rows = work[b], lanes = work[0] - rows, sum = (rows * 0.9f + lanes * 0.2f) / 1024;
    const float lane_t = b ? 15.0f * lmax[b - 1] : 0, wave_t = rows > 0 ? 1.1f * lmax[511] : 0;
    best[b] = fmaxf(sum, fmaxf(lane_t, wave_t)) + 0.1f * sum;
    arg[b] = b;
    __syncthreads();
    for (uint32_t o = 256; o > 0; o >>= 1) {
        if (b < o && best[b + o] < best[b]) best[b] = best[b + o], arg[b] = arg[b + o];
        __syncthreads();
    }
    if (b < PIP_BINS) plan->cursor[b] = cnt[b] - t;
    if (b == 0) {
        plan->items = cnt[0];
        plan->waves = cnt[arg[0]];
    }
}
// the representative chains (row * 1024 + window * 16 + digit) into their classes' places
__global__ __launch_bounds__(1024) void k_pip_scatter(const uint32_t* __restrict__ offs,
                                                      const uint16_t* __restrict__ alias,
                                                      PipPlan* __restrict__ plan, uint32_t* __restrict__ items) {
    __shared__ uint32_t hist[PIP_BINS], base[PIP_BINS];
    const uint32_t row = blockIdx.x, c = threadIdx.x, d = c & 15;
    for (uint32_t b = c; b < PIP_BINS; b += 1024) hist[b] = 0;
    __syncthreads();
    const uint32_t* o = offs + (size_t)row * 1024 + (c & ~15u);
    const uint32_t len = d ? (d == 15 ? o[0] : o[d + 1]) - o[d] : 0;
    const bool mine = len && alias[(size_t)row * 1024 + c] == c;
    const uint32_t bin = pip_bin(len);
    uint32_t at = 0;
    if (mine) at = atomicAdd(&hist[bin], 1u);
    __syncthreads();
    for (uint32_t b = c; b < PIP_BINS; b += 1024)
        if (hist[b]) base[b] = atomicAdd(&plan->cursor[b], hist[b]);
    __syncthreads();
    if (mine) items[base[bin] + at] = row * 1024 + c;
}
// the lists of a chain
__device__ __forceinline__ const uint16_t* pip_list(uint32_t item, const uint16_t* lists, const uint32_t* offs,
                                                    uint32_t n, uint32_t& len) {
    const uint32_t d = item & 15;
    const uint32_t* o = offs + (item & ~15u);
    const uint32_t beg = o[d];
    len = (d == 15 ? o[0] : o[d + 1]) - beg;
    return lists + (size_t)(item >> 4) * n + beg;
}
// Persistent waves, two per SIMD: odd blocks take wave chains while there are any and then lane
// groups, even blocks the other way round, so both kinds start with their longest at once.
// A wave ends when both queues are empty.
__global__ __launch_bounds__(64, 2) void k_pip_bucket(const uint32_t* __restrict__ tab,
                                                      const uint16_t* __restrict__ lists,
                                                      const uint32_t* __restrict__ offs,
                                                      const uint32_t* __restrict__ items, uint32_t n,
                                                      PipPlan* __restrict__ plan, uint32_t* __restrict__ buckets) {
    const uint32_t nrow = plan->waves, nall = plan->items, ngrp = (nall - nrow + 63) / 64;
    const fpr_k c = fpr_consts();
    for (uint32_t turn = 0; turn < 2; turn++) {
        const bool rows = (blockIdx.x & 1) != turn;
        const uint32_t tasks = rows ? nrow : ngrp;
        for (;;) {
            uint32_t task = 0;
            if (threadIdx.x == 0) task = atomicAdd(&plan->taken[rows ? 0 : 1], 1u);
            task = __builtin_amdgcn_readfirstlane(task);
            if (task >= tasks) break;
            if (rows) {
                const uint32_t item = items[task];
                uint32_t len;
                const uint16_t* L = pip_list(item, lists, offs, n, len);
                const uint32_t last = len - 1;
                auto fetch = [&](uint32_t i) { return g1z_fetch(tab + G1Z_WORDS * (size_t)i, c); };
                auto index = [&](uint32_t k) { return (uint32_t)L[k < last ? k : last]; };
                g1r_t acc = g1z_take(fetch(L[0]), c).p;
                // the next generator is loaded one addition ahead, its index two (past the end:
                // the last one again)
                g1z_raw nxt = fetch(index(1));
                uint32_t idx = index(2);
                for (uint32_t k = 1; k < len; k++) {
                    const g1z_raw g = nxt;
                    nxt = fetch(idx);
                    idx = index(k + 2);
                    acc = g1z_add(acc, g1z_take(g, c), c);
                }
                g1r_put(buckets + (size_t)item * G1R_WORDS, acc, c);
            } else {
                const uint32_t at = nrow + task * 64 + threadIdx.x;
                const bool mine = at < nall;
                const uint32_t item = items[mine ? at : nall - 1];
                uint32_t len;
                const uint16_t* L = pip_list(item, lists, offs, n, len);
                bool inf;
                g28_t acc = g28_load(tab + G1Z_WORDS * (size_t)L[0], inf);
                uint32_t idx = len > 1 ? L[1] : 0;
                for (uint32_t k = 1; k < len; k++) {
                    const uint32_t* p = tab + G1Z_WORDS * (size_t)idx;
                    if (k + 1 < len) idx = L[k + 1];
                    bool binf;
                    const g28_t b = g28_load(p, binf);
                    if (!binf) g28_add(acc, inf, b, f28_load(p + G1R_WORDS), f28_load(p + G1R_WORDS + 16));
                }
                if (mine) g28_store(buckets + (size_t)item * G1R_WORDS, acc, inf);
            }
        }
    }
}

// sum_b b * bucket[b] by the running sum acc += bucket[b]; run += acc, b = 15..1
// (commitment.cu:73-77), a chain of up to 30 additions, for the windows that stand in for
// themselves: on one wave each in row form (40 us a chain) or, where there are more than the
// SIMDs take that way in a lane chain's 0.42 ms, on one lane each
#define PIP_WIN_LANES 13000u
__global__ __launch_bounds__(64) void k_pip_window_rows(const uint32_t* __restrict__ buckets,
                                                        const uint32_t* __restrict__ offs,
                                                        const uint16_t* __restrict__ alias,
                                                        const PipPlan* __restrict__ plan,
                                                        const uint32_t* __restrict__ wins,
                                                        uint32_t* __restrict__ partials) {
    const uint32_t nw = plan->nwin;
    if (nw > PIP_WIN_LANES) return;
    const fpr_k c = fpr_consts();
    for (uint32_t k = blockIdx.x; k < nw; k += gridDim.x) {
        const size_t t = wins[k], row0 = t / 64 * 64;
        const uint32_t* o = offs + t * 16;
        g1r_t acc = g1r_zero(c), run = acc;
        for (int b = 15; b >= 1; b--) {
            const uint32_t e = b == 15 ? o[0] : o[b + 1];
            if (e != o[b]) acc = g1r_add(acc, g1r_get(buckets + (row0 * 16 + alias[t * 16 + b]) * G1R_WORDS, c), c);
            run = g1r_add(run, acc, c);
        }
        g1r_put(partials + t * G1R_WORDS, run, c);
    }
}
__global__ __launch_bounds__(64) void k_pip_window_lanes(const uint32_t* __restrict__ buckets,
                                                         const uint32_t* __restrict__ offs,
                                                         const uint16_t* __restrict__ alias,
                                                         const PipPlan* __restrict__ plan,
                                                         const uint32_t* __restrict__ wins,
                                                         uint32_t* __restrict__ partials) {
    const uint32_t nw = plan->nwin;
    if (nw <= PIP_WIN_LANES) return;
    for (uint32_t k = blockIdx.x * 64 + threadIdx.x; k < nw; k += gridDim.x * 64) {
        const size_t t = wins[k], row0 = t / 64 * 64;
        const uint32_t* o = offs + t * 16;
        bool ainf = true, rinf = true;
        g28_t acc = g28_zero(), run = acc;
#pragma unroll 1
        for (int step = 29; step >= 0; step--) {  // odd: acc += bucket, even: run += acc
            const int b = step / 2 + 1;
            g28_t x = acc;
            bool xinf = ainf;
            if (step & 1) {
                const uint32_t e = b == 15 ? o[0] : o[b + 1];
                xinf = e == o[b];
                if (!xinf) x = g28_load(buckets + (row0 * 16 + alias[t * 16 + b]) * G1R_WORDS, xinf);
            }
            if (xinf) continue;
            const f28_t zz = f28_sqr(x.z), zzz = f28_mul(zz, x.z);
            g28_t y = step & 1 ? acc : run;
            bool yinf = step & 1 ? ainf : rinf;
            g28_add(y, yinf, x, zz, zzz);
            if (step & 1) acc = y, ainf = yinf;
            else run = y, rinf = yinf;
        }
        g28_store(partials + t * G1R_WORDS, run, rinf);
    }
}

// Horner over the windows, most significant first (commitment.cu:81-89): 252 doublings and 64
// additions in sequence, one wave per row in row form (0.33 ms; 2.5 ms on a lane quad)
__global__ __launch_bounds__(64) void k_pip_combine(const uint32_t* __restrict__ partials,
                                                    const uint16_t* __restrict__ walias,
                                                    uint32_t* __restrict__ out) {
    const uint32_t row = blockIdx.x;
    const fpr_k c = fpr_consts();
    g1r_t acc = g1r_zero(c);
    for (int w = 63; w >= 0; w--) {
        for (int k = 0; k < 4; k++) acc = g1r_dbl(acc, c);
        acc = g1r_add(acc, g1r_get(partials + ((size_t)row * 64 + walias[(size_t)row * 64 + w]) * G1R_WORDS, c), c);
    }
    g1r_store(out + (size_t)row * 36, acc, c);
}

// ---- G1Jacobian_mul (g1-tensor.cu:445-454): double-and-add over the scalar's raw bits, low bit
// first.  The doubling chain a, 2a, 4a, ... does not depend on the scalar, so a product is a
// doubling chain and a chain of the ones whose bit is set; the operations and their order are
// those of the one loop, so the representative is the same.  A base's chain is kept as a table
// (2^i a with its Z^2 and Z^3 for i < 255, 80 KiB) where more than one scalar multiplies it.
// The tables of a launch's bases lie entry by entry (entry i of every base, then entry i + 1):
// its waves run through the bits side by side, so they write and read neighbouring entries.
#define G1_BITS 255u  // scalars are below 2^255
__device__ __forceinline__ uint32_t limb8(const uint32_t s[8], uint32_t l) {
    return l == 0 ? s[0] : l == 1 ? s[1] : l == 2 ? s[2] : l == 3 ? s[3]
         : l == 4 ? s[4] : l == 5 ? s[5] : l == 6 ? s[6] : s[7];
}
__device__ __forceinline__ int top_bit(const uint32_t s[8]) {
    int top = -1;
    for (int l = 7; l >= 0 && top < 0; l--)
        if (s[l]) top = 32 * l + 31 - __builtin_clz(s[l]);
    return top;
}
// the set bits of a scalar in ascending order, -1 after the last
struct SetBits {
    uint32_t w, l;
    __device__ __forceinline__ explicit SetBits(const uint32_t s[8]) : w(s[0]), l(0) {}
    __device__ __forceinline__ int next(const uint32_t s[8]) {
        while (!w && l < 7) w = limb8(s, ++l);
        if (!w) return -1;
        const int b = __builtin_ctz(w);
        w &= w - 1;
        return (int)(32 * l) + b;
    }
};
// a base's table: entry i at p + i * step
struct G1Tab {
    uint32_t* p;
    size_t step;
    __device__ __forceinline__ uint32_t* at(uint32_t i) const { return p + i * step; }
};
// that of the k-th of n bases
__device__ __forceinline__ G1Tab g1_tab(uint32_t* tab, uint32_t k, uint32_t n) {
    return {tab + (size_t)k * G1Z_WORDS, (size_t)n * G1Z_WORDS};
}
// one product from its base's table, one wave in row form: 1.1 us per set bit
__device__ __forceinline__ g1r_t g1r_tab_mul(const G1Tab& tab, const uint32_t s[8], const fpr_k& c) {
    g1r_t acc = g1r_zero(c);
    SetBits bits(s);
    // two points are loaded ahead of the addition, each into its own registers (moving one to
    // the other's would wait for it); past the last bit: entry 0
    int b0 = bits.next(s), b1 = b0 < 0 ? -1 : bits.next(s);
    auto fetch = [&](int b) { return g1z_fetch(tab.at(b < 0 ? 0 : b), c); };
    g1z_raw p0 = fetch(b0), p1 = fetch(b1);
    for (;;) {
        if (b0 < 0) return acc;
        g1z_t p = g1z_take(p0, c);
        b0 = b1 < 0 ? -1 : bits.next(s);
        p0 = fetch(b0);
        acc = g1z_add(acc, p, c);
        if (b1 < 0) return acc;
        p = g1z_take(p1, c);
        b1 = b0 < 0 ? -1 : bits.next(s);
        p1 = fetch(b1);
        acc = g1z_add(acc, p, c);
    }
}
// the same on a lane quad
__device__ __forceinline__ g28_t g28q_tab_mul(const G1Tab& tab, const uint32_t s[8], int q, bool& inf) {
    g28_t acc = g28_zero();
    inf = true;
    SetBits bits(s);
    int b = bits.next(s);
    // the next point is loaded during the addition (past the last bit: entry 0), as soon as the
    // addition has read its own
    g28_raw p;
    f28_t zz, zzz;
    auto fetch = [&] {
        const uint32_t* e = tab.at(b < 0 ? 0 : b);
        p = g28_fetch(e);
        zz = f28_load(e + G1R_WORDS);
        zzz = f28_load(e + G1R_WORDS + 16);
    };
    fetch();
    while (b >= 0) {
        bool pinf;
        const g28_t x = g28_take(p, pinf);
        const f28_t xz = zz, xzz = zzz;
        b = bits.next(s);
        if (pinf) fetch();
        else g28q_add(acc, inf, x, xz, xzz, q, fetch);
    }
    return acc;
}
// a base's table on a lane quad: lane q < 3 stores coordinate q, lane 3 Z^2 and Z^3; signed limbs
// as they are (the tables of quads are read by quads); entries below `bits`
__device__ __forceinline__ void g28q_table(g28_t a, bool inf, const G1Tab& tab, int q, uint32_t bits) {
    for (uint32_t i = 0; i < bits; i++) {
        f28_t zz = {}, zzz = {};
        g28_t d = a;
        bool dinf = inf;
        if (!inf) {
            dinf = f28_zero(a.y);  // Z3 = 2 Y Z
            d = g28q_dbl(a, q, zz, zzz);
        }
        uint32_t* e = tab.at(i);
        f28_put(e + 16 * q, f28_sel4(q, a.x, a.y, a.z, zz), q == 0 && inf ? 1u : 0u);
        if (q == 3) f28_put(e + 64, zzz, 0);
        a = d;
        inf = dinf;
    }
}
// One product on two waves in row form: wave 0 of the pair runs the doubling chain and hands
// each 2^i a to wave 1 through LDS, G1P_B doublings per block barrier; wave 1 adds the ones
// whose bit is set one barrier later.  The chain is latency-bound (0.77 us per doubling, 1.05
// per addition on an idle SIMD): 255 doublings and 127 additions side by side take 0.23 ms.
// At 16 doublings per barrier the additions of a chunk (8.4 +- 2.1 us) rarely outlast its
// doublings (12.3 us).  Every wave of the block calls it (dbl: its part), with one scalar per
// pair; the product is in the adding wave, which does not read `a`.  tab: where the base's
// table is wanted too (all 255 doublings then), else null and the doublings after the highest
// set bit are skipped.
#define G1P_B 16
typedef uint32_t g1_pipe_buf[2][G1P_B][G1Z_WORDS];
__device__ __forceinline__ g1r_t g1r_mul_pipe(g1r_t a, const uint32_t s[8], bool dbl, g1_pipe_buf& buf,
                                              const G1Tab& tab, const fpr_k& c) {
    static_assert(32 % G1P_B == 0, "a chunk's bits lie in one scalar limb");
    const int top = top_bit(s), last = tab.p ? (int)G1_BITS - 1 : top;
    g1r_t acc = g1r_zero(c);
    constexpr int NC = 256 / G1P_B;
    for (int k = 0; k <= NC; k++) {
        if (dbl) {
            for (int j = 0; j < G1P_B; j++) {
                const int i = k * G1P_B + j;
                if (i > last) break;
                g1z_t z{a, 0, 0};
                a = g1z_dbl(z, c);
                const uint32_t v = g1z_word(z, c);
                g1z_put(buf[k & 1][j], v, z, c);
                if (tab.p) g1z_put(tab.at(i), v, z, c);
            }
        } else if (k > 0) {
            const uint32_t w = limb8(s, (uint32_t)((k - 1) * G1P_B) >> 5);
            for (int j = 0; j < G1P_B; j++) {
                const int i = (k - 1) * G1P_B + j;
                if (i <= top && ((w >> (i & 31)) & 1u))
                    acc = g1z_add(acc, g1z_take(g1z_fetch(buf[(k - 1) & 1][j], c), c), c);
            }
        }
        __syncthreads();
    }
    return acc;
}

// elementwise with a broadcast base (G1_jacobian_elementwise_mul_broadcast,
// g1-tensor.cu:463-468): out[i] = base[i % nb] * s[i].
// The tables of bases [b0, b0 + nt): one wave each in row form (0.2 ms a chain) or, from
// G1_QUADS on, where the SIMDs are full that way, one quad each (1.0 ms; a third of the work).
// They end at the highest bit of the launch's scalars, which a reduction ahead of them leaves
// per block in tops: with 16-bit scalars whole tables took 1.1 ms at 5000 bases and 6.0 at 65536
// (0.18 and 0.72 so).
#define G1_QUADS 5000u
// tops[block] = bits of the block's longest scalar
__global__ __launch_bounds__(256) void k_g1_top(const uint32_t* __restrict__ lo, const uint32_t* __restrict__ hi,
                                                uint32_t n, uint32_t* __restrict__ tops) {
    __shared__ int red[4];
    int top = -1;
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        const uint4 s0 = ((const uint4*)lo)[i], s1 = ((const uint4*)hi)[i];
        const uint32_t sc[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
        const int t = top_bit(sc);
        top = t > top ? t : top;
    }
    for (int o = 32; o >= 1; o >>= 1) {
        const int t = __shfl_xor(top, o);
        top = t > top ? t : top;
    }
    if ((threadIdx.x & 63) == 0) red[threadIdx.x / 64] = top;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 0; w < 4; w++) top = red[w] > top ? red[w] : top;
        tops[blockIdx.x] = (uint32_t)(top + 1);
    }
}
// the longest of them all, at least 1 (entry 0 is read past a scalar's last bit); the whole wave
__device__ __forceinline__ uint32_t g1_bits(const uint32_t* tops, uint32_t ntops) {
    uint32_t b = 1;
    for (uint32_t i = threadIdx.x & 63; i < ntops; i += 64) b = tops[i] > b ? tops[i] : b;
    for (int o = 32; o >= 1; o >>= 1) {
        const uint32_t t = (uint32_t)__shfl_xor((int)b, o);
        b = t > b ? t : b;
    }
    return __builtin_amdgcn_readfirstlane(b);
}
__global__ __launch_bounds__(64) void k_g1_tables(const uint32_t* __restrict__ base, uint32_t b0,
                                                  const uint32_t* __restrict__ tops, uint32_t ntops,
                                                  uint32_t* __restrict__ tab) {
    const uint32_t i = blockIdx.x, bits = g1_bits(tops, ntops);
    const fpr_k c = fpr_consts();
    g1r_t a = g1r_load(base + 36 * (size_t)(b0 + i), c);
    const G1Tab t = g1_tab(tab, i, gridDim.x);
    for (uint32_t k = 0; k < bits; k++) {
        g1z_t z{a, 0, 0};
        a = g1z_dbl(z, c);
        g1z_put(t.at(k), g1z_word(z, c), z, c);
    }
}
// out[i] = base[i % nb] * s[i], two waves per product, no table
__global__ __launch_bounds__(128) void k_g1_mul(const uint32_t* __restrict__ base, uint32_t nb,
                                                const uint32_t* __restrict__ lo, const uint32_t* __restrict__ hi,
                                                uint32_t* __restrict__ out) {
    __shared__ g1_pipe_buf buf;
    const uint32_t i = blockIdx.x;
    const fpr_k c = fpr_consts();
    const bool dbl = __builtin_amdgcn_readfirstlane(threadIdx.x / 64) == 0;
    const uint4 s0 = ((const uint4*)lo)[i], s1 = ((const uint4*)hi)[i];
    const uint32_t sc[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
    g1r_t p = g1r_zero(c);
    if (dbl) p = g1r_load(base + 36 * (size_t)(i % nb), c);
    const g1r_t m = g1r_mul_pipe(p, sc, dbl, buf, G1Tab{}, c);
    if (!dbl) g1r_store(out + 36 * (size_t)i, m, c);
}
__global__ __launch_bounds__(64) void k_g1_tables4(const uint32_t* __restrict__ base, uint32_t b0, uint32_t nt,
                                                   const uint32_t* __restrict__ tops, uint32_t ntops,
                                                   uint32_t* __restrict__ tab) {
    const uint32_t i = blockIdx.x * 16 + threadIdx.x / 4, bits = g1_bits(tops, ntops);
    if (i >= nt) return;
    bool inf;
    const g28_t a = g28q_load(base + 36 * (size_t)(b0 + i), threadIdx.x & 3, inf);
    g28q_table(a, inf, g1_tab(tab, i, nt), threadIdx.x & 3, bits);
}
// products i0 + k (k < count) of the bases at hand (base (i0 + k) % nb - b0): one wave each
__global__ __launch_bounds__(64) void k_g1_tab_mul(uint32_t* __restrict__ tab, uint32_t nt, uint32_t nb, uint32_t b0,
                                                   const uint32_t* __restrict__ lo, const uint32_t* __restrict__ hi,
                                                   uint32_t i0, uint32_t* __restrict__ out) {
    const uint32_t i = i0 + blockIdx.x;
    const fpr_k c = fpr_consts();
    const uint4 s0 = ((const uint4*)lo)[i], s1 = ((const uint4*)hi)[i];
    const uint32_t sc[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
    g1r_store(out + 36 * (size_t)i, g1r_tab_mul(g1_tab(tab, i % nb - b0, nt), sc, c), c);
}
// one quad each
__global__ __launch_bounds__(64, 2) void k_g1_tab_mul4(uint32_t* __restrict__ tab, uint32_t nt, uint32_t nb, uint32_t b0,
                                                    const uint32_t* __restrict__ lo, const uint32_t* __restrict__ hi,
                                                    uint32_t i0, uint32_t count, uint32_t* __restrict__ out) {
    const uint32_t k = blockIdx.x * 16 + threadIdx.x / 4, i = i0 + k;
    if (k >= count) return;
    const uint4 s0 = ((const uint4*)lo)[i], s1 = ((const uint4*)hi)[i];
    const uint32_t sc[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
    const int q = threadIdx.x & 3;
    bool inf;
    g28q_store(out + 36 * (size_t)i, g28q_tab_mul(g1_tab(tab, i % nb - b0, nt), sc, q, inf), q);
}
// out[i] = b[i] + a[i] * s: one scalar for every row, the sum with b[i] as first operand
// (hb_addmul with mul_first = false, zkob_fastg1.cuh:56-88: k_g1_mul then k_g1_addsub).  Two
// waves per row in row form, its latency while the SIMDs are not full, or from G1_ADDMUL_QUADS
// rows on a lane quad per row: every quad adds at the same bits, so the chain needs no table.
// Full scalar, waves and quads: 1.20 and 1.59 ms at 4096 rows, 1.48 and 1.70 at 5000, 2.29 and
// 1.56 at 8192, 16.5 and 5.6 at 65536; a 14-bit scalar 98 and 106 us at 4096, 178 and 106 at 8192
__global__ __launch_bounds__(128) void k_g1_addmul(const uint32_t* __restrict__ a, G1Scalar sc,
                                                   const uint32_t* __restrict__ b, uint32_t* __restrict__ out) {
    __shared__ g1_pipe_buf buf;
    const uint32_t i = blockIdx.x;
    const fpr_k c = fpr_consts();
    const bool dbl = __builtin_amdgcn_readfirstlane(threadIdx.x / 64) == 0;
    g1r_t p = g1r_zero(c);
    if (dbl) p = g1r_load(a + 36 * (size_t)i, c);
    const g1r_t m = g1r_mul_pipe(p, sc.v, dbl, buf, G1Tab{}, c);
    if (!dbl) g1r_store(out + 36 * (size_t)i, g1r_add(g1r_load(b + 36 * (size_t)i, c), m, c), c);
}
#define G1_ADDMUL_QUADS 6000u
__global__ __launch_bounds__(64, 2) void k_g1_addmul4(const uint32_t* __restrict__ a, G1Scalar sc,
                                                      const uint32_t* __restrict__ b, uint32_t n,
                                                      uint32_t* __restrict__ out) {
    const uint32_t i = blockIdx.x * 16 + threadIdx.x / 4;
    if (i >= n) return;
    const int q = threadIdx.x & 3, top = top_bit(sc.v);
    bool inf, minf = true;
    g28_t p = g28q_load(a + 36 * (size_t)i, q, inf), m = g28_zero();
    f28_t zz, zzz;
#pragma unroll 1
    for (int k = 0; k <= top && !inf; k++) {
        const bool dinf = f28_zero(p.y);  // Z3 = 2 Y Z
        const g28_t d = g28q_dbl(p, q, zz, zzz);
        if (limb8(sc.v, (uint32_t)k >> 5) >> (k & 31) & 1u)
            g28q_add(m, minf, p, f28_quad<3>(zz), f28_quad<3>(zzz), q, [] {});
        p = d;
        inf = dinf;
    }
    g28_t r = g28q_load(b + 36 * (size_t)i, q, inf);
    if (!minf) {
        zz = f28_sqr(m.z);
        g28q_add(r, inf, m, zz, f28_mul(zz, m.z), q, [] {});
    }
    g28q_store(out + 36 * (size_t)i, r, q);
}

// ---- inner-product argument rounds (ipa_prove, vrf_common.cuh:302-336) ----
// a, b: plain Fr, 8 words per entry; g, Q, P: points in row form (G1R_WORDS each).  Round of
// size 2h:
//   ip = (<a_lo, b_hi>, <a_hi, b_lo>)
//   P[j] = g_hi[j] a_lo[j], P[h + j] = g_lo[j] a_hi[j], P[2h] = Q ip_L, P[2h+1] = Q ip_R
//   pairwise trees over P[0, h) and P[h, 2h)                  (dev_msm's order)
//   L = P[0] + P[2h], R = P[h] + P[2h+1]
//   fold: a' = x a_lo + x^-1 a_hi, b' = x^-1 b_lo + x b_hi, g' = x^-1 g_lo + x g_hi
// A round of few points is the latency of its two scalar-multiply chains (scale and fold): one
// product per block, doublings and additions on a wave each.  One of many points is the
// instruction rate: the points' doubling tables once on lane quads, then the additions of both
// products of a point from them.

// the working copies of g and Q in row form, one wave per point (point n of a job is Q)
__global__ __launch_bounds__(256) void k_ipa_points(IpaBatchDev B) {
    const IpaJobDev& J = B.j[blockIdx.y];
    const uint32_t n = 2 * J.h, i = blockIdx.x * 4 + threadIdx.x / 64;
    if (i > n) return;
    const fpr_k c = fpr_consts();
    g1r_put(J.g0 + G1R_WORDS * (size_t)i, g1r_load(i < n ? J.g_in + 36 * (size_t)i : J.Q, c), c);
}
// Scale and fold launches hold exactly the blocks of the jobs still folding (job j's from
// scale0 / fold0 on), and ask for so much LDS that a CU takes no more than its share of them:
// the dispatcher otherwise stacks blocks on some CUs while others idle, and a chain sharing
// its SIMD runs at the SIMD's rate, not at its own latency.
__device__ __forceinline__ uint32_t ipa_job(const IpaBatchDev& B, uint32_t nj, uint32_t blk, bool scale) {
    uint32_t job = 0;
    for (uint32_t j = 1; j < nj; j++)
        if (B.j[j].h && blk >= (scale ? B.j[j].scale0 : B.j[j].fold0)) job = j;
    return job;
}
// dynamic LDS per block beside `used` static bytes; `least` blocks give every SIMD of a CU one wave
static uint32_t lds_share(uint32_t blocks, uint32_t least, uint32_t used) {
    const uint32_t per_cu = blocks <= 256 * least ? least : (blocks + 255) / 256;
    if (per_cu > 8) return 0;
    const uint32_t want = 160 * 1024 / (per_cu + 1) + 512;  // per_cu + 1 blocks do not fit
    return want > used ? want - used : 0;
}
// <a_lo, b_hi> (side 0) or <a_hi, b_lo> (side 1) by the block's threads, plain, to `out` (LDS)
__device__ __forceinline__ void ipa_inner(const IpaJobDev& J, uint32_t side, const fr_t& r2, fr_t* red,
                                          uint32_t* out) {
    const uint32_t h = J.h, nt = blockDim.x;
    fr_t s = fr_zero();
    for (uint32_t i = threadIdx.x; i < h; i += nt)
        s = fr_add(s, mont_mul(ld_aos(J.a, side ? h + i : i), ld_aos(J.b, side ? i : h + i)));
    red[threadIdx.x] = s;
    __syncthreads();
    for (uint32_t o = nt / 2; o > 0; o >>= 1) {
        if (threadIdx.x < o) red[threadIdx.x] = fr_add(red[threadIdx.x], red[threadIdx.x + o]);
        __syncthreads();
    }
    // a sum of a b 2^-256; times R^2 2^-256 gives the plain sum
    if (threadIdx.x == 0) st_aos(out, 0, mont_mul(red[0], r2));
    __syncthreads();
}
// L and R terms (vrf_common.cuh:316-319): P[j] = g[h + j] a[j], P[h + j] = g[j] a[h + j],
// P[2h], P[2h + 1] = Q <a_lo, b_hi>, Q <a_hi, b_lo>.  The fold multiplies the same generators,
// so their tables are kept for it: point id 2 i + hi of a job is g[i + hi h], its table the
// (pt0 + id - slice0)-th.
__device__ __forceinline__ G1Tab ipa_table(const IpaBatchDev& B, const IpaJobDev& J, uint32_t id) {
    return g1_tab(B.D, J.pt0 + id - B.slice0, B.slice);
}
// one product by waves 0 and 1 of the block (more only take its barriers): blk 0, 1 the Q
// products with their inner products (first, since they are the longest), then P[blk - 2] with its generator's table
__device__ __forceinline__ void ipa_product(const IpaBatchDev& B, const IpaJobDev& J, uint32_t blk, const fr_t& r2,
                                            g1_pipe_buf& buf, fr_t* red, uint32_t* ip) {
    const uint32_t h = J.h;
    const fpr_k c = fpr_consts();
    const uint32_t j = blk < 2 ? 2 * h + blk : blk - 2;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const bool dbl = wave == 0;
    if (blk < 2) ipa_inner(J, blk, r2, red, ip);
    const uint32_t* sp = blk < 2 ? ip : J.a + 8 * (size_t)j;
    uint32_t sc[8];
#pragma unroll
    for (int k = 0; k < 8; k++) sc[k] = wave < 2 ? __builtin_amdgcn_readfirstlane(sp[k]) : 0;
    const uint32_t* bp = j < h ? J.g + G1R_WORDS * (size_t)(h + j) : j < 2 * h ? J.g + G1R_WORDS * (size_t)(j - h) : J.Qr;
    g1r_t base = g1r_zero(c);
    if (dbl) base = g1r_get(bp, c);
    const G1Tab tab = blk < 2 ? G1Tab{} : ipa_table(B, J, j < h ? 2 * j + 1 : 2 * (j - h));
    const g1r_t r = g1r_mul_pipe(base, sc, dbl, buf, tab, c);
    if (wave == 1) g1r_put(J.P + G1R_WORDS * (size_t)j, r, c);
}
// few points: one product per block
__global__ __launch_bounds__(128) void k_ipa_scale(IpaBatchDev B, uint32_t nj, fr_t r2) {
    __shared__ g1_pipe_buf buf;
    __shared__ fr_t red[128];
    __shared__ uint32_t ip[8];
    const IpaJobDev& J = B.j[ipa_job(B, nj, blockIdx.x, true)];
    const uint32_t blk = blockIdx.x - J.scale0;
    if (blk >= 2 * J.h + 2) return;  // whole block
    ipa_product(B, J, blk, r2, buf, red, ip);
}
// many points (G1_QUADS): the Q products on two waves each (blocks below 2 nj, where asked),
// the tables of points [slice0, slice0 + count) on quads; then every product on a quad
__device__ __forceinline__ uint32_t ipa_point(const IpaBatchDev& B, uint32_t nj, uint32_t pt) {
    uint32_t job = 0;
    for (uint32_t j = 1; j < nj; j++)
        if (B.j[j].h && pt >= B.j[j].pt0) job = j;
    return job;
}
__global__ __launch_bounds__(256) void k_ipa_tables4(IpaBatchDev B, uint32_t nj, uint32_t nq, uint32_t count, fr_t r2) {
    __shared__ g1_pipe_buf buf;
    __shared__ fr_t red[256];
    __shared__ uint32_t ip[8];
    if (blockIdx.x < nq) {
        const IpaJobDev& J = B.j[blockIdx.x / 2];
        if (J.h) ipa_product(B, J, blockIdx.x & 1, r2, buf, red, ip);
        return;
    }
    const uint32_t k = (blockIdx.x - nq) * 64 + threadIdx.x / 4;
    if (k >= count) return;
    const IpaJobDev& J = B.j[ipa_point(B, nj, B.slice0 + k)];
    const uint32_t id = B.slice0 + k - J.pt0;
    bool inf;
    const g28_t a = g28_load(J.g + G1R_WORDS * (size_t)(id / 2 + (id & 1) * J.h), inf);
    g28q_table(a, inf, ipa_table(B, J, id), threadIdx.x & 3, G1_BITS);
}
__global__ __launch_bounds__(64, 2) void k_ipa_scale4(IpaBatchDev B, uint32_t nj, uint32_t count) {
    const uint32_t k = blockIdx.x * 16 + threadIdx.x / 4;
    if (k >= count) return;
    const IpaJobDev& J = B.j[ipa_point(B, nj, B.slice0 + k)];
    const uint32_t id = B.slice0 + k - J.pt0, j = id / 2 + (id & 1 ? 0 : J.h);
    uint32_t sc[8];
#pragma unroll
    for (int l = 0; l < 8; l++) sc[l] = J.a[8 * (size_t)j + l];
    bool inf;
    const g28_t r = g28q_tab_mul(ipa_table(B, J, id), sc, threadIdx.x & 3, inf);
    if ((threadIdx.x & 3) == 0) g28_store(J.P + G1R_WORDS * (size_t)j, r, inf);
}
// pairwise trees over P[0, h) and P[h, 2h): of a side's m = h >> shift remaining points a block
// takes the K = min(m, 64) at distance m / K (six levels of the tree: level by level the halves
// are added, as dev_msm does) and leaves their sum in the first; the block that takes the last
// ones adds the side's Q term and writes L or R, canonical, to the host.  Sixteen waves, one
// addition each per level; partial sums stay in LDS.
static_assert(ZKH_ROW_WORDS == G1R_WORDS && ZKH_POINTZ_WORDS == G1Z_WORDS, "point sizes");
__global__ __launch_bounds__(1024) void k_ipa_tree(IpaBatchDev B, uint32_t shift) {
    const IpaJobDev& J = B.j[blockIdx.y];
    const uint32_t h = J.h, side = blockIdx.z, m = h >> shift;
    if (!m || (shift >= 6 && (h >> (shift - 6)) <= 64)) return;  // no such job, or done before
    const uint32_t K = m < 64 ? m : 64, dist = m / K;
    if (blockIdx.x >= dist) return;
    __shared__ uint32_t sum[32][G1R_WORDS];
    const fpr_k c = fpr_consts();
    const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    uint32_t* P = J.P + G1R_WORDS * (size_t)(side * h + blockIdx.x);
    auto at = [&](uint32_t i) { return g1r_get(P + G1R_WORDS * (size_t)(i * dist), c); };
    if (K == 1) {
        if (w == 0) g1r_put(sum[0], at(0), c);
    } else {
        for (uint32_t i = w; i < K / 2; i += 16) g1r_put(sum[i], g1r_add(at(i), at(i + K / 2), c), c);
    }
    __syncthreads();
    for (uint32_t half = K / 4; half >= 1; half >>= 1) {
        if (w < half) g1r_put(sum[w], g1r_add(g1r_get(sum[w], c), g1r_get(sum[w + half], c), c), c);
        __syncthreads();
    }
    if (w) return;
    const g1r_t r = g1r_get(sum[0], c);
    if (dist > 1) g1r_put(P, r, c);
    else g1r_store(J.LR + 36 * side, g1r_add(r, g1r_get(J.P + G1R_WORDS * (size_t)(2 * h + side), c), c), c);
}
// a' and b' of entry i, on lane 0 (a) and 1 (b) of a pair
__device__ __forceinline__ void ipa_fold_ab(const IpaJobDev& J, uint32_t i, uint32_t sel) {
    const uint32_t h = J.h;
    fr_t xm, xim;
#pragma unroll
    for (int k = 0; k < 8; k++) xm.v[k] = J.xm[k], xim.v[k] = J.xim[k];
    const uint32_t* src = sel ? J.b : J.a;
    st_aos(sel ? J.b2 : J.a2, i,
           fr_add(mont_mul(sel ? xim : xm, ld_aos(src, i)), mont_mul(sel ? xm : xim, ld_aos(src, i + h))));
}
// one folded generator per block, from the tables: wave 0 computes x^-1 g_lo[i], wave 1
// x g_hi[i] (k_g1_fold2's two products, vrf_common.cuh:71-76), then wave 0 adds them in that
// order; two lanes of wave 1 fold a and b first
__global__ __launch_bounds__(128) void k_ipa_fold(IpaBatchDev B, uint32_t nj) {
    const IpaJobDev& J = B.j[ipa_job(B, nj, blockIdx.x, false)];
    const uint32_t i = blockIdx.x - J.fold0;
    if (i >= J.h) return;  // whole block
    __shared__ uint32_t other[G1R_WORDS];
    const fpr_k c = fpr_consts();
    const uint32_t hi = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    uint32_t sc[8];
#pragma unroll
    for (int k = 0; k < 8; k++) sc[k] = hi ? J.x[k] : J.xi[k];
    if (hi && c.lane == 0 && c.row < 2) ipa_fold_ab(J, i, c.row);
    const g1r_t r = g1r_tab_mul(ipa_table(B, J, 2 * i + hi), sc, c);
    if (hi) g1r_put(other, r, c);
    __syncthreads();
    if (!hi) g1r_put(J.g2 + G1R_WORDS * (size_t)i, g1r_add(r, g1r_get(other, c), c), c);
}
// many points: the same on two quads per generator
__global__ __launch_bounds__(64, 2) void k_ipa_fold4(IpaBatchDev B, uint32_t nj, uint32_t count) {
    const uint32_t k = blockIdx.x * 16 + threadIdx.x / 4;
    if (k >= count) return;  // count is even: both quads of a generator or neither
    const IpaJobDev& J = B.j[ipa_point(B, nj, B.slice0 + k)];
    const uint32_t id = B.slice0 + k - J.pt0, i = id / 2, hi = id & 1;
    const int q = threadIdx.x & 3;
    uint32_t sc[8];
#pragma unroll
    for (int l = 0; l < 8; l++) sc[l] = hi ? J.x[l] : J.xi[l];
    if (hi && q < 2) ipa_fold_ab(J, i, q);
    bool inf;
    g28_t r = g28q_tab_mul(ipa_table(B, J, id), sc, q, inf);
    // the upper quad's product to the lower one
    g28_t o;
#pragma unroll
    for (int l = 0; l < 14; l++) {
        o.x.v[l] = __shfl_xor(r.x.v[l], 4);
        o.y.v[l] = __shfl_xor(r.y.v[l], 4);
        o.z.v[l] = __shfl_xor(r.z.v[l], 4);
    }
    const bool oinf = __shfl_xor((int)inf, 4) != 0;
    if (hi) return;
    if (!oinf) {
        const f28_t zz = f28_sqr(o.z);
        g28q_add(r, inf, o, zz, f28_mul(zz, o.z), q, [] {});
    }
    if (q == 0) g28_store(J.g2 + G1R_WORDS * (size_t)i, r, inf);
}
void launch_ipa_points(hipStream_t s, const IpaBatchDev& B, uint32_t nj, uint32_t hmax) {
    hipLaunchKernelGGL(k_ipa_points, dim3((2 * hmax + 1 + 3) / 4, nj), dim3(256), 0, s, B);
}
// blocks of four waves, one per SIMD (of two, the dispatcher put three waves on one SIMD: 2.6 ms
// for 20480 tables)
static void launch_ipa_tables(hipStream_t s, const IpaBatchDev& B, uint32_t nj, uint32_t nq, uint32_t count, fr_t r2) {
    const uint32_t blocks = nq + (count + 63) / 64;
    hipLaunchKernelGGL(k_ipa_tables4, dim3(blocks), dim3(256), lds_share(blocks, 1, sizeof(g1_pipe_buf) + 257 * 32), s, B,
                       nj, nq, count, r2);
}
void launch_ipa_scale(hipStream_t s, IpaBatchDev& B, uint32_t nj, const uint32_t r2[8]) {
    fr_t R2;
    for (int k = 0; k < 8; k++) R2.v[k] = r2[k];
    uint32_t blocks = 0, points = 0;
    for (uint32_t j = 0; j < nj; j++) {
        blocks += B.j[j].h ? 2 * B.j[j].h + 2 : 0;
        points += 2 * B.j[j].h;
    }
    B.slice0 = 0;
    B.slice = points < B.cap ? points : B.cap;
    if (points < G1_QUADS && points <= B.cap) {
        hipLaunchKernelGGL(k_ipa_scale, dim3(blocks), dim3(128), lds_share(blocks, 2, sizeof(g1_pipe_buf) + 129 * 32), s,
                           B, nj, R2);
        return;
    }
    for (; B.slice0 < points; B.slice0 += B.cap) {
        const uint32_t count = points - B.slice0 < B.cap ? points - B.slice0 : B.cap;
        const uint32_t nq = B.slice0 ? 0 : 2 * nj;
        launch_ipa_tables(s, B, nj, nq, count, R2);
        hipLaunchKernelGGL(k_ipa_scale4, dim3((count + 15) / 16), dim3(64), lds_share((count + 15) / 16, 4, 0), s, B, nj, count);
    }
}
void launch_ipa_tree(hipStream_t s, const IpaBatchDev& B, uint32_t nj, uint32_t hmax) {
    for (uint32_t shift = 0; shift == 0 || (hmax >> (shift - 6)) > 64; shift += 6) {
        const uint32_t m = hmax >> shift;
        hipLaunchKernelGGL(k_ipa_tree, dim3(m > 64 ? m / 64 : 1, nj, 2), dim3(1024), 0, s, B, shift);
    }
}
void launch_ipa_fold(hipStream_t s, IpaBatchDev& B, uint32_t nj) {
    uint32_t blocks = 0;
    for (uint32_t j = 0; j < nj; j++) blocks += B.j[j].h;
    const uint32_t points = 2 * blocks;
    B.slice0 = 0;
    B.slice = points < B.cap ? points : B.cap;
    if (points < G1_QUADS && points <= B.cap) {
        hipLaunchKernelGGL(k_ipa_fold, dim3(blocks), dim3(128), lds_share(blocks, 2, G1R_WORDS * 4), s, B, nj);
        return;
    }
    fr_t none = {};
    for (; B.slice0 < points; B.slice0 += B.cap) {
        const uint32_t count = points - B.slice0 < B.cap ? points - B.slice0 : B.cap;
        if (points > B.cap)  // more than the tables hold: this slice's again
            launch_ipa_tables(s, B, nj, 0, count, none);
        hipLaunchKernelGGL(k_ipa_fold4, dim3((count + 15) / 16), dim3(64), lds_share((count + 15) / 16, 4, 0), s, B, nj, count);
    }
}
// planes -> 8-word entries
__global__ __launch_bounds__(256) void k_planes_to_aos(const uint32_t* __restrict__ lo, const uint32_t* __restrict__ hi,
                                                       uint32_t n, uint32_t* __restrict__ out) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    st_aos(out, i, ld_fr((const uint4*)lo, (const uint4*)hi, i));
}
void launch_planes_to_aos(hipStream_t s, const uint32_t* lo, const uint32_t* hi, uint32_t n, uint32_t* out) {
    hipLaunchKernelGGL(k_planes_to_aos, dim3((n + 255) / 256), dim3(256), 0, s, lo, hi, n, out);
}
void launch_g1_addmul(hipStream_t s, const uint32_t* a, const G1Scalar& sc, const uint32_t* b, uint32_t n,
                      uint32_t* out) {
    if (n < G1_ADDMUL_QUADS)
        hipLaunchKernelGGL(k_g1_addmul, dim3(n), dim3(128), lds_share(n, 2, sizeof(g1_pipe_buf)), s, a, sc, b, out);
    else
        hipLaunchKernelGGL(k_g1_addmul4, dim3((n + 15) / 16), dim3(64), lds_share((n + 15) / 16, 4, 0), s, a, sc, b, n, out);
}
// Tables where bases are shared, or where there are enough products for quads; slices of fewer
// bases down to G1_QUADS, below which every product runs its own doublings as without tables
void g1_mul_tables(uint32_t nb, uint32_t n, uint32_t* want, uint32_t* least) {
    const uint32_t used = nb < n ? nb : n;
    *want = used == n && n < G1_QUADS ? 0 : used < ZKH_IPA_TABLES ? used : ZKH_IPA_TABLES;
    *least = *want < G1_QUADS ? *want : G1_QUADS;
}
void launch_g1_mul(hipStream_t s, const uint32_t* base, uint32_t nb, const uint32_t* lo, const uint32_t* hi,
                   uint32_t n, uint32_t* out, uint32_t* tab, uint32_t nt, uint32_t* tops) {
    const uint32_t used = nb < n ? nb : n;
    if (!nt) {
        hipLaunchKernelGGL(k_g1_mul, dim3(n), dim3(128), lds_share(n, 2, sizeof(g1_pipe_buf)), s, base, nb, lo, hi, out);
        return;
    }
    const uint32_t ntops = n < 256 * ZKH_G1_TOPS ? (n + 255) / 256 : ZKH_G1_TOPS;
    hipLaunchKernelGGL(k_g1_top, dim3(ntops), dim3(256), 0, s, lo, hi, n, tops);
    for (uint32_t b0 = 0; b0 < used; b0 += nt) {
        const uint32_t bases = used - b0 < nt ? used - b0 : nt;
        if (bases < G1_QUADS)
            hipLaunchKernelGGL(k_g1_tables, dim3(bases), dim3(64), 0, s, base, b0, tops, ntops, tab);
        else
            hipLaunchKernelGGL(k_g1_tables4, dim3((bases + 15) / 16), dim3(64), 0, s, base, b0, bases, tops, ntops, tab);
        // the products of these bases: all at once if they are all the bases, else pass by pass
        const bool all = bases == nb;
        for (uint64_t i0 = b0; i0 < n; i0 += nb) {
            const uint32_t count = all ? n : (uint32_t)(n - i0 < bases ? n - i0 : bases);
            if (count < G1_QUADS && bases < G1_QUADS) {  // quads leave signed limbs: read by quads
                hipLaunchKernelGGL(k_g1_tab_mul, dim3(count), dim3(64), 0, s, tab, bases, nb, b0, lo, hi, (uint32_t)i0, out);
            } else {
                hipLaunchKernelGGL(k_g1_tab_mul4, dim3((count + 15) / 16), dim3(64), 0, s, tab, bases, nb, b0, lo, hi,
                                   (uint32_t)i0, count, out);
            }
            if (all) break;
        }
    }
}
void launch_pip_sort(hipStream_t s, const uint32_t* lo, const uint32_t* hi, uint32_t m, uint32_t n,
                     uint16_t* lists, uint32_t* offs) {
    hipLaunchKernelGGL(k_pip_sort, dim3(m), dim3(64 * PIP_SEG), 0, s, lo, hi, n, lists, offs);
}
void launch_pip_gens(hipStream_t s, const uint32_t* gens, uint32_t n, uint32_t* tab, PipPlan* plan) {
    hipLaunchKernelGGL(k_pip_gens, dim3((n + 3) / 4), dim3(256), 0, s, gens, n, tab, plan);
}
void launch_pip_alias(hipStream_t s, const uint16_t* lists, const uint32_t* offs, uint32_t m, uint32_t n,
                      uint16_t* alias, uint16_t* walias, PipPlan* plan, uint32_t* wins) {
    hipLaunchKernelGGL(k_pip_alias, dim3(m), dim3(1024), 0, s, lists, offs, n, alias, walias, plan, wins);
}
void launch_pip_bucket(hipStream_t s, const uint32_t* tab, const uint16_t* lists, const uint32_t* offs,
                       const uint16_t* alias, uint32_t m, uint32_t n, PipPlan* plan, uint32_t* items,
                       uint32_t* buckets) {
    hipLaunchKernelGGL(k_pip_plan, dim3(1), dim3(512), 0, s, plan);
    hipLaunchKernelGGL(k_pip_scatter, dim3(m), dim3(1024), 0, s, offs, alias, plan, items);
    hipLaunchKernelGGL(k_pip_bucket, dim3(2048), dim3(64), 0, s, tab, lists, offs, items, n, plan, buckets);
}
void launch_pip_window(hipStream_t s, const uint32_t* buckets, const uint32_t* offs, const uint16_t* alias,
                       uint32_t m, const PipPlan* plan, const uint32_t* wins, uint32_t* partials) {
    const uint32_t most = m * 64;
    hipLaunchKernelGGL(k_pip_window_rows, dim3(most < 8192 ? most : 8192), dim3(64), 0, s, buckets, offs, alias, plan,
                       wins, partials);
    if (most > PIP_WIN_LANES)
        hipLaunchKernelGGL(k_pip_window_lanes, dim3(2048), dim3(64), 0, s, buckets, offs, alias, plan, wins, partials);
}
void launch_pip_combine(hipStream_t s, const uint32_t* partials, const uint16_t* walias, uint32_t m, uint32_t* out) {
    hipLaunchKernelGGL(k_pip_combine, dim3(m), dim3(64), 0, s, partials, walias, out);
}
