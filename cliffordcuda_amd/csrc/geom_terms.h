// Geometric product of single rows term by term, for the rows that a matrix
// representation must not serve, and the test that tells them apart.
//
// A representation mixes all coefficients of a row: a coefficient of the result
// carries a rounding error of about 1.4e-7 |a||b| / sqrt(N) whatever its own
// size (N = 2^n), an exact zero becomes that error, and one infinity reaches
// every coefficient. A sum of terms is accurate against the sum of its own
// |terms|. The two agree for rows whose coefficients are of one scale. A row
// (or the part of it that holds one blade of the ext generators) counts as such
// if its sum of squares is in 2^-80 .. 2^80 and at least 5/8 of its coefficients
// are no smaller than a quarter of the root mean square r. For two such operands
// every coefficient has at least N / 4 terms with both factors that large, so its
// sum of |terms| is at least N r_a r_b / 64 and the representation's error at
// most 1.4e-7 * 64 / sqrt(N) of it (2.8e-7 at n = 10): what the term sums'
// own roundings come to (1.6e-7 to 1.4e-6 at n = 10). N(0, 1) coefficients hold
// 80 % that large and pass at 7 standard deviations of N = 256, uniform ones 86 %.
// Graded rows (vectors, rotors near 1, points), rows with zeros, infinities or
// NaN take the term sums, as all rows did before the representation.
//
// The term sums work on 16-coefficient blocks of four generators with one square
// (+1 or -1; e_0 .. e_3 where these have one): a lane forms one block of the
// result from the blocks of both operands, read from global memory (one operand's
// block is the same for all lanes of a row, so the loads are few against the 256
// multiply-adds of a pair). With the four in front, e_I = chi(I) e_L e_H, L the
// four's part and chi(I) = (-1)^{pairs (l in L, h in H), h < l}, and
//   e_L e_H e_L' e_H' = (-1)^{|H||L'|} (e_L e_L') (e_H e_H').
#pragma once

#include "rep_common.h"

namespace clf {

// ---- the signature with four equal generators in front -----------------------

struct TermSpec {
    int n;
    unsigned c;           // the four, ascending, a byte each
    bool lowneg;          // their square is -1
    bool front;           // they are e_0 .. e_3
    unsigned negh, nulh;  // masks of the others, compressed
};

// false: no four non-null generators have the same square
inline bool term_spec(int n, uint32_t neg, uint32_t nul, TermSpec& t) {
    const unsigned full = (1u << n) - 1u, sets[2] = {full & ~neg & ~nul, full & neg};
    int pick = -1;
    for (int s = 0; s < 2 && pick < 0; ++s)
        if ((sets[s] & 15u) == 15u) pick = s;
    for (int s = 0; s < 2 && pick < 0; ++s)
        if (host_popc(sets[s]) >= 4) pick = s;
    if (n < 4 || pick < 0) return false;
    t = TermSpec{};
    t.n = n;
    t.lowneg = pick == 1;
    unsigned four = 0, h = 0;
    for (int g = 0, k = 0; g < n; ++g) {
        if (k < 4 && ((sets[pick] >> g) & 1u)) {
            t.c |= (unsigned)g << (8 * k++);
            four |= 1u << g;
            continue;
        }
        t.negh |= ((neg >> g) & 1u) << h;
        t.nulh |= ((nul >> g) & 1u) << h;
        ++h;
    }
    t.front = four == 15u;
    return true;
}

// ---- blocks -------------------------------------------------------------------

__host__ __device__ constexpr bool term_negative(bool lowneg, unsigned i, unsigned j) {
    return ((creorder(i, j) + (lowneg ? cpopc(i & j) : 0)) & 1) != 0;
}

__device__ __forceinline__ unsigned term_gen(unsigned c, int k) { return (c >> (8 * k)) & 31u; }

// block index (the others' bits) to coefficient index
template <bool FRONT>
__device__ __forceinline__ unsigned term_place(unsigned h, const TermSpec& t) {
    if constexpr (FRONT) return h << 4;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const unsigned below = h & ((1u << term_gen(t.c, k)) - 1u);
        h = below | ((h ^ below) << 1);
    }
    return h;
}

// bit k: the sign chi changes with the k-th of the four
__device__ __forceinline__ unsigned term_chi(unsigned place, const TermSpec& t) {
    unsigned m = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) m |= (unsigned)(__popc(place & ((1u << term_gen(t.c, k)) - 1u)) & 1) << k;
    return m;
}

__device__ __forceinline__ unsigned term_offset(unsigned l, const TermSpec& t) {
    unsigned o = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) o |= ((l >> k) & 1u) << term_gen(t.c, k);
    return o;
}

// x[L] *= s (-1)^{popc(L & m)}, s in the sign bit of sbit
__device__ __forceinline__ void term_flip(float (&x)[16], unsigned m, unsigned sbit) {
    unsigned f[16];
    f[0] = sbit;
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int l = 0; l < (1 << k); ++l) f[l | (1 << k)] = f[l] ^ ((m << (31 - k)) & 0x80000000u);
#pragma unroll
    for (int l = 0; l < 16; ++l) x[l] = __uint_as_float(__float_as_uint(x[l]) ^ f[l]);
}

// the same for m = 0 or 15 (odd: the sign bit if 15)
__device__ __forceinline__ void term_flip_odd(float (&x)[16], unsigned odd, unsigned sbit) {
#pragma unroll
    for (unsigned l = 0; l < 16; ++l)
        x[l] = __uint_as_float(__float_as_uint(x[l]) ^ ((cpopc(l) & 1) ? sbit ^ odd : sbit));
}

template <bool FRONT>
__device__ __forceinline__ void term_load(const float* __restrict__ row, unsigned place, const TermSpec& t,
                                          float (&x)[16]) {
    if constexpr (FRONT) {
        const float4* p = reinterpret_cast<const float4*>(row + place);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float4 v = p[q];
            x[4 * q] = v.x;
            x[4 * q + 1] = v.y;
            x[4 * q + 2] = v.z;
            x[4 * q + 3] = v.w;
        }
    } else {
#pragma unroll
        for (unsigned l = 0; l < 16; ++l) x[l] = row[place | term_offset(l, t)];
    }
}

template <bool FRONT>
__device__ __forceinline__ void term_store(float* __restrict__ row, unsigned place, const TermSpec& t,
                                           const float (&x)[16]) {
    if constexpr (FRONT) {
        float4* p = reinterpret_cast<float4*>(row + place);
#pragma unroll
        for (int q = 0; q < 4; ++q) p[q] = make_float4(x[4 * q], x[4 * q + 1], x[4 * q + 2], x[4 * q + 3]);
    } else {
#pragma unroll
        for (unsigned l = 0; l < 16; ++l) row[place | term_offset(l, t)] = x[l];
    }
}

// v plus its copy in the lane whose number differs in bit 5 (4)
__device__ __forceinline__ float swap32_sum(float v) {
    float w = v;
    permlane_swap32(v, w);
    return v + w;
}
__device__ __forceinline__ float swap16_sum(float v) {
    float w = v;
    permlane_swap16(v, w);
    return v + w;
}

template <class Sum>
__device__ __forceinline__ void term_add(float (&acc)[16], Sum&& sum) {
#pragma unroll
    for (int l = 0; l < 16; ++l) acc[l] = sum(acc[l]);
}

// The block pair's 256 terms. TERM_C: acc[i ^ j] += s x[i] y[j]; TERM_GA:
// acc[i] += s x[j] y[i ^ j]; TERM_GB: acc[j] += s x[i] y[i ^ j].
enum { TERM_C = 0, TERM_GA = 1, TERM_GB = 2 };

template <int MODE, bool LOWNEG>
__device__ __forceinline__ void term_pair(float (&acc)[16], const float (&x)[16], const float (&y)[16]) {
#pragma unroll
    for (unsigned i = 0; i < 16; ++i)
#pragma unroll
        for (unsigned j = 0; j < 16; ++j) {
            const bool neg = term_negative(LOWNEG, i, j);
            if constexpr (MODE == TERM_C) acc[i ^ j] = __builtin_fmaf(neg ? -x[i] : x[i], y[j], acc[i ^ j]);
            else if constexpr (MODE == TERM_GA) acc[i] = __builtin_fmaf(neg ? -x[j] : x[j], y[i ^ j], acc[i]);
            else acc[j] = __builtin_fmaf(neg ? -x[i] : x[i], y[i ^ j], acc[j]);
        }
}

// Block h of one row of c = a b (X = a, Y = b), ga (X = b, Y = gc) or gb
// (X = a, Y = gc); X's block runs over all, Y's is that ^ h. A pair that a null
// generator takes away is passed over. The lanes of a wave may share a block: 2^log
// of them (log <= 4), whose numbers differ in the lane's top bits, take every
// 2^log-th pair each (from `slice` on), and the first stores the sum; all lanes
// of the wave are then active, with a block each, and may leave it unstored.
template <int MODE, bool FRONT>
__device__ __forceinline__ void term_block_of(const float* __restrict__ X, const float* __restrict__ Y,
                                              float* __restrict__ out, unsigned h, const TermSpec& t, unsigned slice,
                                              int log, bool keep) {
    float acc[16];
#pragma unroll
    for (int l = 0; l < 16; ++l) acc[l] = 0.f;
    const unsigned nb = 1u << (t.n - 4);
#pragma unroll 1
    for (unsigned first = 0; first < nb; first += 1u << log) {
        const unsigned m = first + slice;
        const unsigned i = MODE == TERM_GA ? h : m, j = MODE == TERM_C ? m ^ h : MODE == TERM_GA ? m : h;
        if (i & j & t.nulh) continue;
        const unsigned px = term_place<FRONT>(m, t), py = term_place<FRONT>(m ^ h, t);
        float x[16], y[16];
        term_load<FRONT>(X, px, t, x);
        term_load<FRONT>(Y, py, t, y);
        const unsigned s = (unsigned)(reorder_parity(i, j) ^ __popc(i & j & t.negh)) << 31;
        const unsigned odd = (unsigned)__popc(i) << 31;  // (-1)^{|H||L'|}
        // (gb: |L'| of the result is |L| of a plus that of gc)
        if (MODE == TERM_C) term_flip_odd(y, odd, s);
        else term_flip_odd(x, odd, s);
        if (MODE == TERM_GB) term_flip_odd(y, odd, 0u);
        if (!FRONT) {
            term_flip(x, term_chi(px, t), 0u);
            term_flip(y, term_chi(py, t), 0u);
        }
        if (t.lowneg) term_pair<MODE, true>(acc, x, y);
        else term_pair<MODE, false>(acc, x, y);
    }
    if (log >= 1) term_add(acc, [](float v) { return swap32_sum(v); });
    if (log >= 2) term_add(acc, [](float v) { return swap16_sum(v); });
    if (log >= 3) term_add(acc, [](float v) { return v + xor16<8>(v); });
    if (log >= 4) term_add(acc, [](float v) { return v + xor16<4>(v); });
    if (slice != 0u || !keep) return;
    const unsigned ph = term_place<FRONT>(h, t);
    if (!FRONT) term_flip(acc, term_chi(ph, t), 0u);
    term_store<FRONT>(out, ph, t, acc);
}

template <int MODE>
__device__ __forceinline__ void term_block(const float* __restrict__ X, const float* __restrict__ Y,
                                           float* __restrict__ out, unsigned h, const TermSpec& t, unsigned slice = 0,
                                           int log = 0, bool keep = true) {
    if (t.front) term_block_of<MODE, true>(X, Y, out, h, t, slice, log, keep);  // uniform
    else term_block_of<MODE, false>(X, Y, out, h, t, slice, log, keep);
}

// ---- coefficients of one scale -------------------------------------------------

constexpr float kEvenMin = 0x1p-80f, kEvenMax = 0x1p80f;  // of a part's sum of squares

__device__ __forceinline__ bool even_range(float sumsq) { return sumsq >= kEvenMin && sumsq <= kEvenMax; }

// a quarter of the root mean square of 2^log_n values
__device__ __forceinline__ float even_level(float sumsq, int log_n) {
    return __builtin_amdgcn_sqrtf(__builtin_ldexpf(sumsq, -4 - log_n));
}

__device__ __forceinline__ bool even_count(int large, int of) { return 8 * large >= 5 * of; }

__device__ __forceinline__ float sumsq4(const float4& v) {
    return __builtin_fmaf(v.x, v.x, __builtin_fmaf(v.y, v.y, __builtin_fmaf(v.z, v.z, v.w * v.w)));
}

// sums over the 16-lane row and over the wave, in all lanes
__device__ __forceinline__ float row16_sum(float v) {
    v += dpp16<0xB1>(v);   // quad_perm [1,0,3,2]
    v += dpp16<0x4E>(v);   // quad_perm [2,3,0,1]
    v += dpp16<0x141>(v);  // row_half_mirror: the other quad of eight
    v += dpp16<0x140>(v);  // row_mirror: the other eight
    return v;
}

__device__ __forceinline__ float wave_total(float v) {
    return swap32_sum(swap16_sum(row16_sum(v)));
}

// coefficients of the lanes' float4 that reach the level, over the lanes of mask
__device__ __forceinline__ int even_large(const float4& v, float level, unsigned long long mask = ~0ull) {
    return __popcll(__ballot(__builtin_fabsf(v.x) >= level) & mask) +
           __popcll(__ballot(__builtin_fabsf(v.y) >= level) & mask) +
           __popcll(__ballot(__builtin_fabsf(v.z) >= level) & mask) +
           __popcll(__ballot(__builtin_fabsf(v.w) >= level) & mask);
}

}  // namespace clf
