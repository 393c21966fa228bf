// Geometric product of the large algebras (n = 9 .. 12) through 32 x 32 real
// matrices on the matrix cores.
//
// Ten generators ("base") form a signature with Cl = M_32(R) (p - q = 0 or 2
// mod 8): 10 - D of the n generators and D dummies that no blade of a row
// holds (their coefficients are staged as zeros), which lets in the signatures
// of which no ten (n = 9: no nine) generators are of real type. The other
// K = n - 10 + D generators ("ext", any square, null too) extend it. With every
// blade written e_I e_S (I base, S ext) a row is 2^K base rows x_S, and for
// (A_S e_S)(B_J e_J):
//   C_R = sum_{S ^ J = R} sigma(S, J) A_S alpha^{|S|}(B_J),
// alpha the grade involution of the base (e_S passes B_J's blades) and sigma
// the ext signs. In the representation phi each term is one 32 x 32 x 32
// product: 4^K products of 32768 multiply-adds a row instead of 4^n terms
// (without dummies 1/32 of them). Backward:
//   gA_S = sum_J sigma(S, J) G_{S^J} alpha^{|S|}(B_J)^T,
//   gB_J = sum_S sigma(S, J) alpha^{|S|}(A_S)^T alpha^{|S|}(G_{S^J}).
// alpha is the conjugation by the base pseudoscalar, phi = +-P(ox, oz):
//   alpha(B)[k][j] = (-1)^{popc(oz & (k ^ j))} B[k ^ ox][j ^ ox],
// so an operand of alpha(B) is B's own read at another column with two signs.
//
// Layout. One wave takes one base row (K = 0: four rows per workgroup, K = 1
// two, K = 2 one; the 2^K waves of a row share their blocks through LDS; the
// dummies are the top bits of a blade's place there). Lane
// (h, x) gathers the 16 blades of the labels (x, 16h + zl) (real Pauli products
// P(x, z) as in rep.hip), runs the 32-point transform over z (16 points in
// registers, the last stage across the lane halves by permlane swaps) and
// writes P[r][p] = W[r][p] of the plain conversion or W'[r][p] = W[r][p ^ r] of
// the transposed one. Operand k of MFMA lane i is then column i of row i ^ k:
//   phi[i][k] = W'[i ^ k][i],  phi^T[i][k] = W[i ^ k][i],
// one LDS address per lane, xor-ed with a step constant. Element (r, p) sits at
//   word 32 rho(r) + (p ^ 4 (r & 7)),  rho(r) = r ^ ((r >> 3) & 1),
// which is linear over xor and free of bank conflicts for the b128 row writes
// (8 lanes, 8 groups), the b32 column reads (32 lanes, 32 banks), the b32 result
// writes at [i ^ j][j] and the b128 row reads (16 lanes of a set, 16 groups).
// Staged rows are chunk-swizzled (chunk group bit t flipped by the parity of
// the chunk index under a host-chosen mask) so that the 32 gathers of a step
// fall on 32 banks.
//
// Rows whose coefficients are not of one scale are formed term by term in the
// same launch (geom_terms.h). The test costs about 90 of 740 vector instructions
// of a forward wave.
//
// Bound: 12 (forward) and 20 (backward) 2^n bytes a row over HBM against 4^K
// 1024 matrix-core cycles a row forward and twice that backward; vector
// instructions beside them (the test added 3 to 10 %); a workgroup's own latency
// for a few rows. Measured (us, forward + backward; before: the per-term kernels),
// N(0, 1) rows: n = 10, 16384 rows 37 + 75 (5.4 and 4.5 TB/s; 358 + 690); n = 11,
// 4096 rows 27.5 + 50 (3.7 and 3.4 TB/s; 542 + 1180); n = 12, 1024 rows 22.7 + 41
// (660 + 2580), 64 rows 9 + 15 (35 + 63). With dummies, 8000 rows: n = 9 20 + 36
// (62 + 115), Cl(7,2) 48 + 86 (57 + 105), Cl(8,2) 45 + 84 (184 + 355), Cl(8,3)
// 123 + 244 (950 + 2070). Rows that all go by their terms: n = 9 68 + 148, Cl(7,2)
// 67 + 136, n = 10 431 + 893, n = 11 422 + 852, n = 12 440 + 913 and 32 + 67,
// Cl(8,2) 211 + 439, Cl(8,3) 792 + 1604.
#include <map>
#include <mutex>

#include "geom_terms.h"

namespace clf {

constexpr int kBig = 32;         // matrix side
constexpr int kBigBase = 10;     // base generators
constexpr int kBigMaxExt = 2;

struct Rep32Table {
    unsigned lane_pos[64];          // staged position (floats) of the blade of label (x, 16h), lane = 32h + x, ext blade 1
    unsigned z_pos[16];             // xor for the low label bits zl
    unsigned ext_pos[1 << kBigMaxExt];      // xor for ext blade S
    unsigned sgn[1 << kBigMaxExt][64];      // bit zl: the coefficient enters with -1; bit 16 + zl: the transposed conversion's sign
    unsigned chunk_mask[3];         // chunk group bit t is flipped by the parity of chunk & chunk_mask[t]
    unsigned ox, oz;                // label of the base pseudoscalar
    unsigned neg_pairs, zero_pairs; // ext signs: bit 4 S + J
    TermSpec terms;                 // for the rows that are not of one scale
};

// word of element (r, p), split into its xor-linear row part and p itself
__host__ __device__ constexpr unsigned big_row(unsigned r) { return ((r ^ ((r >> 3) & 1u)) << 5) ^ ((r & 7u) << 2); }

__device__ __forceinline__ float big_ld(const float* base, unsigned byte) {
    return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(base) + byte);
}

__device__ __forceinline__ void big_st(float* base, unsigned byte, float v) {
    *reinterpret_cast<float*>(reinterpret_cast<char*>(base) + byte) = v;
}

template <int K>
__device__ __forceinline__ void big_sync() {
    if constexpr (K == 0) wave_lds_sync();  // a row is one wave's own
    else __syncthreads();
}

__device__ __forceinline__ unsigned big_chunk(unsigned q, const Rep32Table& T) {
    unsigned s = 0;
#pragma unroll
    for (int t = 0; t < 3; ++t) s |= (unsigned)(__popc(q & T.chunk_mask[t]) & 1) << t;
    return q ^ s;
}

struct BigRow {
    float4 v[4];
};

// places (chunks) in the row's region of the wave's four chunks per lane: the
// first 4 >> D hold its part of the row, the others the dummies' zeros
template <int K, int D>
__device__ __forceinline__ void big_places(unsigned S, unsigned lane, const Rep32Table& T, unsigned (&cpos)[4]) {
    constexpr unsigned RC = 4u >> D;
#pragma unroll
    for (unsigned j = 0; j < 4; ++j)
        cpos[j] = big_chunk(((j / RC) << (8 + K - D)) | (S * (256u >> D) + 64u * (j % RC) + lane), T);
}

// first float of the wave's part of a row; ld 0: one row read for every batch row
template <int K, int D>
__device__ __forceinline__ long long big_off(long long row, long long ld, unsigned S) {
    return ((row & row_mask(ld)) << (kBigBase + K - D)) + S * (1024u >> D);
}

// the wave's 1024 >> D floats of its row
template <int D, bool NT>
__device__ __forceinline__ BigRow big_fetch(const float* __restrict__ src, int lane) {
    BigRow r;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if (j >= (4 >> D)) {
            r.v[j] = make_float4(0.f, 0.f, 0.f, 0.f);
            continue;
        }
        const float4* q = reinterpret_cast<const float4*>(src) + lane + 64 * j;
        r.v[j] = NT ? load_stream(q) : *q;
    }
    return r;
}

// Which of the wave's parts of its rows are not of one scale (geom_terms.h), bit
// i for rows[i]. Each part is converted by itself and two parts' products meet
// in plain sums, so the parts of a row may differ in scale.
template <int D, int COUNT>
__device__ __forceinline__ unsigned big_uneven(const BigRow* const (&rows)[COUNT]) {
    unsigned bad = 0;
#pragma unroll
    for (int i = 0; i < COUNT; ++i) {
        float q = 0.f;
#pragma unroll
        for (int j = 0; j < (4 >> D); ++j) q += sumsq4(rows[i]->v[j]);
        q = wave_total(q);
        const float level = even_level(q, kBigBase - D);
        int large = 0;
#pragma unroll
        for (int j = 0; j < (4 >> D); ++j) large += even_large(rows[i]->v[j], level);
        bad |= even_range(q) && even_count(large, 1024 >> D) ? 0u : 1u << i;
    }
    return __builtin_amdgcn_readfirstlane(bad);
}

// The or of the row's waves' marks; every wave writes its own before a big_sync
// and calls this after it.
template <int K>
__device__ __forceinline__ unsigned big_marks(const unsigned (&marks)[4], unsigned first, unsigned own) {
    if constexpr (K == 0) return own;
    unsigned m = 0;
#pragma unroll
    for (unsigned s = 0; s < (1u << K); ++s) m |= marks[first + s];
    return __builtin_amdgcn_readfirstlane(m);
}

// Whether no row of the workgroup (K = 0: of the wave) has use for its matrices
template <int K, class All>
__device__ __forceinline__ bool big_skip(const unsigned (&marks)[4], bool own, All&& all) {
    if constexpr (K == 0) return own;
    constexpr unsigned NS = 1u << K;
    bool skip = true;
#pragma unroll
    for (unsigned r = 0; r < 4; r += NS) {
        unsigned m = 0;
#pragma unroll
        for (unsigned s = 0; s < NS; ++s) m |= marks[r + s];
        skip = skip && all(m);
    }
    return __builtin_amdgcn_readfirstlane(skip);
}

// one row by its terms: the lanes of the row's waves (of all its workgroups),
// 2^log to a block
template <int K, int D, int MODE>
__device__ __forceinline__ void big_terms(const float* __restrict__ X, long long ldx, const float* __restrict__ Y,
                                          long long ldy, float* __restrict__ out, long long row, unsigned S,
                                          unsigned lane, const TermSpec& t, int log) {
    const unsigned per = 6 - log;  // a wave's blocks, log2
    const unsigned h = ((blockIdx.y << K | S) << per) | (lane & ((1u << per) - 1u));
    term_block<MODE>(X + big_off<K, D>(row, ldx, 0), Y + big_off<K, D>(row, ldy, 0), out + big_off<K, D>(row, 1, 0), h,
                     t, lane >> per, log);
}

__device__ __forceinline__ void big_stage(float* __restrict__ region, const BigRow& r, const unsigned (&cpos)[4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) reinterpret_cast<float4*>(region)[cpos[j]] = r.v[j];
}

template <int D, bool NT>
__device__ __forceinline__ void big_store(float* __restrict__ dst, const float* __restrict__ region,
                                          const unsigned (&cpos)[4], int lane) {
    float4 v[4];
#pragma unroll
    for (int j = 0; j < (4 >> D); ++j) v[j] = reinterpret_cast<const float4*>(region)[cpos[j]];
#pragma unroll
    for (int j = 0; j < (4 >> D); ++j) {
        float4* q = reinterpret_cast<float4*>(dst) + lane + 64 * j;
        if (NT) store_stream(q, v[j]);
        else *q = v[j];
    }
}

// Keeps values derived from v (addresses, signs) from being held in registers
// across the loop: they are recomputed where they are used.
__device__ __forceinline__ unsigned big_fresh(unsigned v) {
    asm volatile("" : "+v"(v));
    return v;
}

// raw coefficients of the lane's 16 labels
__device__ __forceinline__ void big_gather(const float* __restrict__ region, unsigned pos, const Rep32Table& T,
                                           float (&t)[16]) {
    pos = big_fresh(pos);
#pragma unroll
    for (int z = 0; z < 16; ++z) t[z] = region[pos ^ T.z_pos[z]];
}

// t with the conversion's signs (bits SHIFT .. SHIFT + 15 of m), transformed over z, written as the rows of P
template <int SHIFT>
__device__ __forceinline__ void big_convert(const float (&raw)[16], unsigned m, float* __restrict__ P, unsigned x,
                                            unsigned h) {
    float t[16];
    m = big_fresh(m);
#pragma unroll
    for (int z = 0; z < 16; ++z)
        t[z] = __uint_as_float(__float_as_uint(raw[z]) ^ ((m << (31 - SHIFT - z)) & 0x80000000u));
    wht_inplace<16>(t);
    // last stage: after the swaps t[j] and t[j + 8] hold z bit 4 = 0 and 1 of
    // column 8h + j, on both halves
    float w[2][8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        permlane_swap32(t[j], t[j + 8]);
        w[0][j] = t[j] + t[j + 8];
        w[1][j] = t[j] - t[j + 8];
    }
    float4* row = reinterpret_cast<float4*>(P + ((x ^ ((x >> 3) & 1u)) << 5));
#pragma unroll
    for (int c4 = 0; c4 < 2; ++c4)
#pragma unroll
        for (int u = 0; u < 2; ++u)
            row[(4u * c4 + 2u * h + u) ^ (x & 7u)] =
                make_float4(w[c4][4 * u], w[c4][4 * u + 1], w[c4][4 * u + 2], w[c4][4 * u + 3]);
}

// acc(i, j) = C[i][j] to P[i ^ j][j] (the plain conversion of C), the inverse
// transform, and the lane's 16 signed coefficients
__device__ __forceinline__ void big_unconvert(const floatx16& acc, float* __restrict__ P, unsigned m, unsigned lane,
                                              float (&t)[16]) {
    const unsigned x = lane & 31u, h = lane >> 5;
    m = big_fresh(m);
    const unsigned base = (big_row(x) ^ x ^ (h ? big_row(4u) : 0u)) << 2;
#pragma unroll
    for (int q = 0; q < 16; ++q) big_st(P, base ^ (big_row(8u * (q >> 2) + (q & 3u)) << 2), acc[q]);
    wave_lds_sync();
    float w[2][8];
    const float4* row = reinterpret_cast<const float4*>(P + ((x ^ ((x >> 3) & 1u)) << 5));
#pragma unroll
    for (int c4 = 0; c4 < 2; ++c4)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const float4 v = row[(4u * c4 + 2u * h + u) ^ (x & 7u)];
            w[c4][4 * u] = v.x;
            w[c4][4 * u + 1] = v.y;
            w[c4][4 * u + 2] = v.z;
            w[c4][4 * u + 3] = v.w;
        }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        t[j] = w[0][j] + w[1][j];
        t[j + 8] = w[0][j] - w[1][j];
        permlane_swap32(t[j], t[j + 8]);
    }
    wht_inplace<16>(t);
#pragma unroll
    for (int z = 0; z < 16; ++z)
        t[z] = __uint_as_float(__float_as_uint(t[z] * 0.03125f) ^ ((m << (31 - z)) & 0x80000000u));
}

__device__ __forceinline__ void big_scatter(float* __restrict__ region, unsigned pos, const Rep32Table& T,
                                            const float (&t)[16]) {
    pos = big_fresh(pos);
#pragma unroll
    for (int z = 0; z < 16; ++z) region[pos ^ T.z_pos[z]] = t[z];
}

// acc += A B, A[i][k] at byte abase ^ (row constant of k) of P, B[k][j] at
// bbase likewise with the sign bsign ^ (parity of k & kmask)
template <bool SIGNED>
__device__ __forceinline__ void big_mac(floatx16& acc, const float* __restrict__ PA, unsigned abase, unsigned asign,
                                        const float* __restrict__ PB, unsigned bbase, unsigned bsign,
                                        unsigned kmask) {
    float a[16], b[16];
    abase = big_fresh(abase);
    bbase = big_fresh(bbase);
#pragma unroll
    for (int s = 0; s < 16; ++s) {
        a[s] = big_ld(PA, abase ^ (big_row(s) << 2));
        b[s] = big_ld(PB, bbase ^ (big_row(s) << 2));
        if (SIGNED) {
            a[s] = __uint_as_float(__float_as_uint(a[s]) ^ asign);
            b[s] = __uint_as_float(__float_as_uint(b[s]) ^ bsign ^ ((unsigned)(__popc(kmask & s) & 1) << 31));
        }
    }
    // two short chains per product, then plain sums: half the rounding of one
    // running sum over all products' steps
    floatx16 c0 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, c1 = c0;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        c0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s], b[s], c0, 0, 0, 0);
        c1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s + 8], b[s + 8], c1, 0, 0, 0);
    }
#pragma unroll
    for (int q = 0; q < 16; ++q) acc[q] += c0[q] + c1[q];
}

// What a lane needs of its place: its matrix index i (= j), half h, and the
// byte bases of its operand columns, plain and of alpha.
struct BigLane {
    unsigned plain, alpha;  // byte of [i ^ 16h][i], of [i ^ 16h][i ^ ox]
    unsigned sign_i;        // (-1)^{popc(oz & i)} as a sign bit
    unsigned sign_ik;       // (-1)^{popc(oz & (i ^ 16h))}
};

__device__ __forceinline__ BigLane big_lane(unsigned lane, const Rep32Table& T) {
    const unsigned i = lane & 31u, h = lane >> 5;
    BigLane L;
    L.plain = (big_row(i) ^ (h ? big_row(16u) : 0u) ^ i) << 2;
    L.alpha = L.plain ^ (T.ox << 2);
    L.sign_i = (unsigned)(__popc(T.oz & i) & 1) << 31;
    L.sign_ik = (unsigned)(__popc(T.oz & (i ^ (h << 4))) & 1) << 31;
    return L;
}

template <int K, int D, bool NT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void rep32_fwd_kernel(
    const float* __restrict__ A, long long lda, const float* __restrict__ B, long long ldb, float* __restrict__ C,
    long long batch, int terms_log, Rep32Table T) {
    constexpr unsigned NS = 1u << K;  // base rows per row
    constexpr int kRows = 4 >> K;     // rows per workgroup
    __shared__ __attribute__((aligned(4096))) float lds[2][4 * 1024];
    __shared__ unsigned marks[4];
    const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63u;
    const unsigned x = lane & 31u, h = lane >> 5;
    const unsigned S = wave & (NS - 1u), first = wave - S;
    float* ra = &lds[0][first * 1024];  // the row's region: staged a, then its P blocks
    float* rb = &lds[1][first * 1024];
    const unsigned pos = T.lane_pos[lane] ^ T.ext_pos[S];
    const unsigned m = T.sgn[S][lane];
    const BigLane L = big_lane(lane, T);
    unsigned cpos[4];
    big_places<K, D>(S, lane, T, cpos);
    long long row = (long long)blockIdx.x * kRows + (wave >> K);
    const bool live = row < batch;  // rows past the end recompute the last row and are not stored
    row = live ? row : batch - 1;
    const long long off = big_off<K, D>(row, 1, S);
    const BigRow va = big_fetch<D, NT>(A + big_off<K, D>(row, lda, S), lane);
    const BigRow vb = big_fetch<D, NT>(B + big_off<K, D>(row, ldb, S), lane);
    big_stage(ra, va, cpos);
    big_stage(rb, vb, cpos);
    big_sync<K>();
    float ta[16], tb[16];
    big_gather(ra, pos, T, ta);
    big_gather(rb, pos, T, tb);
    const unsigned own = big_uneven<D, 2>({&va, &vb});
    if (K > 0 && lane == 0) marks[wave] = own;
    big_sync<K>();
    const unsigned by_terms = big_marks<K>(marks, first, own);
    if (blockIdx.y == 0 && !big_skip<K>(marks, own != 0u, [](unsigned r) { return r != 0u; })) {
        big_convert<16>(ta, m, ra + S * 1024, x, h);
        big_convert<0>(tb, m, rb + S * 1024, x, h);
        big_sync<K>();
        floatx16 acc = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (unsigned I = 0; I < NS; ++I) {
            const unsigned J = I ^ S, pair = 4u * I + J;
            const bool odd = (__popc(I) & 1) != 0;
            if (K == 0) {
                big_mac<false>(acc, ra, L.plain, 0u, rb, L.plain, 0u, 0u);
            } else if (!((T.zero_pairs >> pair) & 1u)) {
                const unsigned flip = ((T.neg_pairs >> pair) & 1u) << 31;
                big_mac<true>(acc, ra + I * 1024, L.plain, 0u, rb + J * 1024, odd ? L.alpha : L.plain,
                              odd ? (L.sign_ik ^ flip) : flip, odd ? T.oz : 0u);
            }
        }
        big_sync<K>();
        big_unconvert(acc, ra + S * 1024, m, lane, ta);
        big_scatter(rb, pos, T, ta);
        big_sync<K>();
        if (live && !by_terms) big_store<D, NT>(C + off, rb, cpos, lane);
    }
    if (live && by_terms) big_terms<K, D, TERM_C>(A, lda, B, ldb, C, row, S, lane, T.terms, terms_log);
}

constexpr unsigned kMarkGA = 1 | 2, kMarkGB = 1 | 4;  // rows (gc, b, a) that a gradient needs of one scale

template <int K, int D, bool NT, bool WA, bool WB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void rep32_bwd_kernel(
    const float* __restrict__ A, long long lda, const float* __restrict__ B, long long ldb,
    const float* __restrict__ GC, long long ldg, float* __restrict__ GA, float* __restrict__ GB, long long batch,
    int terms_log, Rep32Table T) {
    constexpr unsigned NS = 1u << K;
    constexpr int kRows = 4 >> K;
    __shared__ __attribute__((aligned(4096))) float lds[3][4 * 1024];
    __shared__ unsigned marks[4];
    const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63u;
    const unsigned x = lane & 31u, h = lane >> 5;
    const unsigned S = wave & (NS - 1u), first = wave - S;
    float* r0 = &lds[0][first * 1024];  // staged gc, then P blocks of gc
    float* r1 = &lds[1][first * 1024];  // staged b, then P blocks of b, of a, then gb in blade order
    float* r2 = &lds[2][first * 1024];  // staged a, then ga in blade order
    const unsigned pos = T.lane_pos[lane] ^ T.ext_pos[S];
    const unsigned m = T.sgn[S][lane];
    const BigLane L = big_lane(lane, T);
    unsigned cpos[4];
    big_places<K, D>(S, lane, T, cpos);
    const floatx16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    long long row = (long long)blockIdx.x * kRows + (wave >> K);
    const bool live = row < batch;
    row = live ? row : batch - 1;
    const long long off = big_off<K, D>(row, 1, S);
    const BigRow vg = big_fetch<D, NT>(GC + big_off<K, D>(row, ldg, S), lane);
    BigRow va, vb;
    if (WA) vb = big_fetch<D, NT>(B + big_off<K, D>(row, ldb, S), lane);
    if (WB) va = big_fetch<D, NT>(A + big_off<K, D>(row, lda, S), lane);
    big_stage(r0, vg, cpos);
    if (WA) big_stage(r1, vb, cpos);
    if (WB) big_stage(r2, va, cpos);
    big_sync<K>();
    float tg[16], ta[16], tb[16];
    big_gather(r0, pos, T, tg);
    if (WA) big_gather(r1, pos, T, tb);
    if (WB) big_gather(r2, pos, T, ta);
    unsigned own;  // gc, b, a
    if constexpr (WA && WB) own = big_uneven<D, 3>({&vg, &vb, &va});
    else if constexpr (WA) own = big_uneven<D, 2>({&vg, &vb});
    else own = big_uneven<D, 2>({&vg, &va}) != 0u ? kMarkGB : 0u;
    if (K > 0 && lane == 0) marks[wave] = own;
    big_sync<K>();
    const unsigned by_terms = big_marks<K>(marks, first, own);
    const auto all = [](unsigned r) { return (!WA || (r & kMarkGA)) && (!WB || (r & kMarkGB)); };
    if (blockIdx.y == 0 && !big_skip<K>(marks, all(own), all)) {
        if (WA) {
            // gA_S = sum_J sigma(S, J) G_{S^J} alpha^{|S|}(B_J)^T
            big_convert<16>(tg, m, r0 + S * 1024, x, h);
            big_convert<16>(tb, m, r1 + S * 1024, x, h);
            big_sync<K>();
            const bool odd = (__popc(S) & 1) != 0;
            floatx16 acc = zero;
#pragma unroll 1
            for (unsigned J = 0; J < NS; ++J) {
                const unsigned pair = 4u * S + J;
                if (K == 0) {
                    big_mac<false>(acc, r0, L.plain, 0u, r1, L.plain, 0u, 0u);
                } else if (!((T.zero_pairs >> pair) & 1u)) {
                    const unsigned flip = ((T.neg_pairs >> pair) & 1u) << 31;
                    big_mac<true>(acc, r0 + (S ^ J) * 1024, L.plain, 0u, r1 + J * 1024, odd ? L.alpha : L.plain,
                                  odd ? (L.sign_ik ^ flip) : flip, odd ? T.oz : 0u);
                }
            }
            // r2 is free (a was gathered before the last two syncs); the block
            // is the wave's own until the scatter
            big_unconvert(acc, r2 + S * 1024, m, lane, tb);
            big_sync<K>();
            big_scatter(r2, pos, T, tb);
        }
        if (WB) {
            // gB_S = sum_I sigma(I, S) alpha^{|I|}(A_I)^T alpha^{|I|}(G_{I^S}); the two
            // alphas' signs of k cancel
            big_convert<0>(tg, m, r0 + S * 1024, x, h);
            big_convert<0>(ta, m, r1 + S * 1024, x, h);
        }
        big_sync<K>();
        if (WA && live && !(by_terms & kMarkGA)) big_store<D, NT>(GA + off, r2, cpos, lane);
        if (WB) {
            floatx16 acc = zero;
#pragma unroll 1
            for (unsigned I = 0; I < NS; ++I) {
                const unsigned pair = 4u * I + S;
                const bool odd = (__popc(I) & 1) != 0;
                if (K == 0) {
                    big_mac<false>(acc, r1, L.plain, 0u, r0, L.plain, 0u, 0u);
                } else if (!((T.zero_pairs >> pair) & 1u)) {
                    const unsigned flip = ((T.neg_pairs >> pair) & 1u) << 31;
                    big_mac<true>(acc, r1 + I * 1024, odd ? L.alpha : L.plain, odd ? L.sign_i : 0u,
                                  r0 + (I ^ S) * 1024, odd ? L.alpha : L.plain, odd ? (L.sign_i ^ flip) : flip, 0u);
                }
            }
            big_sync<K>();
            big_unconvert(acc, r0 + S * 1024, m, lane, ta);
            big_scatter(r1, pos, T, ta);
            big_sync<K>();
            if (live && !(by_terms & kMarkGB)) big_store<D, NT>(GB + off, r1, cpos, lane);
        }
    }
    if (!live) return;
    if (WA && (by_terms & kMarkGA)) big_terms<K, D, TERM_GA>(B, ldb, GC, ldg, GA, row, S, lane, T.terms, terms_log);
    if (WB && (by_terms & kMarkGB)) big_terms<K, D, TERM_GB>(A, lda, GC, ldg, GB, row, S, lane, T.terms, terms_log);
}

// ---- host side --------------------------------------------------------------

namespace {

// How a signature is served: the ext generators, the number D of dummies and
// how many of them are negative. The first choice (fewest dummies, so fewest
// products; highest ext generators first) for which the base holds no null
// generator and is of real type.
struct BigSplit {
    unsigned ext;
    int k, d, dneg;
};

bool big_split(int n, uint32_t neg, uint32_t nul, BigSplit& c) {
    for (int d = 0; d <= 2; ++d) {
        const int k = n - kBigBase + d;
        if (k < 0 || k > kBigMaxExt || (d == 2 && k != 1)) continue;
        for (unsigned pick = 0; pick < (k == 0 ? 1u : k == 1 ? 16u : 256u); ++pick) {
            const int a = n - 1 - (int)(pick & 15u), b = n - 1 - (int)(pick >> 4);
            if ((k >= 1 && a < 0) || (k == 2 && (b < 0 || b <= a))) continue;
            const unsigned ext = (k >= 1 ? 1u << a : 0u) | (k == 2 ? 1u << b : 0u);
            const unsigned base = ((1u << n) - 1u) & ~ext;
            if (base & nul) continue;
            for (int dneg = 0; dneg <= d; ++dneg) {
                const int t = ((kBigBase - 2 * (host_popc(base & neg) + dneg)) % 8 + 8) % 8;
                if (t != 0 && t != 2) continue;
                c = {ext, k, d, dneg};
                return true;
            }
        }
    }
    return false;
}

// Anticommuting real Pauli products on five qubits with the wanted squares
// (the first q of them -1), by depth-first search in a fixed order.
bool big_generators(int q, unsigned* gx, unsigned* gz) {
    unsigned cand[kBigBase] = {0};
    int g = 0;
    while (g >= 0 && g < kBigBase) {
        bool found = false;
        for (unsigned c = cand[g] + 1; c < kBig * kBig; ++c) {
            const unsigned cx = c / kBig, cz = c % kBig;
            if ((host_popc(cx & cz) & 1) != (g < q ? 1 : 0)) continue;
            bool ok = true;
            for (int p = 0; p < g && ok; ++p) ok = ((host_popc(cz & gx[p]) + host_popc(gz[p] & cx)) & 1) == 1;
            if (!ok) continue;
            cand[g] = c;
            gx[g] = cx;
            gz[g] = cz;
            found = true;
            break;
        }
        if (found) {
            ++g;
            if (g < kBigBase) cand[g] = 0;
        } else {
            --g;
        }
    }
    return g == kBigBase;
}

// Adds v to a basis kept in echelon form; false if it is in the span already.
bool big_independent(unsigned (&basis)[5], int& rank, unsigned v) {
    for (int i = 0; i < rank; ++i)
        if ((v ^ basis[i]) < v) v ^= basis[i];
    if (!v) return false;
    basis[rank++] = v;
    for (int i = rank - 1; i > 0 && basis[i] > basis[i - 1]; --i) std::swap(basis[i], basis[i - 1]);
    return true;
}

// n, neg: with the dummies as the top generators
bool big_table_build(int n, uint32_t neg, uint32_t nul, unsigned ext, Rep32Table& T) {
    const int k = n - kBigBase;
    const unsigned full = (1u << n) - 1u, base = full & ~ext;
    unsigned px[kBigBase], pz[kBigBase];
    if (!big_generators(host_popc(base & neg), px, pz)) return false;

    // The search's generators may be dealt to the metric's generators of the
    // same square in any order: take the first deal (of a fixed sequence of
    // shuffles) for which the blades of one label column fall on 32 banks.
    // For fixed z the position's five low bits, as functions of x, are those of
    // the blade: bits 0, 1 as they are, bits 2..4 plus any higher bits through
    // the chunk masks.
    unsigned gx[16] = {0}, gz[16] = {0}, blade_of[kBig * kBig] = {0};
    unsigned long long seed = 1;
    int best = -1;
    unsigned bgx[16] = {0}, bgz[16] = {0}, bmask[3] = {0, 0, 0};
    for (int attempt = 0; attempt < 64 && best < 5; ++attempt) {
        int slot[kBigBase];
        int np = 0, nn = 0;
        const int q = host_popc(base & neg);
        int perm[kBigBase];
        for (int i = 0; i < kBigBase; ++i) perm[i] = i;
        auto shuffle = [&](int lo, int hi) {
            for (int i = hi - 1; i > lo; --i) {
                seed = seed * 6364136223846793005ULL + 1442695040888963407ULL;
                std::swap(perm[i], perm[lo + (int)((seed >> 33) % (unsigned)(i - lo + 1))]);
            }
        };
        if (attempt) {
            shuffle(0, q);
            shuffle(q, kBigBase);
        }
        int idx = 0;
        for (int g = 0; g < n; ++g) {
            if (!((base >> g) & 1u)) continue;
            slot[idx] = ((neg >> g) & 1u) ? perm[nn++] : perm[q + np++];
            gx[g] = px[slot[idx]];
            gz[g] = pz[slot[idx]];
            ++idx;
        }
        // blade of every label; column z = 0 gives x -> blade
        for (unsigned c = 0; c < (1u << kBigBase); ++c) {
            unsigned I = 0, x = 0, z = 0, r = c;
            for (int g = 0; g < n; ++g)
                if ((base >> g) & 1u) {
                    if (r & 1u) {
                        I |= 1u << g;
                        x ^= gx[g];
                        z ^= gz[g];
                    }
                    r >>= 1;
                }
            blade_of[z * kBig + x] = I;
        }
        // a functional on the column: the 5-bit vector of its values at x = 1, 2, 4, 8, 16
        auto functional = [&](unsigned mask) {
            unsigned f = 0;
            for (int b = 0; b < 5; ++b) f |= (unsigned)(host_popc(blade_of[1u << b] & mask) & 1) << b;
            return f;
        };
        unsigned basis[5], mask[3] = {0, 0, 0};
        int rank = 0;
        big_independent(basis, rank, functional(1u));
        big_independent(basis, rank, functional(2u));
        for (int t = 0; t < 3; ++t)
            for (unsigned hm = 0; hm < (1u << (n - 5)); ++hm)
                if (big_independent(basis, rank, functional((4u << t) | (hm << 5)))) {
                    mask[t] = hm << 3;  // chunk bits
                    break;
                }
        if (rank > best) {
            best = rank;
            for (int g = 0; g < n; ++g) {
                bgx[g] = gx[g];
                bgz[g] = gz[g];
            }
            for (int t = 0; t < 3; ++t) bmask[t] = mask[t];
        }
    }
    for (int t = 0; t < 3; ++t) T.chunk_mask[t] = bmask[t];

    auto position = [&](unsigned I) {
        unsigned q = I >> 2;
        for (int t = 0; t < 3; ++t) q ^= (unsigned)(host_popc((I >> 2) & bmask[t]) & 1) << t;
        return (q << 2) | (I & 3u);
    };
    auto deposit = [&](unsigned s) {  // ext blade s (its generators in ascending order) as index bits
        unsigned I = 0;
        for (int g = 0; g < n; ++g)
            if ((ext >> g) & 1u) {
                if (s & 1u) I |= 1u << g;
                s >>= 1;
            }
        return I;
    };
    // label and sign of every base blade
    unsigned sign_of[kBig * kBig];
    for (unsigned c = 0; c < (1u << kBigBase); ++c) {
        unsigned I = 0, x = 0, z = 0, r = c;
        bool negsign = false;
        for (int g = 0; g < n; ++g)
            if ((base >> g) & 1u) {
                if (r & 1u) {
                    I |= 1u << g;
                    if (host_popc(z & bgx[g]) & 1) negsign = !negsign;
                    x ^= bgx[g];
                    z ^= bgz[g];
                }
                r >>= 1;
            }
        blade_of[x * kBig + z] = I;
        sign_of[x * kBig + z] = negsign;
        if (c == (1u << kBigBase) - 1u) {
            T.ox = x;
            T.oz = z;
        }
    }
    for (unsigned z = 0; z < 16; ++z) T.z_pos[z] = position(blade_of[z]);
    for (unsigned s = 0; s < (1u << k); ++s) T.ext_pos[s] = position(deposit(s));
    for (unsigned l = 0; l < 64; ++l) {
        const unsigned x = l & 31u, h = l >> 5;
        T.lane_pos[l] = position(blade_of[x * kBig + 16 * h]);
        for (unsigned s = 0; s < (1u << k); ++s) {
            const unsigned E = deposit(s);
            unsigned m = 0;
            for (unsigned zl = 0; zl < 16; ++zl) {
                const unsigned z = 16 * h + zl, I = blade_of[x * kBig + z];
                // e_I e_E = (-1)^{pairs (i in I, e in E), i > e} e_{I | E}
                const unsigned neg1 = (sign_of[x * kBig + z] + (unsigned)reorder_parity(I, E)) & 1u;
                m |= neg1 << zl;
                m |= ((neg1 + (unsigned)host_popc(x & z)) & 1u) << (16 + zl);
                if (position(I) != (T.lane_pos[l] ^ T.z_pos[zl])) return false;  // the labels are linear
            }
            T.sgn[s][l] = m;
        }
    }
    T.neg_pairs = T.zero_pairs = 0;
    for (unsigned s = 0; s < (1u << k); ++s)
        for (unsigned j = 0; j < (1u << k); ++j) {
            const unsigned S = deposit(s), J = deposit(j);
            if (S & J & nul) T.zero_pairs |= 1u << (4 * s + j);
            else if ((reorder_parity(S, J) + host_popc(S & J & neg)) & 1) T.neg_pairs |= 1u << (4 * s + j);
        }
    return true;
}

// Tables of the signatures in use, built once each; past the bound a table is
// built per call.
constexpr size_t kBigTables = 512;

bool big_table(int n, uint32_t neg, uint32_t nul, const BigSplit& c, Rep32Table& T) {
    static std::mutex mu;
    static std::map<unsigned long long, Rep32Table> cache;
    const unsigned long long key = ((unsigned long long)n << 48) | ((unsigned long long)nul << 24) | neg;
    {
        std::lock_guard<std::mutex> lock(mu);
        const auto it = cache.find(key);
        if (it != cache.end()) {
            T = it->second;
            return true;
        }
    }
    T = Rep32Table{};
    if (!big_table_build(n + c.d, neg | (((1u << c.dneg) - 1u) << n), nul, c.ext, T)) return false;
    if (!term_spec(n, neg, nul, T.terms)) return false;  // (ten of one square or two always hold four of one)
    std::lock_guard<std::mutex> lock(mu);
    if (cache.size() < kBigTables) cache.emplace(key, T);
    return true;
}

// One workgroup per 4 / 2^K rows (no row loop in the kernels: nothing that only
// the term sums need is held across the matrix part), at most 2^22 in a launch,
// well inside the 2^32 work-items of one launch dimension. Few rows get more
// workgroups, which share a row's term sums if it needs them and end otherwise:
// enough for two on each CU, and at most 16 lanes for a block.
// launch(r0, rows, grid, lanes of a block log2) runs for each chunk of rows.
template <class Launch>
void big_chunks(int n, int k, int64_t batch, Launch&& launch) {
    const int64_t per = 4 >> k, most = per << 22;
    for (int64_t r0 = 0; r0 < batch; r0 += most) {
        const int64_t rows = batch - r0 < most ? batch - r0 : most, groups = (rows + per - 1) / per;
        int log = 6 + k - (n - 4), more = 0;
        while (log < 4 && groups << (more + 1) <= 512) {
            ++log;
            ++more;
        }
        launch(r0, rows, dim3((unsigned)groups, 1u << more), log);
    }
}

}  // namespace

bool rep32_applicable(int op, int n, uint32_t neg, uint32_t nul) {
    BigSplit c;
    return op == CLF_OP_GEOM && big_split(n, neg, nul, c);
}

// Rows up to which the small-batch per-term kernels are faster: a row's 2^K
// waves of the 32 x 32 kernels are one dependent chain of 2^K products each,
// the per-term kernels spread it over more workgroups. Forward + backward on the
// device, us, per-term against 32 x 32, N(0, 1) rows, on both sides of each line:
// n = 9 (K = 1) 768 rows 21.6 against 22.4, 1024 rows 67 against 23 (Cl(8,0,1) 18.9
// against 21.5, 68 against 22); n = 10 (K = 1) 128 rows 16.1 against 17.5, 192 rows
// 22.1 against 17.1; n = 11, K = 1, 32 rows 17.1 against 17.8, 64 rows 28 against 18
// (Cl(10,0,1) 16.7 against 17.9, 27 against 18); n = 11, K = 2, 32 rows 17.1 against
// 22.6, 48 rows 23.9 against 22.6; n = 12, 8 rows 18.3 against 23.5, 16 rows 31
// against 24 (Cl(10,0,2) 17.4 against 23.2, 28 against 23). K = 0 has no such rows
// (n = 10, 1 row: 12.8 against 11.8).
int64_t rep32_rows(int n, uint32_t neg, uint32_t nul) {
    BigSplit c;
    if (!big_split(n, neg, nul, c) || c.k == 0) return 0;
    return n == 9 ? 768 : n == 10 ? 128 : n == 11 ? 32 : 8;
}

// M(K, D) for the (K, D) of c, one of big_split's
#define CLF_BIG_SWITCH(M)        \
    switch (4 * c.k + c.d) {     \
        case 0: M(0, 0); break;  \
        case 1: M(0, 1); break;  \
        case 4: M(1, 0); break;  \
        case 5: M(1, 1); break;  \
        case 6: M(1, 2); break;  \
        case 8: M(2, 0); break;  \
        default: M(2, 1); break; \
    }

template <int K, int D>
static void launch_rep32_fwd(int n, hipStream_t s, bool nt, const float* a, int64_t lda, const float* b, int64_t ldb,
                             float* c, int64_t batch, const Rep32Table& T) {
    big_chunks(n, K, batch, [&](int64_t r0, int64_t rows, dim3 grid, int log) {
        const int64_t off = r0 << n;
        const float *ar = a + (lda ? off : 0), *br = b + (ldb ? off : 0);
        if (nt)
            hipLaunchKernelGGL((rep32_fwd_kernel<K, D, true>), grid, dim3(256), 0, s, ar, (long long)lda, br,
                               (long long)ldb, c + off, (long long)rows, log, T);
        else
            hipLaunchKernelGGL((rep32_fwd_kernel<K, D, false>), grid, dim3(256), 0, s, ar, (long long)lda, br,
                               (long long)ldb, c + off, (long long)rows, log, T);
    });
}

int rep32_fwd(int n, uint32_t neg, uint32_t nul, const float* a, int64_t lda, const float* b, int64_t ldb, float* out,
              int64_t batch, void* stream) {
    BigSplit c;
    Rep32Table T;
    if (!big_split(n, neg, nul, c) || !big_table(n, neg, nul, c, T))
        return set_error(CLF_ERR_UNSUPPORTED, "signature has no 32 x 32 base");
    const bool nt = stream_nt(3.0 * 4.0 * (double)(1LL << n) * (double)batch);
#define CLF_BIG_FWD(K, D) \
    launch_rep32_fwd<K, D>(n, (hipStream_t)stream, nt, a, lda, b, ldb, out, batch, T)
    CLF_BIG_SWITCH(CLF_BIG_FWD)
#undef CLF_BIG_FWD
    CLF_HIP_CHECK(hipGetLastError());
    return CLF_OK;
}

template <int K, int D, bool NT>
static void launch_rep32_bwd(int n, hipStream_t s, const float* a, int64_t lda, const float* b, int64_t ldb,
                             const float* gc, int64_t ldg, float* ga, float* gb, int64_t batch,
                             const Rep32Table& T) {
    big_chunks(n, K, batch, [&](int64_t r0, int64_t rows, dim3 grid, int log) {
        const int64_t off = r0 << n;
        const float *ar = a + (lda ? off : 0), *br = b + (ldb ? off : 0), *gr = gc + (ldg ? off : 0);
        float *gar = ga ? ga + off : nullptr, *gbr = gb ? gb + off : nullptr;
#define CLF_BIG_BWD_W(WA, WB)                                                                                 \
    hipLaunchKernelGGL((rep32_bwd_kernel<K, D, NT, WA, WB>), grid, dim3(256), 0, s, ar, (long long)lda, br,    \
                       (long long)ldb, gr, (long long)ldg, gar, gbr, (long long)rows, log, T)
        if (ga && gb) CLF_BIG_BWD_W(true, true);
        else if (ga) CLF_BIG_BWD_W(true, false);
        else CLF_BIG_BWD_W(false, true);
#undef CLF_BIG_BWD_W
    });
}

int rep32_bwd(int n, uint32_t neg, uint32_t nul, const float* a, int64_t lda, const float* b, int64_t ldb,
              const float* gc, int64_t ldg, float* ga, float* gb, int64_t batch, void* stream) {
    BigSplit c;
    Rep32Table T;
    if (!big_split(n, neg, nul, c) || !big_table(n, neg, nul, c, T))
        return set_error(CLF_ERR_UNSUPPORTED, "signature has no 32 x 32 base");
    hipStream_t s = (hipStream_t)stream;
    const bool nt = stream_nt((3 + (ga != nullptr) + (gb != nullptr)) * 4.0 * (double)(1LL << n) * (double)batch);
#define CLF_BIG_BWD(K, D)                                                                          \
    do {                                                                                           \
        if (nt) launch_rep32_bwd<K, D, true>(n, s, a, lda, b, ldb, gc, ldg, ga, gb, batch, T);  \
        else launch_rep32_bwd<K, D, false>(n, s, a, lda, b, ldb, gc, ldg, ga, gb, batch, T);    \
    } while (0)
    CLF_BIG_SWITCH(CLF_BIG_BWD)
#undef CLF_BIG_BWD
#undef CLF_BIG_SWITCH
    CLF_HIP_CHECK(hipGetLastError());
    return CLF_OK;
}

}  // namespace clf
