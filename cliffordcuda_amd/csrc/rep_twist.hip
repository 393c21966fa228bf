// Geometric product at n = 8 for signatures one generator away from a real
// matrix algebra: p - q = 4, 6 (mod 8) (quaternionic type, Cl(7,1) and the
// like) and most signatures with one null generator.
//
// Let e_s be that generator and o the product of the algebra in which e_s has
// the square mu = +-1 that makes it M_16(R) (rep.hip's representation phi).
// Splitting a row by whether its blades hold e_s (a = a0 + a1),
//   a b = a0 o (b0 + b1) + a1 o (b0 + lambda b1),   lambda = e_s^2 / mu in {-1, 0},
// two 16 x 16 x 16 products a row (8192 multiply-adds against 65536 terms), and
//   ga = g0 o (b0 + lambda b1)^T + g1 o (b0 + b1)^T,
//   gb = a0^T o (g0 + g1) + a1^T o (lambda g0 + g1).
// Whether a blade holds e_s is a linear function of its label (x, z): its
// symplectic product with the label of u, the product of the other seven
// generators. The host searches generators with u = P(8, 8 d), d = 1 if
// u^2 = -1, so that the function is z3 + d x3: of a lane's 16 entries eight
// belong to part 0 and eight to part 1. With the table's entries ordered part
// 0 first, each part takes an 8-point transform V_j[c & 7], and
//   W_j[x][c] = V_j[c & 7] (-1)^{c3 z3}, z3 = d x3 (part 0) or 1 + d x3 (part 1).
// MFMA operand k of lane x is W_j[x ^ k][k]: a row shuffle of V_j[k & 7], for
// k >= 8 with the sign sigma(x) = (-1)^{d (1 + x3)} (part 0) or -sigma (part 1).
// The combinations of parts are taken before the shuffles.
//
// Layout, LDS slots and relayout as in rep.hip (four rows per wave, one group
// per wave). Rows that are not of one scale are formed term by term in the same
// launch (geom_terms.h).
//
// Bound: 3 and 5 KB a row over HBM, 1024 / 2048 matrix-core cycles and about 500 /
// 960 vector instructions per four rows (the scale test is 100 / 160 of them).
// Measured (us, forward + backward, 50001 N(0, 1) rows): Cl(7,1) 30 + 57 (28 + 52
// without the test; the per-term kernels 91 + 170), Cl(7,0,1) 31 + 53 (28 + 48;
// 78 + 150); rows that all go by their terms 146 + 232 and 119 + 190. The backward
// keeps each gradient's relayout and rows over its second operand's slot, four
// workgroups on a CU (with a slot of their own, three: 60 and 57).
#include <mutex>

#include "geom_terms.h"

namespace clf {

struct TwistTable {
    RepTable rep;   // entries of part 0, then of part 1
    float lambda;   // e_s^2 over its square in the representation
    int d;          // u^2 = -1
    int s;          // e_s
    TermSpec terms; // for the rows that are not of one scale
};

// Which of a wave's rows are not of one scale (geom_terms.h), bit j for row j.
// With e_s null the result's part without e_s is a0 b0 alone, so each part of a
// row has to hold its share of large coefficients.
__device__ __forceinline__ unsigned twist_uneven(const Pre16& p, const TwistTable& T, int lane) {
    // sums of squares, row j's total in the lanes 16j .. 16j + 15
    float q0 = sumsq4(p.v[0]), q1 = sumsq4(p.v[1]), q2 = sumsq4(p.v[2]), q3 = sumsq4(p.v[3]);
    permlane_swap32(q0, q2);
    permlane_swap32(q1, q3);
    float u = q0 + q2, v = q1 + q3;
    permlane_swap16(u, v);
    const float q = row16_sum(u + v);
    const unsigned long long ranged = __ballot(even_range(q));
    const unsigned level = __float_as_uint(even_level(q, 8));
    unsigned bad = 0;
    if (T.lambda != 0.f) {  // uniform
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (!even_count(even_large(p.v[j], __uint_as_float(__builtin_amdgcn_readlane(level, 16 * j))), 256))
                bad |= 1u << j;
    } else {
        // the lanes (s >= 2) or components that hold blades with e_s
        const unsigned long long with = T.s < 2 ? 0ull : __ballot((lane >> (T.s - 2)) & 1);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float lev = __uint_as_float(__builtin_amdgcn_readlane(level, 16 * j));
            const float c[4] = {p.v[j].x, p.v[j].y, p.v[j].z, p.v[j].w};
            int all = 0, part = 0;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const unsigned long long large = __ballot(__builtin_fabsf(c[k]) >= lev);
                all += __popcll(large);
                part += __popcll(large & (T.s >= 2 ? with : (k >> T.s) & 1 ? ~0ull : 0ull));
            }
            if (!even_count(part, 128) || !even_count(all - part, 128)) bad |= 1u << j;
        }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (!((ranged >> (16 * j)) & 1ull)) bad |= 1u << j;
    return bad;
}

// store16 for the rows that are not in `bad`
template <bool NT>
__device__ __forceinline__ void twist_store(float* __restrict__ dst, const float* __restrict__ src, long long row0,
                                            long long batch, int lane, unsigned oddc, unsigned bad) {
    float4 v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = reinterpret_cast<const float4*>(src + j * 256)[(j & 1) ? (lane ^ oddc) : lane];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if (row0 + j >= batch || ((bad >> j) & 1u)) continue;  // uniform
        float4* q = reinterpret_cast<float4*>(dst + ((row0 + j) << 8)) + lane;
        if (NT) store_stream(q, v[j]);
        else *q = v[j];
    }
}

// the rows of `bad` by their terms, a block per lane of the row's sixteen
template <int MODE>
__device__ __forceinline__ void twist_terms(const float* __restrict__ X, long long ldx, const float* __restrict__ Y,
                                            long long ldy, float* __restrict__ out, long long row0, long long batch,
                                            int lane, unsigned bad, const TermSpec& t) {
    const long long row = row0 + (lane >> 4);
    if (row >= batch || !((bad >> (lane >> 4)) & 1u)) return;
    term_block<MODE>(X + ((row & row_mask(ldx)) << 8), Y + ((row & row_mask(ldy)) << 8), out + (row << 8),
                     lane & 15u, t);
}

__device__ __forceinline__ void wht8(const float (&t)[16], int half, float (&v)[8]) {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = t[8 * half + i];
    wht_inplace<8>(v);
}

// A lane's transforms of both parts of its row's x
struct Parts {
    float v0[8], v1[8];
};

template <int SIGNSHIFT>
__device__ __forceinline__ Parts twist_convert(const float* __restrict__ row, const unsigned (&ent)[16]) {
    float t[16];
    gather16<SIGNSHIFT>(row, ent, t);
    Parts p;
    wht8(t, 0, p.v0);
    wht8(t, 1, p.v1);
    return p;
}

// operand k from the registers lo (k < 8) and hi (k >= 8, times s)
template <unsigned K>
__device__ __forceinline__ float twist_operand(const float (&lo)[8], const float (&hi)[8], float s) {
    if constexpr (K < 8u) return xor16<K>(lo[K]);
    else return s * xor16<K>(hi[K & 7u]);
}

template <unsigned... K>
__device__ __forceinline__ floatx16 twist_chain(floatx16 acc, const float (&alo)[8], const float (&ahi)[8], float as,
                                                const float (&blo)[8], const float (&bhi)[8], float bs,
                                                std::integer_sequence<unsigned, K...>) {
    ((acc = __builtin_amdgcn_mfma_f32_16x16x1f32(twist_operand<K>(alo, ahi, as), twist_operand<K>(blo, bhi, bs), acc,
                                                 0, 0, 0)),
     ...);
    return acc;
}

// X0 (a0 Y0 + a1 Y1) + X1 (b0 Y0 + b1 Y1)
__device__ __forceinline__ floatx16 twist_products(const Parts& X, const Parts& Y, float a0, float a1, float b0,
                                                   float b1, float sigma) {
    floatx16 acc = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    float lo[8], hi[8];
    constexpr auto seq = std::make_integer_sequence<unsigned, 16>{};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        lo[i] = __builtin_fmaf(a1, Y.v1[i], a0 * Y.v0[i]);
        hi[i] = __builtin_fmaf(-a1, Y.v1[i], a0 * Y.v0[i]);
    }
    acc = twist_chain(acc, X.v0, X.v0, sigma, lo, hi, sigma, seq);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        lo[i] = __builtin_fmaf(b1, Y.v1[i], b0 * Y.v0[i]);
        hi[i] = __builtin_fmaf(-b1, Y.v1[i], b0 * Y.v0[i]);
    }
    return twist_chain(acc, X.v1, X.v1, -sigma, lo, hi, sigma, seq);
}

// inverse transform of W_c[x][.] into the lane's entries (part 0 first), rho = (-1)^{d x3}
__device__ __forceinline__ void twist_unconvert(const float (&w)[16], float rho, float* __restrict__ row,
                                                const unsigned (&ent)[16]) {
    float e[8], o[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        e[i] = w[i] + w[i + 8];
        o[i] = w[i] - w[i + 8];
    }
    wht_inplace<8>(e);  // z3 = 0
    wht_inplace<8>(o);  // z3 = 1
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const bool swap = rho < 0.f;
        const float p0 = swap ? o[i] : e[i], p1 = swap ? e[i] : o[i];
        row[ent[i] & 0xffffu] = __uint_as_float(__float_as_uint(p0 * 0.0625f) ^ (ent[i] & 0x80000000u));
        row[ent[i + 8] & 0xffffu] = __uint_as_float(__float_as_uint(p1 * 0.0625f) ^ (ent[i + 8] & 0x80000000u));
    }
}

template <bool NT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void twist16_fwd_kernel(
    const float* __restrict__ A, long long lda, const float* __restrict__ B, long long ldb, float* __restrict__ C,
    long long batch, TwistTable T) {
    __shared__ float lds[4][2 * 4 * 256];  // staged a | staged b; the relayout over a and the start of b, then c over b
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const unsigned x = lane & 15u;
    const int rb = lane >> 4;
    float* sa = &lds[wave][0];
    float* sb = sa + 4 * 256;
    const unsigned oddx = (rb & 1) ? T.rep.odd_xor : 0u, oddc = T.rep.odd_xor >> 2;
    const float rho = (T.d && (x & 8u)) ? -1.f : 1.f, sigma = (T.d && !(x & 8u)) ? -1.f : 1.f;
    unsigned ent[16];
#pragma unroll
    for (int z = 0; z < 16; ++z) ent[z] = T.rep.e[x * 16 + z] ^ oddx;
    const long long row0 = ((long long)blockIdx.x * 4 + wave) * 4;
    if (row0 >= batch) return;  // whole waves; no barrier follows
    const Pre16 pa = fetch16<NT>(A, row0, batch, lane, lda);
    const Pre16 pb = fetch16<NT>(B, row0, batch, lane, ldb);
    stage16(sa, pa, lane, oddc);
    stage16(sb, pb, lane, oddc);
    wave_lds_sync();
    const Parts a = twist_convert<0>(sa + rb * 256, ent);
    const Parts b = twist_convert<1>(sb + rb * 256, ent);
    const unsigned bad = twist_uneven(pa, T, lane) | twist_uneven(pb, T, lane);
    wave_lds_sync();
    const floatx16 acc = twist_products(a, b, 1.f, 1.f, 1.f, T.lambda, sigma);
    relayout_store(sa, acc, lane);
    wave_lds_sync();
    float wc[16];
    relayout_load(sa, rb, x, wc);
    wave_lds_sync();
    twist_unconvert(wc, rho, sb + rb * 256, ent);
    wave_lds_sync();
    twist_store<NT>(C, sb, row0, batch, lane, oddc, bad);
    if (bad) twist_terms<TERM_C>(A, lda, B, ldb, C, row0, batch, lane, bad, T.terms);
}

template <bool NT, bool WA, bool WB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void twist16_bwd_kernel(
    const float* __restrict__ A, long long lda, const float* __restrict__ B, long long ldb,
    const float* __restrict__ GC, long long ldg, float* __restrict__ GA, float* __restrict__ GB, long long batch,
    TwistTable T) {
    // gc | b, over it the relayout and the rows of ga, then a and the same of gb
    __shared__ float lds[4][4 * 256 + kRelayoutFloats];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const unsigned x = lane & 15u;
    const int rb = lane >> 4;
    float* s0 = &lds[wave][0];
    float* s1 = s0 + 4 * 256;
    const unsigned oddx = (rb & 1) ? T.rep.odd_xor : 0u, oddc = T.rep.odd_xor >> 2;
    const float rho = (T.d && (x & 8u)) ? -1.f : 1.f, sigma = (T.d && !(x & 8u)) ? -1.f : 1.f;
    unsigned ent[16];
#pragma unroll
    for (int z = 0; z < 16; ++z) ent[z] = T.rep.e[x * 16 + z] ^ oddx;
    const long long row0 = ((long long)blockIdx.x * 4 + wave) * 4;
    if (row0 >= batch) return;  // whole waves; no barrier follows
    const Pre16 pg = fetch16<NT>(GC, row0, batch, lane, ldg);
    const Pre16 pb = fetch16<NT>(B, row0, batch, lane, ldb);
    stage16(s0, pg, lane, oddc);
    if (WA) stage16(s1, pb, lane, oddc);
    const Pre16 pa = fetch16<NT>(A, row0, batch, lane, lda);
    const unsigned bad_g = twist_uneven(pg, T, lane);
    const unsigned bad_a = WA ? bad_g | twist_uneven(pb, T, lane) : 0u;  // ga's rows by terms
    wave_lds_sync();
    if (WA && bad_a != 15u) {
        const Parts g = twist_convert<0>(s0 + rb * 256, ent);
        const Parts b = twist_convert<0>(s1 + rb * 256, ent);
        wave_lds_sync();
        const floatx16 acc = twist_products(g, b, 1.f, T.lambda, 1.f, 1.f, sigma);
        relayout_store(s1, acc, lane);
        wave_lds_sync();
        float w[16];
        relayout_load(s1, rb, x, w);
        wave_lds_sync();
        twist_unconvert(w, rho, s1 + rb * 256, ent);
        wave_lds_sync();
        twist_store<NT>(GA, s1, row0, batch, lane, oddc, bad_a);
    }
    const unsigned bad_b = WB ? bad_g | twist_uneven(pa, T, lane) : 0u;
    if (WB && bad_b != 15u) {
        wave_lds_sync();
        stage16(s1, pa, lane, oddc);
        wave_lds_sync();
        const Parts a = twist_convert<1>(s1 + rb * 256, ent);
        const Parts g = twist_convert<1>(s0 + rb * 256, ent);
        wave_lds_sync();
        const floatx16 acc = twist_products(a, g, 1.f, 1.f, T.lambda, 1.f, sigma);
        relayout_store(s1, acc, lane);
        wave_lds_sync();
        float w[16];
        relayout_load(s1, rb, x, w);
        wave_lds_sync();
        twist_unconvert(w, rho, s1 + rb * 256, ent);
        wave_lds_sync();
        twist_store<NT>(GB, s1, row0, batch, lane, oddc, bad_b);
    }
    if (WA && bad_a) twist_terms<TERM_GA>(B, ldb, GC, ldg, GA, row0, batch, lane, bad_a, T.terms);
    if (WB && bad_b) twist_terms<TERM_GB>(A, lda, GC, ldg, GB, row0, batch, lane, bad_b, T.terms);
}

// ---- host side --------------------------------------------------------------

namespace {

constexpr int kTwistN = 8;

// Generators of the metric (the representation's: neg over all eight) in which
// the product of all but e_s is P(8, 8 d): depth-first search over the seven
// others (they commute with u, the last one completes it), then e_s (it
// anticommutes with u).
bool twist_generators(uint32_t neg, int s, int d, unsigned* gx, unsigned* gz) {
    const unsigned ux = 8u, uz = d ? 8u : 0u;
    int order[kTwistN], cnt = 0;
    for (int g = 0; g < kTwistN; ++g)
        if (g != s) order[cnt++] = g;
    order[cnt++] = s;
    unsigned cand[kTwistN] = {0};
    int i = 0;
    while (i >= 0 && i < kTwistN) {
        const int g = order[i];
        bool found = false;
        unsigned sx = ux, sz = uz;  // what the seven still have to add up to
        for (int p = 0; p < i && p < 7; ++p) {
            sx ^= gx[order[p]];
            sz ^= gz[order[p]];
        }
        for (unsigned c = cand[i] + 1; c < 256; ++c) {
            const unsigned cx = c >> 4, cz = c & 15u;
            if (i == 6 && (cx != sx || cz != sz)) continue;
            if ((host_popc(cx & cz) & 1) != (int)((neg >> g) & 1u)) continue;
            if (((host_popc(cz & ux) + host_popc(uz & cx)) & 1) != (i == 7)) continue;
            bool ok = true;
            for (int p = 0; p < i && ok; ++p)
                ok = ((host_popc(cz & gx[order[p]]) + host_popc(gz[order[p]] & cx)) & 1) == 1;
            if (!ok) continue;
            cand[i] = c;
            gx[g] = cx;
            gz[g] = cz;
            found = true;
            break;
        }
        if (found) {
            if (++i < kTwistN) cand[i] = 0;
        } else {
            --i;
        }
    }
    return i == kTwistN;
}

// The generator to treat apart: the null one, or the first whose other square
// gives a real type. neg_rep: the representation's negative generators.
bool twist_choice(uint32_t neg, uint32_t nul, int& s, uint32_t& neg_rep, float& lambda) {
    auto real_type = [](uint32_t m) {
        const int q = host_popc(m) & 3;
        return q == 0 || q == 3;  // p - q = 8 - 2 q = 0 or 2 (mod 8)
    };
    if (host_popc(nul) > 1 || (nul == 0 && real_type(neg))) return false;
    for (s = 0; s < kTwistN; ++s) {
        if (nul && !((nul >> s) & 1u)) continue;
        for (uint32_t bit = 0; bit < 2; ++bit) {
            const uint32_t m = (neg & ~(1u << s)) | (bit << s);
            if (!real_type(m) || (!nul && m == neg)) continue;
            neg_rep = m;
            lambda = nul ? 0.f : -1.f;
            return true;
        }
    }
    return false;
}

bool twist_build(uint32_t neg, uint32_t nul, TwistTable& T) {
    int s;
    uint32_t m;
    if (!twist_choice(neg, nul, s, m, T.lambda)) return false;
    // u^2 = (-1)^{7 * 6 / 2} times the squares of the seven others
    T.d = ((21 + host_popc(m & ~(1u << s))) & 1) ? 1 : 0;
    unsigned gx[kTwistN], gz[kTwistN];
    if (!twist_generators(m, s, T.d, gx, gz)) return false;
    for (unsigned I = 0; I < 256; ++I) {
        unsigned x = 0, z = 0;
        bool negsign = false;
        for (int g = 0; g < kTwistN; ++g)
            if ((I >> g) & 1u) {
                if (host_popc(z & gx[g]) & 1) negsign = !negsign;
                x ^= gx[g];
                z ^= gz[g];
            }
        const bool tsign = negsign != ((host_popc(x & z) & 1) != 0);
        const unsigned part = (I >> s) & 1u;
        if ((((z >> 3) ^ (T.d ? x >> 3 : 0u)) & 1u) != part) return false;
        const unsigned slot = (z & 7u) | (part << 3);
        T.rep.e[x * 16 + slot] = I | (negsign ? 0x80000000u : 0u) | (tsign ? 0x40000000u : 0u);
    }
    rep16_odd_xor(T.rep);
    T.s = s;
    return term_spec(kTwistN, neg, nul, T.terms);
}

}  // namespace

// One table per (neg, null generator or none).
static bool twist_table(uint32_t neg, uint32_t nul, TwistTable& T) {
    static TableCache<TwistTable, 9 * 256> cache;
    if (neg >= 256u || nul >= 256u || host_popc(nul) > 1) return false;
    int slot = 8;
    for (int g = 0; g < kTwistN; ++g)
        if ((nul >> g) & 1u) slot = g;
    return cache.get(slot * 256 + (int)neg, T, [&](TwistTable& t) { return twist_build(neg, nul, t); });
}

bool twist_applicable(uint32_t neg, uint32_t nul) {
    TwistTable T;
    return twist_table(neg, nul, T);
}

// One workgroup per 16 rows, at most 2^22 in a launch (well inside the 2^32
// work-items of one launch dimension); launch(r0, rows, grid) for each chunk.
template <class Launch>
static void twist_chunks(int64_t batch, Launch&& launch) {
    const int64_t most = 16LL << 22;
    for (int64_t r0 = 0; r0 < batch; r0 += most) {
        const int64_t rows = batch - r0 < most ? batch - r0 : most;
        launch(r0, rows, dim3((unsigned)((rows + 15) / 16)));
    }
}

int twist_fwd(uint32_t neg, uint32_t nul, const float* a, int64_t lda, const float* b, int64_t ldb, float* c,
              int64_t batch, void* stream) {
    TwistTable T;
    if (!twist_table(neg, nul, T)) return set_error(CLF_ERR_UNSUPPORTED, "signature is not one generator from M_16(R)");
    hipStream_t s = (hipStream_t)stream;
    const bool nt = stream_nt(3.0 * 1024.0 * (double)batch);
    twist_chunks(batch, [&](int64_t r0, int64_t rows, dim3 grid) {
        const int64_t off = r0 << kTwistN;
        const float *ar = a + (lda ? off : 0), *br = b + (ldb ? off : 0);
        if (nt)
            hipLaunchKernelGGL((twist16_fwd_kernel<true>), grid, dim3(256), 0, s, ar, (long long)lda, br,
                               (long long)ldb, c + off, (long long)rows, T);
        else
            hipLaunchKernelGGL((twist16_fwd_kernel<false>), grid, dim3(256), 0, s, ar, (long long)lda, br,
                               (long long)ldb, c + off, (long long)rows, T);
    });
    CLF_HIP_CHECK(hipGetLastError());
    return CLF_OK;
}

int twist_bwd(uint32_t neg, uint32_t nul, const float* a, int64_t lda, const float* b, int64_t ldb, const float* gc,
              int64_t ldg, float* ga, float* gb, int64_t batch, void* stream) {
    TwistTable T;
    if (!twist_table(neg, nul, T)) return set_error(CLF_ERR_UNSUPPORTED, "signature is not one generator from M_16(R)");
    hipStream_t s = (hipStream_t)stream;
    const bool nt = stream_nt((3 + (ga != nullptr) + (gb != nullptr)) * 1024.0 * (double)batch);
    twist_chunks(batch, [&](int64_t r0, int64_t rows, dim3 grid) {
        const int64_t off = r0 << kTwistN;
        const float *ar = a + (lda ? off : 0), *br = b + (ldb ? off : 0), *gr = gc + (ldg ? off : 0);
        float *gar = ga ? ga + off : nullptr, *gbr = gb ? gb + off : nullptr;
#define CLF_TWIST_BWD2(NT, WA, WB)                                                                       \
    hipLaunchKernelGGL((twist16_bwd_kernel<NT, WA, WB>), grid, dim3(256), 0, s, ar, (long long)lda, br,   \
                       (long long)ldb, gr, (long long)ldg, gar, gbr, (long long)rows, T)
#define CLF_TWIST_BWD(WA, WB)                  \
    do {                                       \
        if (nt) CLF_TWIST_BWD2(true, WA, WB);  \
        else CLF_TWIST_BWD2(false, WA, WB);    \
    } while (0)
        if (ga && gb) CLF_TWIST_BWD(true, true);
        else if (ga) CLF_TWIST_BWD(true, false);
        else if (gb) CLF_TWIST_BWD(false, true);
#undef CLF_TWIST_BWD
#undef CLF_TWIST_BWD2
    });
    CLF_HIP_CHECK(hipGetLastError());
    return CLF_OK;
}

}  // namespace clf
