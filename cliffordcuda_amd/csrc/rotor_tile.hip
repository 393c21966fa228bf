// The plane-rotation chain of a rotor at n = 9 .. 12 on tiles of generators:
// y = chain(cs) x, its transpose, and the composite backward's statistics
// (rotor.hip states the maps and the statistics).
//
// A plane (p, q) mixes blades that differ in the index bits p and q. A wave
// holds 2^(RB + 6) floats (one row, or 2, 4 rows at n = 10, 9) with RB index
// bits in registers and six in the lanes, and walks a fixed sequence of
// layouts (which bits are the register bits). In each layout every plane with
// both bits in registers whose lex-earlier neighbours (planes that share a
// generator) are done runs as plain FMAs on registers: no lane exchange, and
// the only lane-dependent part is the sign of the lane bits between p and q,
// one xor per plane. Planes that share no generator commute, so this is the
// lex chain in another order; the order depends on n alone, so a row's bits do
// not depend on the batch. Between layouts the rows go through the wave's LDS
// once. The transposed map walks the same sequence backwards.
//
// Layout sequences (kTileRegs): found offline over all sequences that start
// and end with the bits of a coalesced float4 access ({0, 1} and the bits from
// 8 up), cover all planes, and keep two common register bits between
// neighbours, which makes every exchange float4: component = the two common
// bits, chunk bit i = the i-th lane bit of both layouts. A lane bit that
// changes from x to y puts y on chunk bits i and its own high bit, so the low
// chunk bits are the lane number on both sides: free of bank conflicts for
// ds_write_b128 (8 lanes) and ds_read_b128 (its 16-lane sets) alike (counted:
// none forward, 0.04 to 0.36 cycles an LDS instruction in the composite backward).
//
// Bound: at batches that fill the card the planes' arithmetic (vector issue 55 to
// 77 % of the time forward, 41 to 54 % backward) and the rows over HBM (8, with
// gradient 12 bytes a coefficient); the n = 12 backward also the spills of 106
// registers (139 MiB written for 64 MiB of rows); for a few rows the serial chain
// of one wave. Five
// register bits at n <= 11 keep that chain short (32 floats a lane) at two to
// three more exchanges than six bits would take. Measured, forward (before: one
// wave per row with lane shuffles, or rows in LDS with a barrier per plane), us:
// n = 9 64 rows 7.8 -> 6.9, 32768 rows 55 -> 29; n = 10 64 rows 14.4 -> 6.6,
// 32768 rows 129 -> 57 (4.7 TB/s); n = 11 64 rows 26.6 -> 8.1, 32768 rows
// 307 -> 131 (4.1 TB/s); n = 12 64 rows 52 -> 14, 8192 rows 289 -> 83. Composite
// backward kernel, 8192 rows: n = 9 47 -> 29, n = 10 80 -> 51, n = 11 178 -> 99,
// n = 12 (with the compile's gradient) 781 -> 295.
#include <utility>

#include "rep_common.h"

namespace clf {

constexpr int kTileMinN = 9, kTileMaxN = 12;
constexpr int kTileMaxLayouts = 11;

constexpr int tile_rb(int n) { return n == 12 ? 6 : 5; }
constexpr int tile_layouts(int n) { return n == 9 ? 8 : n == 10 ? 9 : n == 11 ? 11 : 8; }
constexpr int tile_planes(int n) { return n * (n - 1) / 2; }

constexpr unsigned tile_bits(std::initializer_list<int> b) {
    unsigned m = 0;
    for (int x : b) m |= 1u << x;
    return m;
}

// register bits of the layouts; bits n and up number the rows of a wave
constexpr unsigned kTileRegs[4][kTileMaxLayouts] = {
    {tile_bits({0, 1, 8, 9, 10}), tile_bits({0, 1, 2, 3, 4}), tile_bits({0, 1, 5, 6, 7}), tile_bits({2, 3, 4, 5, 6}),
     tile_bits({0, 1, 2, 3, 8}), tile_bits({2, 3, 4, 7, 8}), tile_bits({0, 5, 6, 7, 8}), tile_bits({0, 1, 8, 9, 10})},
    {tile_bits({0, 1, 8, 9, 10}), tile_bits({0, 1, 2, 3, 4}), tile_bits({0, 1, 2, 5, 6}), tile_bits({0, 1, 7, 8, 9}),
     tile_bits({2, 3, 7, 8, 9}), tile_bits({3, 4, 5, 6, 7}), tile_bits({3, 4, 5, 8, 9}), tile_bits({0, 6, 7, 8, 9}),
     tile_bits({0, 1, 8, 9, 10})},
    {tile_bits({0, 1, 8, 9, 10}), tile_bits({0, 1, 2, 3, 4}), tile_bits({0, 1, 2, 5, 6}), tile_bits({0, 1, 2, 7, 8}),
     tile_bits({3, 5, 6, 7, 8}), tile_bits({4, 5, 6, 7, 8}), tile_bits({0, 4, 5, 9, 10}), tile_bits({1, 2, 3, 9, 10}),
     tile_bits({4, 5, 6, 9, 10}), tile_bits({0, 7, 8, 9, 10}), tile_bits({0, 1, 8, 9, 10})},
    {tile_bits({0, 1, 8, 9, 10, 11}), tile_bits({0, 1, 2, 3, 4, 5}), tile_bits({0, 1, 2, 3, 6, 7}),
     tile_bits({0, 1, 8, 9, 10, 11}), tile_bits({2, 3, 8, 9, 10, 11}), tile_bits({4, 5, 6, 7, 8, 9}),
     tile_bits({4, 5, 6, 7, 10, 11}), tile_bits({0, 1, 8, 9, 10, 11})},
};

// What the kernels need of a sequence, derived at compile time.
struct TileSched {
    int lane[kTileMaxLayouts][6];        // index bit of lane bit i
    int reg[kTileMaxLayouts][6];         // index bits in registers, ascending
    int planes[kTileMaxLayouts][66];     // planes (lex number) run in the layout, in order
    int count[kTileMaxLayouts];
    int stats[kTileMaxLayouts][66];      // planes whose statistic is taken in the layout
    int stat_count[kTileMaxLayouts];
    int stat_last;                       // last layout with a statistic
    bool covers;                         // every plane runs once, every statistic is taken once
    bool exchanges;                      // neighbours share two register bits; only replaced lane bits differ
};

constexpr TileSched tile_sched(int n) {
    TileSched s{};
    const int rb = tile_rb(n), w = rb + 6, m = tile_layouts(n), C = tile_planes(n);
    const unsigned* regs = kTileRegs[n - kTileMinN];
    s.exchanges = true;
    for (int t = 0; t < m; ++t) {
        int k = 0;
        for (int b = 0; b < w; ++b)
            if ((regs[t] >> b) & 1u) s.reg[t][k++] = b;
        if (k != rb) s.exchanges = false;
        // a lane bit keeps its place; replaced ones take the remaining bits in ascending order
        bool used[12] = {};
        for (int i = 0; i < 6; ++i) {
            s.lane[t][i] = -1;
            const int prev = t ? s.lane[t - 1][i] : 2 + i;
            if (!((regs[t] >> prev) & 1u)) {
                s.lane[t][i] = prev;
                used[prev] = true;
            }
        }
        for (int i = 0; i < 6; ++i)
            if (s.lane[t][i] < 0)
                for (int b = 0; b < w; ++b)
                    if (!((regs[t] >> b) & 1u) && !used[b]) {
                        s.lane[t][i] = b;
                        used[b] = true;
                        break;
                    }
        if (t) {
            int common = 0;
            for (int b = 0; b < w; ++b) common += (int)((regs[t] & regs[t - 1]) >> b & 1u);
            if (common < 2) s.exchanges = false;
            for (int i = 0; i < 6; ++i)
                if (s.lane[t][i] != s.lane[t - 1][i] &&
                    (!((regs[t - 1] >> s.lane[t][i]) & 1u) || !((regs[t] >> s.lane[t - 1][i]) & 1u)))
                    s.exchanges = false;
        }
    }
    // planes in lex order per layout, each after the lex-earlier planes that share a generator
    int pp[66] = {}, pq[66] = {};
    for (int p = 0, k = 0; p < n; ++p)
        for (int q = p + 1; q < n; ++q, ++k) {
            pp[k] = p;
            pq[k] = q;
        }
    bool done[66] = {}, taken[66] = {};
    int ndone = 0, ntaken = 0;
    for (int t = 0; t < m; ++t)
        for (int k = 0; k < C; ++k) {
            if (!((regs[t] >> pp[k]) & 1u) || !((regs[t] >> pq[k]) & 1u)) continue;
            if (!taken[k]) {
                taken[k] = true;
                ++ntaken;
                s.stats[t][s.stat_count[t]++] = k;
                s.stat_last = t;
            }
            if (done[k]) continue;
            bool ok = true;
            for (int j = 0; j < k && ok; ++j)
                if ((pp[j] == pp[k] || pq[j] == pp[k] || pp[j] == pq[k] || pq[j] == pq[k]) && !done[j]) ok = false;
            if (!ok) continue;
            done[k] = true;
            ++ndone;
            s.planes[t][s.count[t]++] = k;
        }
    s.covers = ndone == C && ntaken == C;
    return s;
}

template <int N>
struct Tile {
    static constexpr int RB = tile_rb(N), W = RB + 6, V = 1 << RB, M = tile_layouts(N), C = tile_planes(N);
    static constexpr int ROWS = 1 << (W - N);  // rows of a wave
    static constexpr TileSched S = tile_sched(N);
    static_assert(S.covers && S.exchanges, "layout sequence");
    static_assert(S.lane[0][0] == 2 && S.lane[0][5] == 7, "coalesced first layout");
    static constexpr bool same_ends() {
        for (int i = 0; i < RB; ++i)
            if (S.reg[0][i] != S.reg[M - 1][i]) return false;
        return true;
    }
    static_assert(same_ends(), "coalesced last layout");
    static constexpr int plane_p(int k) {
        int p = 0;
        while (k >= N - 1 - p) k -= N - 1 - p++;
        return p;
    }
    static constexpr int plane_q(int k) {
        int p = 0;
        while (k >= N - 1 - p) k -= N - 1 - p++;
        return p + 1 + k;
    }
    // register position of index bit b in layout t
    static constexpr int reg_pos(int t, int b) {
        for (int i = 0; i < RB; ++i)
            if (S.reg[t][i] == b) return i;
        return -1;
    }
    // lane bits of layout t that lie strictly between index bits p and q
    static constexpr unsigned lane_between(int t, int p, int q) {
        unsigned m = 0;
        for (int i = 0; i < 6; ++i)
            if (S.lane[t][i] > p && S.lane[t][i] < q) m |= 1u << i;
        return m;
    }
    // register number bits of layout t whose index bits lie strictly between p and q
    static constexpr int reg_between(int t, int p, int q) {
        int m = 0;
        for (int i = 0; i < RB; ++i)
            if (S.reg[t][i] > p && S.reg[t][i] < q) m |= 1 << i;
        return m;
    }
    // Exchange from layout a to layout b (neighbours): the two common register
    // bits that are the float4 component, and the chunk column of an index bit.
    static constexpr int comp(int a, int b, int which) {
        int k = 0;
        for (int i = 0; i < RB; ++i) {
            if (reg_pos(b, S.reg[a][i]) < 0) continue;
            if (k++ == which) return S.reg[a][i];
        }
        return -1;
    }
    static constexpr unsigned chunk_col(int a, int b, int bit) {
        unsigned col = 0;
        for (int i = 0; i < 6; ++i)
            if (S.lane[a][i] == bit || S.lane[b][i] == bit) col |= 1u << i;
        int h = 6;
        for (int i = 0; i < RB; ++i) {
            const int r = S.reg[a][i];
            if (r == comp(a, b, 0) || r == comp(a, b, 1)) continue;
            if (r == bit) col |= 1u << h;
            ++h;
        }
        return col;
    }
    // chunk column of register bit i of layout t (0 for a component)
    static constexpr unsigned reg_col(int a, int b, int t, int i) {
        if (i >= RB || S.reg[t][i] == comp(a, b, 0) || S.reg[t][i] == comp(a, b, 1)) return 0;
        return chunk_col(a, b, S.reg[t][i]);
    }
    // float4 bit of lane bit i in the last layout
    static constexpr unsigned last_place(int i) { return 1u << (S.lane[M - 1][i] - 2); }
    static constexpr unsigned lane_col(int a, int b, int i) { return chunk_col(a, b, S.lane[b][i]); }
};

// xor of the columns c0 .. c5 over the bits of v
template <unsigned C0, unsigned C1, unsigned C2, unsigned C3, unsigned C4, unsigned C5>
struct Cols {
    static __device__ __forceinline__ constexpr unsigned of(unsigned v) {
        return ((v & 1u) ? C0 : 0u) ^ ((v & 2u) ? C1 : 0u) ^ ((v & 4u) ? C2 : 0u) ^ ((v & 8u) ? C3 : 0u) ^
               ((v & 16u) ? C4 : 0u) ^ ((v & 32u) ? C5 : 0u);
    }
};
template <int N, int A, int B, int T>
using RegCols = Cols<Tile<N>::reg_col(A, B, T, 0), Tile<N>::reg_col(A, B, T, 1), Tile<N>::reg_col(A, B, T, 2),
                     Tile<N>::reg_col(A, B, T, 3), Tile<N>::reg_col(A, B, T, 4), Tile<N>::reg_col(A, B, T, 5)>;
template <int N, int A, int B>
using LaneCols = Cols<Tile<N>::lane_col(A, B, 0), Tile<N>::lane_col(A, B, 1), Tile<N>::lane_col(A, B, 2),
                      Tile<N>::lane_col(A, B, 3), Tile<N>::lane_col(A, B, 4), Tile<N>::lane_col(A, B, 5)>;

// v from layout A to its neighbour B through the wave's LDS
template <int N, int A, int B>
__device__ __forceinline__ void tile_exchange(float (&v)[Tile<N>::V], float4* __restrict__ lds, unsigned lane) {
    using T = Tile<N>;
    constexpr int u = T::comp(A, B, 0), w = T::comp(A, B, 1);
    {
        constexpr int mu = 1 << T::reg_pos(A, u), mw = 1 << T::reg_pos(A, w);
#pragma unroll
        for (int r = 0; r < T::V; ++r) {
            if ((r & mu) || (r & mw)) continue;
            lds[lane ^ RegCols<N, A, B, A>::of(r)] = make_float4(v[r], v[r | mu], v[r | mw], v[r | mu | mw]);
        }
    }
    wave_lds_sync();
    {
        const unsigned base = LaneCols<N, A, B>::of(lane);
        constexpr int mu = 1 << T::reg_pos(B, u), mw = 1 << T::reg_pos(B, w);
#pragma unroll
        for (int r = 0; r < T::V; ++r) {
            if ((r & mu) || (r & mw)) continue;
            const float4 t = lds[base ^ RegCols<N, A, B, B>::of(r)];
            v[r] = t.x;
            v[r | mu] = t.y;
            v[r | mw] = t.z;
            v[r | mu | mw] = t.w;
        }
    }
    wave_lds_sync();
}

// plane K in layout T: y_I = c x_I - s sig x_J, y_J = c x_J + s sig x_I with s = -cs_s forward, +cs_s transposed
template <int N, int T, int K, bool FWD>
__device__ __forceinline__ void tile_plane(float (&v)[Tile<N>::V], const float* __restrict__ cs, unsigned lane) {
    using L = Tile<N>;
    constexpr int p = L::plane_p(K), q = L::plane_q(K);
    constexpr int mp = 1 << L::reg_pos(T, p), mq = 1 << L::reg_pos(T, q);
    constexpr int slot = L::C - 1 - K;
    constexpr unsigned between = L::lane_between(T, p, q);
    constexpr int inner = L::reg_between(T, p, q);
    const float c = cs[2 * slot];
    float s = FWD ? -cs[2 * slot + 1] : cs[2 * slot + 1];
    if constexpr (between != 0u)
        s = __uint_as_float(__float_as_uint(s) ^ ((unsigned)__popc(lane & between) << 31));
#pragma unroll
    for (int r = 0; r < L::V; ++r) {
        if (!(r & mp) || (r & mq)) continue;
        const int j = r ^ mp ^ mq;
        const float sg = (__builtin_popcount(r & inner) & 1) ? -s : s;
        const float xi = v[r], xj = v[j];
        v[r] = __builtin_fmaf(c, xi, -sg * xj);
        v[j] = __builtin_fmaf(c, xj, sg * xi);
    }
}

template <int N, int T, bool FWD, int... Is>
__device__ __forceinline__ void tile_planes_seq(float (&v)[Tile<N>::V], const float* __restrict__ cs, unsigned lane,
                                                std::integer_sequence<int, Is...>) {
    constexpr int cnt = Tile<N>::S.count[T];
    (tile_plane<N, T, Tile<N>::S.planes[T][FWD ? Is : cnt - 1 - Is], FWD>(v, cs, lane), ...);
}

template <int N, int T, bool FWD>
__device__ __forceinline__ void tile_layout(float (&v)[Tile<N>::V], const float* __restrict__ cs, unsigned lane) {
    tile_planes_seq<N, T, FWD>(v, cs, lane, std::make_integer_sequence<int, Tile<N>::S.count[T]>{});
}

// the whole chain, from the coalesced layout to the coalesced layout
template <int N, bool FWD, int... Ts>
__device__ __forceinline__ void tile_chain_seq(float (&v)[Tile<N>::V], const float* __restrict__ cs,
                                               float4* __restrict__ lds, unsigned lane,
                                               std::integer_sequence<int, Ts...>) {
    constexpr int last = Tile<N>::M - 1;
    tile_layout<N, FWD ? 0 : last, FWD>(v, cs, lane);
    ((tile_exchange<N, FWD ? Ts : last - Ts, FWD ? Ts + 1 : last - Ts - 1>(v, lds, lane),
      tile_layout<N, FWD ? Ts + 1 : last - Ts - 1, FWD>(v, cs, lane)),
     ...);
}

template <int N, bool FWD>
__device__ __forceinline__ void tile_chain(float (&v)[Tile<N>::V], const float* __restrict__ cs,
                                           float4* __restrict__ lds, unsigned lane) {
    tile_chain_seq<N, FWD>(v, cs, lds, lane, std::make_integer_sequence<int, Tile<N>::M - 1>{});
}

// The lane's place among the 64 float4 of an access: the lane bits of the first
// and of the last layout are the same index bits, in another order.
template <int N, bool FIRST>
__device__ __forceinline__ unsigned tile_place(unsigned lane) {
    if constexpr (FIRST) return lane;
    return Cols<Tile<N>::last_place(0), Tile<N>::last_place(1), Tile<N>::last_place(2), Tile<N>::last_place(3),
                Tile<N>::last_place(4), Tile<N>::last_place(5)>::of(lane);
}

// The wave's rows in a coalesced layout: registers 4j .. 4j + 3 hold floats
// 256 j + 4 lane .. + 3 of the wave's consecutive rows (lane: tile_place). ld: floats between
// rows (2^N, or 0: one row for all). Rows past the end read the last row, or
// zeros (ZERO).
template <int N, bool NT, bool ZERO>
__device__ __forceinline__ void tile_load(float (&v)[Tile<N>::V], const float* __restrict__ src, long long row0,
                                          long long batch, long long ld, unsigned lane) {
    constexpr int PER = 1 << (N - 8);  // float4 groups per row
#pragma unroll
    for (int j = 0; j < Tile<N>::V / 4; ++j) {
        const long long row = row0 + j / PER;
        const float4* p =
            reinterpret_cast<const float4*>(src + (row < batch ? row : batch - 1) * ld + 256 * (j % PER)) + lane;
        float4 t = NT ? load_stream(p) : *p;
        if (ZERO && row >= batch) t = make_float4(0.f, 0.f, 0.f, 0.f);
        v[4 * j] = t.x;
        v[4 * j + 1] = t.y;
        v[4 * j + 2] = t.z;
        v[4 * j + 3] = t.w;
    }
}

template <int N, bool NT>
__device__ __forceinline__ void tile_store(const float (&v)[Tile<N>::V], float* __restrict__ dst, long long row0,
                                           long long batch, unsigned lane) {
    constexpr int PER = 1 << (N - 8);
#pragma unroll
    for (int j = 0; j < Tile<N>::V / 4; ++j) {
        const long long row = row0 + j / PER;
        if (row >= batch) continue;  // uniform
        float4* p = reinterpret_cast<float4*>(dst + (row << N) + 256 * (j % PER)) + lane;
        const float4 t = make_float4(v[4 * j], v[4 * j + 1], v[4 * j + 2], v[4 * j + 3]);
        if (NT) store_stream(p, t);
        else *p = t;
    }
}

template <int N, bool FWD, bool NT>
__global__ __launch_bounds__(256) void rotor_tile_kernel(const float* __restrict__ cs, const float* __restrict__ X,
                                                         float* __restrict__ Y, long long batch, long long ldx) {
    using L = Tile<N>;
    __shared__ float4 lds[4][(1 << L::W) / 4];
    const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63u;
    const long long row0 = ((long long)blockIdx.x * 4 + wave) * L::ROWS;
    if (row0 >= batch) return;  // whole waves; no barrier follows
    float v[L::V];
    tile_load<N, NT, false>(v, X, row0, batch, ldx, tile_place<N, FWD>(lane));
    tile_chain<N, FWD>(v, cs, lds[wave], lane);
    tile_store<N, NT>(v, Y, row0, batch, tile_place<N, !FWD>(lane));
}

// ---- the composite backward: gx and the statistics -------------------------

// acc[k] += sum over the lane's pairs of sig (x_J g_I - x_I g_J), the lane
// bits' part of sig left to the end
template <int N, int T, int K>
__device__ __forceinline__ void tile_stat(float* __restrict__ acc, const float (&x)[Tile<N>::V],
                                          const float (&g)[Tile<N>::V]) {
    using L = Tile<N>;
    constexpr int p = L::plane_p(K), q = L::plane_q(K);
    constexpr int mp = 1 << L::reg_pos(T, p), mq = 1 << L::reg_pos(T, q);
    constexpr int inner = L::reg_between(T, p, q);
#pragma unroll
    for (int r = 0; r < L::V; ++r) {
        if (!(r & mp) || (r & mq)) continue;
        const int j = r ^ mp ^ mq;
        const bool neg = (__builtin_popcount(r & inner) & 1) != 0;
        acc[K] = __builtin_fmaf(neg ? -x[j] : x[j], g[r], acc[K]);
        acc[K] = __builtin_fmaf(neg ? x[r] : -x[r], g[j], acc[K]);
    }
}

template <int N, int T, int... Is>
__device__ __forceinline__ void tile_stats_seq(float* __restrict__ acc, const float (&x)[Tile<N>::V],
                                               const float (&g)[Tile<N>::V], std::integer_sequence<int, Is...>) {
    (tile_stat<N, T, Tile<N>::S.stats[T][Is]>(acc, x, g), ...);
}

template <int N, int... Ts>
__device__ __forceinline__ void tile_all_stats(float* __restrict__ acc, float (&x)[Tile<N>::V],
                                               float (&g)[Tile<N>::V], float4* __restrict__ lds, unsigned lane,
                                               std::integer_sequence<int, Ts...>) {
    using L = Tile<N>;
    tile_stats_seq<N, 0>(acc, x, g, std::make_integer_sequence<int, L::S.stat_count[0]>{});
    ((tile_exchange<N, Ts, Ts + 1>(x, lds, lane), tile_exchange<N, Ts, Ts + 1>(g, lds, lane),
      tile_stats_seq<N, Ts + 1>(acc, x, g, std::make_integer_sequence<int, L::S.stat_count[Ts + 1]>{})),
     ...);
}

template <int N, int T, int K>
__device__ __forceinline__ void tile_stat_sign(float* __restrict__ acc, unsigned lane) {
    constexpr unsigned between = Tile<N>::lane_between(T, Tile<N>::plane_p(K), Tile<N>::plane_q(K));
    acc[K] = __uint_as_float(__float_as_uint(acc[K]) ^ ((unsigned)__popc(lane & between) << 31));
}

template <int N, int T, int... Is>
__device__ __forceinline__ void tile_stat_signs(float* __restrict__ acc, unsigned lane,
                                                std::integer_sequence<int, Is...>) {
    (tile_stat_sign<N, T, Tile<N>::S.stats[T][Is]>(acc, lane), ...);
}

template <int N, int... Ts>
__device__ __forceinline__ void tile_all_signs(float* __restrict__ acc, unsigned lane,
                                               std::integer_sequence<int, Ts...>) {
    (tile_stat_signs<N, Ts>(acc, lane, std::make_integer_sequence<int, Tile<N>::S.stat_count[Ts]>{}), ...);
}

// Waves walk row groups with a grid stride; parts[blockIdx.x * C + k] is the
// workgroup's sum of plane k's statistic.
template <int N, bool NT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void rotor_tile_bwd_kernel(
    const float* __restrict__ cs, const float* __restrict__ X, const float* __restrict__ GY, float* __restrict__ GX,
    float* __restrict__ parts, long long batch, long long ldg) {
    using L = Tile<N>;
    __shared__ float4 lds[4][(1 << L::W) / 4];
    __shared__ float red[4][L::C];
    const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63u;
    float acc[L::C];
#pragma unroll
    for (int k = 0; k < L::C; ++k) acc[k] = 0.f;
    const long long stride = (long long)gridDim.x * 4 * L::ROWS;
    for (long long row0 = ((long long)blockIdx.x * 4 + wave) * L::ROWS; row0 < batch; row0 += stride) {
        // an opaque copy keeps lane-dependent values inside the loop instead of in registers across it
        unsigned ln = lane;
        asm volatile("" : "+v"(ln));
        float g[L::V], x[L::V];
        tile_load<N, NT, false>(g, GY, row0, batch, ldg, tile_place<N, false>(ln));
        // x is requested before the chain where the registers allow it
        if (N < 12) tile_load<N, NT, true>(x, X, row0, batch, 1LL << N, ln);
        tile_chain<N, false>(g, cs, lds[wave], ln);
        if (N == 12) tile_load<N, NT, true>(x, X, row0, batch, 1LL << N, ln);
        if (GX) tile_store<N, NT>(g, GX, row0, batch, ln);
        tile_all_stats<N>(acc, x, g, lds[wave], ln, std::make_integer_sequence<int, L::S.stat_last>{});
    }
    tile_all_signs<N>(acc, lane, std::make_integer_sequence<int, L::M>{});
#pragma unroll
    for (int k = 0; k < L::C; ++k) {
        float t = acc[k];
        for (int off = 1; off < 64; off <<= 1) t += __shfl_xor(t, off, 64);
        if (lane == 0) red[wave][k] = t;
    }
    __syncthreads();
    for (int k = threadIdx.x; k < L::C; k += 256)
        parts[(long long)blockIdx.x * L::C + k] = (red[0][k] + red[1][k]) + (red[2][k] + red[3][k]);
}

// ---- host side --------------------------------------------------------------

bool rotor_tile_serves(int n) { return n >= kTileMinN && n <= kTileMaxN; }

template <int N>
static int tile_groups_per_block() { return 4 * Tile<N>::ROWS; }

// rows that a workgroup takes at a time
int rotor_tile_rows(int n) {
    switch (n) {
        case 9: return tile_groups_per_block<9>();
        case 10: return tile_groups_per_block<10>();
        case 11: return tile_groups_per_block<11>();
        default: return tile_groups_per_block<12>();
    }
}

template <int N>
static void launch_tile(bool fwd, const float* cs, const float* x, float* y, int64_t batch, hipStream_t s,
                        long long ldx) {
    const long long per = tile_groups_per_block<N>();
    const long long most = (1LL << 22) * per;  // rows of one launch, well inside its 2^32 work-items
    const bool nt = stream_nt(2.0 * 4.0 * (double)(1LL << N) * (double)batch);
    for (long long r0 = 0; r0 < batch; r0 += most) {
        const long long rows = batch - r0 < most ? batch - r0 : most;
        const dim3 grid((unsigned)((rows + per - 1) / per));
        const float* xs = x + r0 * ldx;
        float* ys = y + (r0 << N);
#define CLF_TILE(FWD, NT) \
    hipLaunchKernelGGL((rotor_tile_kernel<N, FWD, NT>), grid, dim3(256), 0, s, cs, xs, ys, rows, ldx)
        if (fwd && nt) CLF_TILE(true, true);
        else if (fwd) CLF_TILE(true, false);
        else if (nt) CLF_TILE(false, true);
        else CLF_TILE(false, false);
#undef CLF_TILE
    }
}

void rotor_tile_apply(int n, bool fwd, const float* cs, const float* x, float* y, int64_t batch, void* stream,
                      long long ldx) {
    hipStream_t s = (hipStream_t)stream;
    switch (n) {
        case 9: launch_tile<9>(fwd, cs, x, y, batch, s, ldx); break;
        case 10: launch_tile<10>(fwd, cs, x, y, batch, s, ldx); break;
        case 11: launch_tile<11>(fwd, cs, x, y, batch, s, ldx); break;
        default: launch_tile<12>(fwd, cs, x, y, batch, s, ldx); break;
    }
}

template <int N>
static int launch_tile_bwd(const float* cs, const float* x, const float* gy, long long ldg, float* gx, float* parts,
                           int64_t batch, int wanted, hipStream_t s) {
    const bool nt = stream_nt((gx ? 3.0 : 2.0) * 4.0 * (double)(1LL << N) * (double)batch);
    const void* kernel = nt ? (const void*)rotor_tile_bwd_kernel<N, true> : (const void*)rotor_tile_bwd_kernel<N, false>;
    const unsigned grid = resident_grid(kernel, 256, 0, wanted);
    if (nt)
        hipLaunchKernelGGL((rotor_tile_bwd_kernel<N, true>), dim3(grid), dim3(256), 0, s, cs, x, gy, gx, parts,
                           (long long)batch, ldg);
    else
        hipLaunchKernelGGL((rotor_tile_bwd_kernel<N, false>), dim3(grid), dim3(256), 0, s, cs, x, gy, gx, parts,
                           (long long)batch, ldg);
    return (int)grid;
}

// Composite backward; at most `wanted` workgroups, returns the partials written.
int rotor_tile_bwd(int n, const float* cs, const float* x, const float* gy, long long ldg, float* gx, float* parts,
                   int64_t batch, int wanted, void* stream) {
    hipStream_t s = (hipStream_t)stream;
    switch (n) {
        case 9: return launch_tile_bwd<9>(cs, x, gy, ldg, gx, parts, batch, wanted, s);
        case 10: return launch_tile_bwd<10>(cs, x, gy, ldg, gx, parts, batch, wanted, s);
        case 11: return launch_tile_bwd<11>(cs, x, gy, ldg, gx, parts, batch, wanted, s);
        default: return launch_tile_bwd<12>(cs, x, gy, ldg, gx, parts, batch, wanted, s);
    }
}

}  // namespace clf
