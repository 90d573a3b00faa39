// A short row's products held in registers (gfx950, wave64): the expansion of
// the row's A entries into products and the ranks of their columns among the
// row's outputs, shared by the row path's symbolic and numeric kernels.
#pragma once

#include "tsg_device.h"

// One group of G lanes owns one row of at most P = G * U products, product
// q = u * G + lane in register u of the lane.  Nothing is visited twice: the
// columns are gathered once and every later step works on registers and LDS.
// A row takes NB <= U registers a lane (a few sizes, each compiled without a
// test per register); lanes past the row's last product repeat it, so only
// the sums are masked.
//
//   entries  the row's A entries with products, compacted: off[i] such that
//            off[i] + q is the position in B of product q of entry i (and the
//            entry's value); and a bit per product, set where an entry's
//            products start.  Product q then belongs to entry (bits at or
//            below q) - 1: one count instead of a search or a running
//            maximum.
//   ranks    by a bitmap of two levels, so that its space depends on the
//            products and not on the columns' span: a bit per 16 columns over
//            a span of up to LW * 512 columns, numbered in order; then the
//            row's own 16-column words, one per level-1 bit set, their bits
//            and the outputs before them in one int.  In a wider span the
//            16-column words are first numbered in blocks of 2^s of them, as
//            many as level 1 has bits for, and the empty blocks between them
//            left out, which divides the span by LW * 32 / P or more; once for
//            2^20 columns, four times for 2^31.
//
// LDS: the steps after the entries reuse the same space one after the other.
// E bounds the entries with products; VALS: their values are kept too; ACC:
// outputs summed at a time.
template <int P, int E, int LW, int ACC>
struct FlatSmem {
    union {
        uint2 l1[LW];             // {bits, bits set before}
        unsigned l2[P];           // bits | outputs before << 16
        int cols[P];
        double acc[ACC];
    };
    double a[ACC > 1 ? E : 1];
    int off[E];
    unsigned starts[P / 32];
};

// A value that every lane of a group holds: a scalar when the group is the
// wave (branches on it then cost no lane masks).
template <int G>
__device__ __forceinline__ int group_uniform(int x) {
    if constexpr (G == 64) return __builtin_amdgcn_readfirstlane(x);
    else return x;
}

template <int G>
__device__ __forceinline__ unsigned long long group_ballot(bool x) {
    if constexpr (G == 64) return __ballot(x);
    else return (__ballot(x) >> (__lane_id() & ~(G - 1))) & ((1ull << G) - 1);
}

template <int G>
__device__ __forceinline__ int group_min_i32(int x) {
#pragma unroll
    for (int d = G / 2; d > 0; d >>= 1) x = min(x, __shfl_xor(x, d, G));
    return x;
}
template <int G>
__device__ __forceinline__ int group_max_i32(int x) {
#pragma unroll
    for (int d = G / 2; d > 0; d >>= 1) x = max(x, __shfl_xor(x, d, G));
    return x;
}

// The entries step: A entries [pa, pe) of a row of at most P products and at
// most E entries with products (with aval, their values too).  Returns the
// row's products.
template <int G, int P, int E, int LW, int ACC>
__device__ __forceinline__ int flat_entries(FlatSmem<P, E, LW, ACC> &S, int pa, int pe,
                                            const int *__restrict__ ja,
                                            const double *__restrict__ aval,
                                            const int *__restrict__ ib) {
    const int l = __lane_id() & (G - 1);
    const unsigned long long below = (1ull << l) - 1;
    for (int i = l; i < P / 32; i += G) S.starts[i] = 0u;
    wave_lds_fence();
    int nprod = 0, nent = 0;
    // (unsigned: g passes 2^31 at the end of 2^31 - 1 entries)
    for (unsigned g = (unsigned)pa; g < (unsigned)pe; g += G) {
        const unsigned p = g + (unsigned)l;
        int cnt = 0, lo = 0;
        double av = 0.0;
        if (p < (unsigned)pe) {
            const int t = ja[p];
            if (ACC > 1) av = aval[p];
            lo = ib[t];
            cnt = max(ib[t + 1] - lo, 0);
        }
        const int incl = group_incl_scan<G>(cnt);
        const int start = nprod + incl - cnt;
        const unsigned long long some = group_ballot<G>(cnt > 0);
        const int i = nent + __popcll(some & below);
        if (cnt > 0 && start < P && i < E) {
            S.off[i] = lo - start;
            if (ACC > 1) S.a[i] = av;
            atomicOr(&S.starts[start >> 5], 1u << (start & 31));
        }
        nprod += group_last<G>(incl);
        nent += __popcll(some);
    }
    wave_lds_fence();
    // a row that is not what it was in the symbolic phase: only products of
    // the entries kept
    if (nent > E) nprod = min(nprod, E);
    return group_uniform<G>(min(nprod, P));
}

// The start bits of a row, kept in a register (G == 64: two lanes hold a
// batch's 64 bits, read as scalars) or read from LDS.
template <int G, int U>
struct FlatHeads {
    const unsigned *starts;
    int sv = 0;
    __device__ __forceinline__ explicit FlatHeads(const unsigned *s) : starts(s) {
        if constexpr (G == 64) sv = (int)starts[min((int)__lane_id(), 2 * U - 1)];
        static_assert(G == 64 || G == 16, "a batch is two words or half a word of start bits");
    }
    // (u past the row's batches: none)
    // bits of batch u where an entry's products start
    __device__ __forceinline__ unsigned long long operator()(int u) const {
        if constexpr (G == 64)
            return ((unsigned long long)(unsigned)__builtin_amdgcn_readlane(sv, 2 * u + 1) << 32) |
                   (unsigned)__builtin_amdgcn_readlane(sv, 2 * u);
        else
            return (starts[u >> 1] >> (16 * (u & 1))) & 0xffffu;
    }
    // base + the bits of m at or below the lane
    __device__ __forceinline__ static int at(unsigned long long m, int base) {
        if constexpr (G == 64) {
            // the bits of m >> 1 below the lane, and bit 0
            const unsigned long long m1 = m >> 1;
            return (int)__builtin_amdgcn_mbcnt_hi(
                (unsigned)(m1 >> 32),
                __builtin_amdgcn_mbcnt_lo((unsigned)m1, (unsigned)(base + (int)(m & 1))));
        } else {
            return base + __popc((unsigned)m & ((2u << (__lane_id() & (G - 1))) - 1u));
        }
    }
};

// Ranks of the products' columns among the row's distinct columns (RANKS), or
// their number alone; returns that number.  repeats: many products share a
// column, so a bit is looked at before it is set (atomics of a wave on one
// word queue up).
template <int G, int NB, bool RANKS, int P, int E, int LW, int ACC>
__device__ __forceinline__ int flat_ranks(FlatSmem<P, E, LW, ACC> &S, const int (&col)[NB],
                                          int (&rank)[NB], bool repeats) {
    const int l = __lane_id() & (G - 1);
    int lo = 0x7fffffff, hi = -1;
#pragma unroll
    for (int u = 0; u < NB; u++) {
        lo = min(lo, col[u]);
        hi = max(hi, col[u]);
    }
    lo = group_uniform<G>(group_min_i32<G>(lo)) & ~15;   // a 16-column word's first
    hi = group_uniform<G>(group_max_i32<G>(hi));
    if constexpr (!RANKS) {
        // counted alone, columns of a span that fits need one level of bits
        if (hi - lo < LW * 64) {
            unsigned *bits = reinterpret_cast<unsigned *>(S.l1);
            uint4 *bits4 = reinterpret_cast<uint4 *>(S.l1);
            const int n4 = ((hi - lo) >> 7) + 1;
            for (int i = l; i < n4; i += G) bits4[i] = make_uint4(0u, 0u, 0u, 0u);
            wave_lds_fence();
#pragma unroll
            for (int u = 0; u < NB; u++) {
                const int cc = col[u] - lo;
                lds_set_bit(&bits[cc >> 5], 1u << (cc & 31));
            }
            wave_lds_fence();
            int n = 0;
            for (int i = l; i < n4; i += G) {
                const uint4 v = bits4[i];
                n += __popc(v.x) + __popc(v.y) + __popc(v.z) + __popc(v.w);
            }
            return group_sum<G>(n);
        }
    }
    auto each = [&](auto f) {
#pragma unroll
        for (int u = 0; u < NB; u++) f(u);
    };
    auto set_all = [&](auto word, auto bit) {
        if (repeats)
            each([&](int u) { lds_set_bit(word(u), bit(u)); });
        else
            each([&](int u) { atomicOr(word(u), bit(u)); });
    };
    // The places at(u), at most top < 32 * LW, numbered in order by level 1's
    // bits; between(u), then put(u, number of the place).  Returns their number.
    auto number = [&](int top, auto at, auto between, auto put) {
        const int n1 = (top >> 5) + 1;
        for (int i = l; i < n1; i += G) S.l1[i] = make_uint2(0u, 0u);
        wave_lds_fence();
        set_all([&](int u) { return &S.l1[at(u) >> 5].x; },
                [&](int u) { return 1u << (at(u) & 31); });
        wave_lds_fence();
        int n = 0;
        for (int i0 = 0; i0 < n1; i0 += G) {
            const int i = i0 + l;
            const int pc = i < n1 ? __popc(S.l1[i].x) : 0;
            const int incl = group_incl_scan<G>(pc);
            if (i < n1) S.l1[i].y = (unsigned)(n + incl - pc);
            n += group_last<G>(incl);
        }
        wave_lds_fence();
        each(between);
        each([&](int u) {
            const uint2 v = S.l1[at(u) >> 5];
            put(u, (int)v.y + __popc(v.x & ((1u << (at(u) & 31)) - 1u)));
        });
        wave_lds_fence();
        return n;
    };
    // rank holds the number of the product's 16-column word until the column's
    // rank replaces it
    constexpr int LOG = 31 - __builtin_clz(LW * 32);
    static_assert(LW * 32 == 1 << LOG && LW * 32 >= 4 * P, "numbering blocks shortens the span");
    auto word = [&](int u) { return (col[u] - lo) >> 4; };
    int top = (hi - lo) >> 4, n2;
    if (top < LW * 32) {
        n2 = number(top, word, [](int) {}, [&](int u, int v) { rank[u] = v; });
    } else {
        // 32768 rows of 900 products, both phases: 0.46 ms over 2^24 columns,
        // 0.54 over 2^30 (0.35 within the span); a span's worth of level 1
        // after the other took 3.5 and 30
        each([&](int u) { rank[u] = word(u); });
        int s;
        do {
            s = max(32 - __builtin_clz(top | 1) - LOG, 0);
            n2 = number(
                top >> s, [&](int u) { return rank[u] >> s; },
                [&](int u) {
                    // places are made again after the scan: kept over it they
                    // cost the kernel a wave per SIMD (134 registers, not 108)
                    int x = rank[u];
                    asm volatile("" : "+v"(x));
                    rank[u] = x;
                },
                [&](int u, int v) { rank[u] = (v << s) | (rank[u] & ((1 << s) - 1)); });
            top = (n2 << s) - 1;
        } while (s > 0);
    }
    for (int i = l; i < n2; i += G) S.l2[i] = 0u;
    wave_lds_fence();
    auto in_word = [&](int u) { return col[u] & 15; };
    set_all([&](int u) { return &S.l2[rank[u]]; }, [&](int u) { return 1u << in_word(u); });
    wave_lds_fence();
    int n = 0;
    if constexpr (RANKS) {
        for (int i0 = 0; i0 < n2; i0 += G) {
            const int i = i0 + l;
            const unsigned v = i < n2 ? S.l2[i] : 0u;
            const int pc = __popc(v);
            const int incl = group_incl_scan<G>(pc);
            if (i < n2) S.l2[i] = v | ((unsigned)(n + incl - pc) << 16);
            n += group_last<G>(incl);
        }
        wave_lds_fence();
        each([&](int u) {
            const unsigned v = S.l2[rank[u]];
            rank[u] = (int)(v >> 16) + __popc(v & ((1u << in_word(u)) - 1u));
        });
        wave_lds_fence();
        return n;
    } else {
        for (int i = l; i < n2; i += G) n += __popc(S.l2[i]);
        return group_sum<G>(n);
    }
}
