// Flat product expansion, LDS hash tables and ordered accumulation shared by
// the row path and the tile path (gfx950, wave64).
#pragma once

#include "tsg_device.h"

// ------------------------------------------------- flat product expansion
// B block pointers: entry (row t, block b) = first position of B row t with
// column >= b << bs, at p[t*tstride + b*bstride].  Row-major (tstride =
// blocks+1, bstride = 1) keeps a row's entries together; block-major
// (tstride = 1, bstride = rows of B) keeps a block's entries for all rows
// together, which suits work that runs in column order: it looks up a few
// blocks at a time, whose entries stay in L2.
struct BlockPtrs {
    const int *p = nullptr;
    int64_t tstride = 0, bstride = 0;
    int bs = 0;
};

// Range of B row t restricted to columns >= c, through the block pointers
// (a binary search inside the block when c is not a block boundary).
__device__ __forceinline__ int brange_lo(const BlockPtrs &bp, const int *__restrict__ jb, int t,
                                         int c) {
    const int b = c >> bp.bs;
    const int64_t e = (int64_t)t * bp.tstride + (int64_t)b * bp.bstride;
    int lo = bp.p[e];
    if (c & ((1 << bp.bs) - 1)) {
        int hi = bp.p[e + bp.bstride];
        lo = lower_bound_i32(jb, lo, hi, c);
    }
    return lo;
}

// A batch of 64 products seen by the functions below: act marks the lanes
// that hold a product; seg is the lane's A entry among the batch's (from 1)
// and nseg their number (uniform); products of one A entry are one B row's:
// distinct columns whenever B's rows are duplicate-free.
struct Batch {
    bool act;
    int col;
    double a, b;
    int seg, nseg;
};

// Products of one group of 64 A entries: lane l's A entry contributes the B
// positions [lo, lo + cnt) with value a.  Batches of 64 products are handed
// to f in product order (see for_products).
//
// A product finds its A entry by counting: the entries with products move to
// the front lanes (a permutation, once per group), a bit is set in LDS (heads:
// 64 ints, any content) where each one's products start, and product q
// belongs to entry (bits at or below q) - 1.  A batch's 64 bits are a scalar,
// so the count is two instructions, against a running maximum over marks
// written per batch (an LDS round trip and six steps): R-MAT 2^18, items of
// more than 512 outputs, 1.19 -> 0.96 ms; R-MAT 2^20 with 8 draws a row, 21.6
// -> 20.7 ms, and its symbolic bands 14.1 -> 13.3 ms.
// PACKED: B's entries are also given as 16-byte {column, -, value} records
// (bpk), so a product's column and value come from one load and, for a short
// range, one cache line.
template <int U, bool VALUES, bool PACKED = false, class F>
__device__ __forceinline__ void expand_group(int lo, int cnt, double a,
                                             const int *__restrict__ jb,
                                             const double *__restrict__ bval, int *heads, F &&f,
                                             const int4 *__restrict__ bpk = nullptr) {
    static_assert(2 * U <= 64, "a round's start bits are a word a lane");
    const int l = __lane_id();
    const int incl = wave_incl_scan(cnt);
    const int total = __builtin_amdgcn_readlane(incl, 63);
    if (total <= 0) return;
    const int start = incl - cnt;
    const unsigned long long some = __ballot(cnt > 0);
    int off;                           // of the l-th entry with products
    double av = 0.0;
    {
        const unsigned long long below = (1ull << l) - 1;
        const int to = 4 * (cnt > 0 ? __popcll(some & below)
                                    : __popcll(some) + __popcll(~some & below));
        off = __builtin_amdgcn_ds_permute(to, lo - start);
        if (VALUES)
            av = __hiloint2double(__builtin_amdgcn_ds_permute(to, __double2hiint(a)),
                                  __builtin_amdgcn_ds_permute(to, __double2loint(a)));
    }
    for (int base = 0; base < total; base += 64 * U) {
        wave_lds_fence();
        if (l < 2 * U) heads[l] = 0;
        wave_lds_fence();
        const int at = start - base;
        if (cnt > 0 && at >= 0 && at < 64 * U)
            atomicOr(reinterpret_cast<unsigned *>(heads) + (at >> 5), 1u << (at & 31));
        wave_lds_fence();
        const int hv = l < 2 * U ? heads[l] : 0;
        // entries that start before the batch, less one
        int before = __popcll(__ballot(cnt > 0 && at < 0)) - 1;
        int e[U], sl[U], seg[U], nseg[U];
        bool act[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const unsigned long long m =
                ((unsigned long long)(unsigned)__builtin_amdgcn_readlane(hv, 2 * u + 1) << 32) |
                (unsigned)__builtin_amdgcn_readlane(hv, 2 * u);
            const int q = base + 64 * u + l;
            // bits at or below the lane: those of m >> 1 below it, bit 0
            const unsigned long long m1 = m >> 1;
            const int first = before + (int)(m & 1);
            sl[u] = (int)__builtin_amdgcn_mbcnt_hi(
                (unsigned)(m1 >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m1, (unsigned)first));
            seg[u] = sl[u] - first + 1;
            nseg[u] = __popcll(m | 1ull);
            act[u] = q < total;
            e[u] = __shfl(off, sl[u], 64) + q;
            before += __popcll(m);
        }
        int col[U];
        double bv[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (PACKED) {
                const int4 rec = act[u] ? bpk[e[u]] : make_int4(0, 0, 0, 0);
                col[u] = rec.x;
                bv[u] = __hiloint2double(rec.w, rec.z);
            } else {
                col[u] = act[u] ? jb[e[u]] : 0;
                bv[u] = (VALUES && act[u]) ? bval[e[u]] : 0.0;
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (base + 64 * u < total) {
                const double as = VALUES ? __shfl(av, sl[u], 64) : 0.0;
                f(Batch{act[u], col[u], as, bv[u], seg[u], nseg[u]});
            }
        }
    }
}

// Visits the products of the A entries [pa, pe) of one row in A-row order, a
// wave's 64 entries at a time, optionally restricted to B columns [c0, c1).
// f(batch) is called once per batch by every lane; batches are issued in
// product order and lane order inside a batch is product order.  U batches
// are gathered before the first is handed to f, so each lane keeps U
// independent loads in flight.  With PARTS > 1 only the A entries part,
// part + PARTS, ... are visited, so several waves can share a row where the
// order of products does not matter (entries, not batches of one group: what
// a group costs before its first product is then spent once, and alternate
// entries, because a row's first ones may name the longest B rows).  heads:
// 64 ints of LDS.
template <int U, int PARTS, bool RANGED, bool VALUES, class F>
__device__ __forceinline__ void for_products(int pa, int pe, const int *__restrict__ ja,
                                             const double *__restrict__ aval,
                                             const int *__restrict__ ib,
                                             const int *__restrict__ jb,
                                             const double *__restrict__ bval, BlockPtrs bp,
                                             int c0, int c1, int *heads, F &&f, int part = 0) {
    const int l = __lane_id();
    // Software pipeline over groups of A entries: the A entry (t, a) of group
    // g+2 and the B range of group g+1 are loaded while group g's products
    // are processed.
    auto load_t = [&](int g, int &t, double &a) {
        const int p = g + PARTS * l + part;
        t = -1;
        a = 0.0;
        if (g < pe && p < pe) {
            t = ja[p];
            if (VALUES) a = aval[p];
        }
    };
    auto load_range = [&](int t, int &lo, int &hi) {
        lo = 0;
        hi = 0;
        if (t >= 0) {
            if (RANGED) {
                lo = brange_lo(bp, jb, t, c0);
                hi = brange_lo(bp, jb, t, c1);
            } else {
                lo = ib[t];
                hi = ib[t + 1];
            }
        }
    };
    int t0, t1;
    double a0, a1;
    load_t(pa, t0, a0);
    load_t(pa + 64 * PARTS, t1, a1);
    int lo, hi;
    load_range(t0, lo, hi);
    for (int g = pa; g < pe; g += 64 * PARTS) {
        const double a = a0;
        int lo_n, hi_n, t2;
        double a2;
        load_range(t1, lo_n, hi_n);                 // next group's B ranges
        load_t(g + 128 * PARTS, t2, a2);            // group after next
        expand_group<U, VALUES>(lo, max(hi - lo, 0), a, jb, bval, heads, f);
        lo = lo_n;
        hi = hi_n;
        t1 = t2;
        a0 = a1;
        a1 = a2;
    }
}

// Insert col into an LDS linear-probing table; returns the slot and whether
// this call created the key.  At most SLOTS probes: a full table (which the
// symbolic phase's sizing rules out) yields -1 instead of spinning.
template <int SLOTS>
__device__ __forceinline__ int hash_insert(int *keys, int col, bool &created) {
    unsigned h = hash_col(col, SLOTS - 1);
    created = false;
    for (int probe = 0; probe < SLOTS; probe++) {
        int k = keys[h];
        if (k == col) return (int)h;
        if (k == -1) {
            int old = atomicCAS(&keys[h], -1, col);
            if (old == -1) { created = true; return (int)h; }
            if (old == col) return (int)h;
        }
        h = (h + 1) & (SLOTS - 1);
    }
    return -1;
}

template <int SLOTS>
__device__ __forceinline__ int hash_find(const int *keys, int col) {
    unsigned h = hash_col(col, SLOTS - 1);
    for (int probe = 0; probe < SLOTS; probe++) {
        if (keys[h] == col) return (int)h;
        h = (h + 1) & (SLOTS - 1);
    }
    return -1;
}

// Ordered read-modify-write of vals[slot] by the active lanes of a batch:
// lanes sharing a tag bucket go one per round, lowest lane (earliest product)
// first, so every slot sees its products in product order.
// With single (all active lanes from one duplicate-free B row, hence distinct
// slots) the update is done in one step.
template <bool FUSED, int NTAGS>
__device__ __forceinline__ void ordered_accumulate(bool act, int slot, double a, double b,
                                                   double *vals, unsigned *tags,
                                                   unsigned me, bool single) {
    if (single) {
        if (act && slot >= 0) vals[slot] = acc_step<FUSED>(vals[slot], a, b);
        wave_lds_fence();
        return;
    }
    bool pending = act && slot >= 0;
    const unsigned bucket = (unsigned)slot & (NTAGS - 1);
    while (__ballot(pending)) {
        if (pending) atomicMin(&tags[bucket], me);
        wave_lds_fence();
        bool win = pending && tags[bucket] == me;
        wave_lds_fence();
        if (win) {
            vals[slot] = acc_step<FUSED>(vals[slot], a, b);
            tags[bucket] = 0xffffffffu;
            pending = false;
        }
        wave_lds_fence();
    }
}
