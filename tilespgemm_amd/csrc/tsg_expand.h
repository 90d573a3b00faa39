// Flat product expansion, LDS hash tables and ordered accumulation shared by
// the row path and the tile path (gfx950, wave64).
#pragma once

#include "tsg_device.h"

// ------------------------------------------------- ranges of B's rows
// B block pointers: entry (row t, block b) = first position of B row t with
// column >= b << bs, at p[t*tstride + b] (a row's entries together).  B's row
// pointers are a table of one block.
struct BlockPtrs {
    const int *p = nullptr;
    int64_t tstride = 0;
    int bs = 0;
};

// Range of B row t restricted to columns >= c, through the block pointers
// (a binary search inside the block when c is not a block boundary).
__device__ __forceinline__ int brange_lo(const BlockPtrs &bp, const int *__restrict__ jb, int t,
                                         int c) {
    const int b = c >> bp.bs;
    const int64_t e = (int64_t)t * bp.tstride + b;
    int lo = bp.p[e];
    if (c & ((1 << bp.bs) - 1)) {
        int hi = bp.p[e + 1];
        lo = lower_bound_i32(jb, lo, hi, c);
    }
    return lo;
}

// How B's rows are cut to an item: by the run directory where it is there,
// else by block pointers.
struct BRows {
    BlockPtrs bp;
    RunDir dir;
};

// B rows' positions with columns in [c0, c1), in two steps so that loads can
// be issued ahead: ahead(t), then range(t, that, lo, hi); t < 0: none.  DIR: by
// the run directory; [c0, c1) then holds all the work's columns in an aligned
// power of two of sub-blocks, so its runs are those of the smallest block that
// holds it.
template <bool DIR>
struct ItemRange {
    const BRows *b;
    const int *jb;
    const uint2 *cells;
    int c0, c1;
    __device__ __forceinline__ ItemRange(const BRows &b_, const int *jb_, int c0_, int c1_)
        : b(&b_), jb(jb_), c0(c0_), c1(c1_) {
        if (DIR) {
            const unsigned x = (unsigned)(c0 ^ (c1 - 1)) >> b->dir.shift;
            const int v = x ? 32 - __clz(x) : 0;
            cells = b->dir.cells + run_dir_block(b->dir.nblk, b->dir.shift, v, c0) * b->dir.ngrp;
        }
    }
    __device__ __forceinline__ uint2 ahead(int t) const {
        return DIR && t >= 0 ? cells[t >> 5] : make_uint2(0u, 0u);
    }
    __device__ __forceinline__ void range(int t, uint2 w, int &lo, int &hi) const {
        lo = 0;
        hi = 0;
        if (DIR) {
            const unsigned bit = 1u << (t & 31);
            if (w.x & bit) {
                const int2 r = b->dir.runs[w.y + __popc(w.x & (bit - 1))];
                lo = r.x;
                hi = r.y;
                if (b->dir.coarse) {       // a block may hold more than the item
                    lo = lower_bound_i32(jb, lo, hi, c0);
                    hi = lower_bound_i32(jb, lo, hi, c1);
                }
            }
        } else if (t >= 0) {
            lo = brange_lo(b->bp, jb, t, c0);
            hi = brange_lo(b->bp, jb, t, c1);
        }
    }
};

// B's whole rows.
struct RowRange {
    const int *ib;
    __device__ __forceinline__ uint2 ahead(int) const { return make_uint2(0u, 0u); }
    __device__ __forceinline__ void range(int t, uint2, int &lo, int &hi) const {
        lo = t >= 0 ? ib[t] : 0;
        hi = t >= 0 ? ib[t + 1] : 0;
    }
};

// Position p of a lane's entry in the group of a row's entries that starts at
// g (PARTS groups interleaved, the lane's the part-th); false past the row's
// end pe.  Groups are asked for up to three ahead of a row's last, so g is
// unsigned and the lane's offset compared with the entries left: g passes 2^31
// at the end of 2^31 - 1 entries.  (Unsigned positions, compared and indexed
// with, cost k_big_numeric_small two registers' spills.)
template <int PARTS>
__host__ __device__ __forceinline__ bool entry_at(unsigned g, unsigned pe, int part, int lane,
                                                  int &p) {
    p = (int)(g + (unsigned)(PARTS * lane + part));
    return PARTS * lane + part < (int)(pe - g);
}

// A row's entries [pa, pe) in groups of 64, loaded ahead of their use: while
// a group's products are processed, the next group's B ranges and values, the
// cells of the group after that and the A columns of the third are loading.
// load() and cells() start it, first() gives group 0's ranges (each uses what
// the one before has loaded, so other work goes between them).  With PARTS > 1
// only the entries part, part + PARTS, ... are visited.
template <bool VALUES, int PARTS>
struct EntryPipe {
    const int *ja;
    const double *aval;
    unsigned pa, pe;
    int part;
    int t1, t2;
    uint2 w1;
    int lo, hi, lo1, hi1;          // the group's ranges, and the next one's
    double a, a1;
    __device__ __forceinline__ int col(unsigned g) const {
        int p;
        return entry_at<PARTS>(g, pe, part, __lane_id(), p) ? ja[p] : -1;
    }
    __device__ __forceinline__ double val(unsigned g) const {
        int p;
        return VALUES && entry_at<PARTS>(g, pe, part, __lane_id(), p) ? aval[p] : 0.0;
    }
    __device__ __forceinline__ void load(int pa_, int pe_) {
        pa = (unsigned)pa_;
        pe = (unsigned)pe_;
        t1 = col(pa);
        t2 = col(pa + 64 * PARTS);
    }
    template <class R>
    __device__ __forceinline__ void cells(const R &rows) {
        w1 = rows.ahead(t1);
    }
    // the next group's ranges, and what lies behind them; g: the group at hand
    template <class R>
    __device__ __forceinline__ void ahead(unsigned g, const R &rows) {
        rows.range(t1, w1, lo1, hi1);
        a1 = val(g + 64 * PARTS);
        t1 = t2;
        w1 = rows.ahead(t2);
        t2 = col(g + 3 * 64 * PARTS);
    }
    __device__ __forceinline__ void take() {
        lo = lo1;
        hi = hi1;
        a = a1;
    }
    template <class R>
    __device__ __forceinline__ void first(const R &rows) {
        ahead(pa - 64 * PARTS, rows);
        take();
    }
};

// ------------------------------------------------- flat product expansion
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

// One round of expand_group: the products [base, base + 64 U) of a group.  A
// short rest takes a round of half or a quarter of the batches (R-MAT 2^20 with
// 8 draws a row: symbolic bands 12.1 -> 11.6 ms, items of more than 512 outputs
// 15.9 -> 15.5).
template <int U, bool VALUES, bool PACKED, class F>
__device__ __forceinline__ void expand_round(int base, int total, int start, int cnt, int off,
                                             double av, const int *__restrict__ jb,
                                             const double *__restrict__ bval, int *heads, F &f,
                                             const int4 *__restrict__ bpk) {
    const int l = __lane_id();
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

// Products of one group of 64 A entries: lane l's A entry contributes the B
// positions [lo, lo + cnt) with value a.  Batches of 64 products are handed
// to f in product order (see for_products).
//
// A product finds its A entry by counting: the entries with products move to
// the front lanes (a permutation, once per group), a bit is set in LDS (heads:
// 2 U ints, any content) where each one's products start, and product q
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
    for (int base = 0; base < total;) {
        const int left = total - base;
        if (U >= 4 && left <= 64 * (U / 4)) {
            expand_round<(U >= 4 ? U / 4 : U), VALUES, PACKED>(base, total, start, cnt, off, av, jb,
                                                               bval, heads, f, bpk);
            break;
        }
        if (U >= 2 && left <= 64 * (U / 2)) {
            expand_round<(U >= 2 ? U / 2 : U), VALUES, PACKED>(base, total, start, cnt, off, av, jb,
                                                               bval, heads, f, bpk);
            break;
        }
        expand_round<U, VALUES, PACKED>(base, total, start, cnt, off, av, jb, bval, heads, f, bpk);
        base += 64 * U;
    }
}

// Visits the products of the A entries [pa, pe) of one row in A-row order, a
// wave's 64 entries at a time, each entry's B positions given by rows (an
// ItemRange or RowRange).  f(batch) is called once per batch by every lane;
// batches are issued in product order and lane order inside a batch is product
// order.  U batches are gathered before the first is handed to f, so each lane
// keeps U independent loads in flight.  With PARTS > 1 only the A entries
// part, part + PARTS, ... are visited, so several waves can share a row where
// the order of products does not matter (entries, not batches of one group:
// what a group costs before its first product is then spent once, and
// alternate entries, because a row's first ones may name the longest B rows).
// heads: 2 U ints of LDS.
template <int U, int PARTS, bool VALUES, class R, class F>
__device__ __forceinline__ void for_products(int pa, int pe, const int *__restrict__ ja,
                                             const double *__restrict__ aval, const R &rows,
                                             const int *__restrict__ jb,
                                             const double *__restrict__ bval, int *heads, F &&f,
                                             int part = 0) {
    EntryPipe<VALUES, PARTS> pipe;
    pipe.ja = ja;
    pipe.aval = aval;
    pipe.part = part;
    pipe.load(pa, pe);
    pipe.cells(rows);
    pipe.first(rows);
    for (unsigned g = pipe.pa; g < pipe.pe; g += 64 * PARTS) {
        pipe.ahead(g, rows);
        expand_group<U, VALUES>(pipe.lo, max(pipe.hi - pipe.lo, 0), pipe.a, jb, bval, heads, f);
        pipe.take();
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
        // both reads in one wait: the value is used by the bucket's winner
        unsigned first = 0u;
        double v = 0.0;
        if (pending) {
            first = tags[bucket];
            v = vals[slot];
        }
        wave_lds_fence();
        if (pending && first == me) {
            vals[slot] = acc_step<FUSED>(v, a, b);
            tags[bucket] = 0xffffffffu;
            pending = false;
        }
        wave_lds_fence();
    }
}
