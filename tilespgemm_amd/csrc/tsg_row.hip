// Row path: row-binned SpGEMM for matrices whose 16x16 tiles are too sparse
// for the tile path (hypersparse / power-law inputs such as R-MAT).
//
// Lineage: the reference bins rows by intermediate products and runs per-bin
// hash kernels (nsparse, spgemm_nsparse_kernel.h:221-311 binning, :331-687
// symbolic hash, :696-1119 structure fill; its value-carrying variant is
// commented out at :805-907).  This path is built for gfx950 instead:
//
//   * Every output entry is accumulated from +0.0 over its products in A-row
//     order (thmkl_dcsrmultcsr.c:61-72), so results are bitwise equal to the
//     CPU reference.  Products are expanded flat, a wave at a time in A-row
//     order ("t-major"); lanes of one batch that hit the same accumulator slot
//     take turns in product order (one B row after the other, or tag rounds:
//     LDS atomicMin on a small bucket table), so the parallel sum equals the
//     sequential one.
//   * Small rows (<= 1024 products, or 1536): one lane group per row with all its
//     products in registers (tsg_flat.h); an output's place is its column's
//     rank in a two-level bitmap, so C comes out sorted with no hash or sort.
//   * Big rows: the symbolic phase cuts each row's column span into bands of
//     65536 columns, marks the row's columns of a band in an LDS bitmap and
//     records the count of every 1024-column sub-block (and, when memory
//     allows, the band's bitmap in sparse form: a mask of non-empty words per
//     sub-block, and those words); the numeric phase splits the row into
//     items of <= ITEM_CAP outputs and <= 16384 columns, each accumulated by
//     one wave into a rank-ordered LDS array (rank from the stored bitmap)
//     and written in column order.  Bands and items of wide matrices run in
//     order of their first column, so those in flight share a band of B, and a
//     run directory of B gives each B row's entries in a band or item; else a
//     table of block pointers does, or a search.
#include "tsg_internal.h"

#include <cmath>
#include "tsg_device.h"
#include "tsg_expand.h"
#include "tsg_flat.h"

#include <algorithm>
#include <map>
#include <mutex>

namespace {

constexpr int BAND_SHIFT = 6;          // symbolic band = 64 sub-blocks (65536 columns)
constexpr int BAND_T = 128;            // threads per band unit
constexpr int BAND_WORDS = (1 << (BAND_SHIFT + SUB_SHIFT)) / 32;
constexpr int BAND_PAD = 4;            // band word lists: words rounded up to this
constexpr int ITEM_CAP = 1024;         // outputs per item
constexpr int ITEM_SLOTS = 2048;       // hash slots per item (load <= 1/2)
constexpr int ITEM_WBITS_SHIFT = 14;   // item width <= 16384 columns
constexpr int ITEM_WORDS = (1 << ITEM_WBITS_SHIFT) / 32;
// items are whole sub-blocks, and one sub-block can hold 1 << SUB_SHIFT outputs
static_assert(ITEM_CAP >= (1 << SUB_SHIFT), "an item must hold a full sub-block");
constexpr int ITEM_TAGS = 256;
constexpr int ITEM_WAVES = 1;          // waves per block (one item per wave)
constexpr int RANK_U = 8;
constexpr int BIG_SYM_U = 8;
constexpr int ITEM_U = 4;

// Rows an XCD takes in a run: neighbours share B rows (stencils) or a matrix of
// a batch.  ER batch of 512, numeric, 16 products a lane: 10.74 ms in turns,
// 10.31 in runs of 64, 10.35 of 512, 10.70 an eighth each; 27-point 64^3 687, 671,
// 667, 677 us.  (Items and bands, which run in column order and read one band of
// B together, gain nothing.)
constexpr unsigned FLAT_CHUNK = 64;

// ------------------------------------------------------ small rows: symbolic
// Output count of each row of at most G * U products (rownnz), G lanes a row:
// the columns gathered into registers and counted by the bitmaps of
// tsg_flat.h.  Bound: random B rows by memory (ER batch, rows of 513..1024
// products: 2.7 ms, 14 GB of column lines), stencils by issue.  Against a
// separate pass for the row's span and a flat expansion in rounds into one
// bitmap or hash: ER batch of 512 9.3 -> 5.6 ms, 27-point 64^3 0.46 -> 0.24 ms,
// rectangular ER 75 -> 58 us, R-MAT 2^18 0.39 -> 0.09 ms.  6 waves per SIMD at
// 16 products a lane: 3.2 ms (ER) and 258 us (stencil) unforced, 2.8 and 225 at
// 5, 2.7 and 213 at 6, 3.4 and 212 at 7 (spills).
template <int G, int U, int NB, int E, int LW>
__device__ __forceinline__ int flat_count_row(FlatSmem<G * U, E, LW, 1> &S, int total,
                                              const int *__restrict__ jb) {
    const int l = threadIdx.x & (G - 1);
    const FlatHeads<G, U> heads(S.starts);
    int col[NB], rank[NB];
    int before = -1;                   // entries that start before the batch, less one
#pragma unroll
    for (int u = 0; u < NB; u++) {
        const unsigned long long m = heads(u);
        col[u] = jb[S.off[heads.at(m, before)] + min(u * G + l, total - 1)];
        before += __popcll(m);
    }
    return flat_ranks<G, NB, false>(S, col, rank, true);
}

template <int G, int U, int E, int LW, int THREADS, int MINW = 1>
__global__ void __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(MINW)))
k_flat_symbolic(int nrows, const int *__restrict__ rows, const int *__restrict__ ia,
                const int *__restrict__ ja, const int *__restrict__ ib,
                const int *__restrict__ jb, int64_t *__restrict__ rownnz) {
    constexpr int RPB = THREADS / G;
    __shared__ __align__(16) FlatSmem<G * U, E, LW, 1> s_row[RPB];
    const int grp = threadIdx.x / G;
    FlatSmem<G * U, E, LW, 1> &S = s_row[grp];
    const int r = xcd_piece<FLAT_CHUNK>(blockIdx.x, gridDim.x) * RPB + grp;
    if (r >= nrows) return;
    const int row = group_uniform<G>(rows[r]);
    const int total = flat_entries<G>(S, ia[row], ia[row + 1], ja, (const double *)nullptr, ib);
    int n = 0;
    if (total > 0)
        n = G == 64 && total <= G * U / 4 * 3 ? flat_count_row<G, U, U / 4 * 3>(S, total, jb)
                                              : flat_count_row<G, U, U>(S, total, jb);
    if ((threadIdx.x & (G - 1)) == 0) rownnz[row] = n;
}

// ------------------------------------------------------- small rows: numeric
// A batch whose products come from at most this many B rows is accumulated
// one B row after the other; past that, tag rounds take fewer steps.  Numeric
// phase of 65537 rows of 9 banded entries: 111 us at 4, 98 at 8, 12, 20 and 64;
// the 27-point product, wider bands and ER the same at all of them.
constexpr int FLAT_SEGS = 12;

// One row of at most G * NB products, G lanes a row (tsg_flat.h), its entries
// in S.  The columns and B values of every product are gathered once into
// registers, the columns ranked, C's columns written, and the values summed
// in LDS in product order, ACC outputs at a time: a batch of G products takes
// one step when they come from one B row (distinct columns) or when a check
// finds their outputs distinct, one step per B row when those are few, else
// tag rounds.
template <bool FUSED, int G, int U, int NB, int E, int LW, int ACC>
__device__ __forceinline__ void flat_numeric_row(FlatSmem<G * U, E, LW, ACC> &S,
                                                 unsigned *tags, int total, int64_t o,
                                                 int64_t nrow, const int *__restrict__ jb,
                                                 const double *__restrict__ b,
                                                 int *__restrict__ jc, double *__restrict__ c,
                                                 int b_strict) {
    constexpr int NT = ACC / 4;                    // a byte per output of a pass
    const int l = threadIdx.x & (G - 1);
    // few products share an output
    const bool sparse = nrow * 4 >= (int64_t)total * 3;
    const FlatHeads<G, U> heads(S.starts);
    int col[NB], rank[NB];
    double bv[NB];
    {
        int e[NB];
        int before = -1;               // entries that start before the batch, less one
#pragma unroll
        for (int u = 0; u < NB; u++) {
            const unsigned long long m = heads(u);
            e[u] = S.off[heads.at(m, before)] + min(u * G + l, total - 1);
            before += __popcll(m);
            col[u] = jb[e[u]];
        }
#pragma unroll
        for (int u = 0; u < NB; u++) bv[u] = b[e[u]];
    }
    const int found = flat_ranks<G, NB, true>(S, col, rank, !sparse);
    // the symbolic phase counted the same outputs
    const int nnz = group_uniform<G>((int)min((int64_t)found, nrow));
#pragma unroll
    for (int u = 0; u < NB; u++) S.cols[rank[u]] = col[u];
    wave_lds_fence();
    for (int i = l; i < nnz; i += G) jc[o + i] = S.cols[i];
    uint8_t *own = reinterpret_cast<uint8_t *>(tags);
    for (int r0 = 0; r0 < nnz; r0 += ACC) {
        const int nout = min(ACC, nnz - r0);
        wave_lds_fence();
        for (int i = l; i < nout; i += G) S.acc[i] = 0.0;
        wave_lds_fence();
        int before = 0;                // entries that start before the batch
#pragma unroll
        for (int u = 0; u < NB; u++) {
            // the batch's B rows: the product's index among them (from 1),
            // their number, the entry of the first
            const unsigned long long hm = heads(u);
            const unsigned long long m = hm | 1ull;
            const int seg = heads.at(m, 0);
            const int nseg = __popcll(m);
            const int first = before - (int)(~hm & 1ull);
            before += __popcll(hm);
            const int out = rank[u] - r0;
            const bool act = u * G + l < total && (unsigned)out < (unsigned)nout;
            const double av = S.a[first + seg - 1];
            bool clash = !b_strict || nseg > 1;
            if (clash && b_strict && sparse) {
                if (act) own[out] = (uint8_t)l;
                wave_lds_fence();
                clash = group_ballot<G>(act && own[out] != (uint8_t)l) != 0;
                wave_lds_fence();
            }
            if (!clash) {
                if (act) S.acc[out] = acc_step<FUSED>(S.acc[out], av, bv[u]);
                wave_lds_fence();
            } else if (b_strict && nseg <= FLAT_SEGS) {
                for (int s = 1; s <= nseg; s++) {
                    if (act && seg == s) S.acc[out] = acc_step<FUSED>(S.acc[out], av, bv[u]);
                    wave_lds_fence();
                }
            } else {
                for (int i = l; i < NT; i += G) tags[i] = 0xffffffffu;
                wave_lds_fence();
                ordered_accumulate<FUSED, NT>(act, out, av, bv[u], S.acc, tags, (unsigned)l,
                                              false);
            }
        }
        for (int i = l; i < nout; i += G) c[o + r0 + i] = S.acc[i];
    }
}

template <bool FUSED, int G, int U, int E, int LW, int ACC, int THREADS, int MINW = 1>
__global__ void __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(MINW)))
k_flat_numeric(
    int nrows, const int *__restrict__ rows, const int *__restrict__ ia,
    const int *__restrict__ ja, const double *__restrict__ a, const int *__restrict__ ib,
    const int *__restrict__ jb, const double *__restrict__ b, const int64_t *__restrict__ ic,
    int *__restrict__ jc, double *__restrict__ c, int b_strict) {
    constexpr int RPB = THREADS / G;
    __shared__ __align__(16) FlatSmem<G * U, E, LW, ACC> s_row[RPB];
    __shared__ unsigned s_tags[RPB][ACC / 4];
    const int grp = threadIdx.x / G;
    FlatSmem<G * U, E, LW, ACC> &S = s_row[grp];
    const int r = xcd_piece<FLAT_CHUNK>(blockIdx.x, gridDim.x) * RPB + grp;
    if (r >= nrows) return;
    const int row = group_uniform<G>(rows[r]);
    const int64_t o = ic[row];
    const int64_t nrow = ic[row + 1] - o;
    const int total = flat_entries<G>(S, ia[row], ia[row + 1], ja, a, ib);
    if (total <= 0) return;
    if (G == 64 && total <= G * U / 4 * 3)
        flat_numeric_row<FUSED, G, U, U / 4 * 3>(S, s_tags[grp], total, o, nrow, jb, b, jc, c,
                                                 b_strict);
    else
        flat_numeric_row<FUSED, G, U, U>(S, s_tags[grp], total, o, nrow, jb, b, jc, c, b_strict);
}

// -------------------------------------------------------- big rows: span
// Column span of each big row, in 1024-column sub-blocks: from the first
// sub-block of the first B column to the last sub-block of the last B column
// over the row's A entries, and a bound on the words of the row's band word
// lists: min(products, span words) plus each band's padding.  One wave per
// big row.
__global__ void __launch_bounds__(256) k_big_span(int nbig, const int *__restrict__ rows,
                                                  const int *__restrict__ ia,
                                                  const int *__restrict__ ja,
                                                  const int *__restrict__ ib,
                                                  const int *__restrict__ jb,
                                                  const int64_t *__restrict__ rowprod,
                                                  int *__restrict__ sb0,
                                                  int64_t *__restrict__ nsb,
                                                  int64_t *__restrict__ nent,
                                                  int64_t *__restrict__ nprod,
                                                  int64_t *__restrict__ lbound) {
    const int l = threadIdx.x & 63;
    for (int64_t r = wave_index(); r < nbig; r += wave_count()) {
        const int row = rows[r];
        int lo = 0x7fffffff, hi = -1;
        const unsigned pe = (unsigned)ia[row + 1];
        for (unsigned p = (unsigned)ia[row] + l; p < pe; p += 64) {
            const int t = ja[p];
            const int b0 = ib[t], b1 = ib[t + 1];
            if (b0 < b1) {
                lo = min(lo, jb[b0] >> SUB_SHIFT);
                hi = max(hi, jb[b1 - 1] >> SUB_SHIFT);
            }
        }
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) {
            lo = min(lo, __shfl_xor(lo, d, 64));
            hi = max(hi, __shfl_xor(hi, d, 64));
        }
        if (l == 0) {
            const int64_t ns = hi >= lo ? (int64_t)(hi - lo + 1) : 0;
            sb0[r] = hi >= lo ? lo : 0;
            nsb[r] = ns;
            nent[r] = ia[row + 1] - ia[row];
            nprod[r] = rowprod[row];
            // a multiple of BAND_PAD, so every band's list starts 16-byte aligned
            lbound[r] = ((min(rowprod[row], ns << (SUB_SHIFT - 5)) + BAND_PAD - 1) & -BAND_PAD) +
                        BAND_PAD * (((ns + (1 << BAND_SHIFT) - 1) >> BAND_SHIFT) + 1);
        }
    }
}

// -------------------------------------------------------- big rows: symbolic
// A big row's span is cut into bands of 64 sub-blocks; a band unit {r, u}
// covers span sub-blocks [64u - lead, 64u + 64 - lead) of big row r.  Units are
// run in order of their first column (like the numeric items), so the units
// in flight read B columns of one narrow band, which the L2 caches keep; bands
// are then the matrix's (lead = the sub-blocks of the first band before the
// span), as the run directory of B has them, else the span's (lead = 0).
__device__ __forceinline__ int band_lead(int span_sb0) {
    return span_sb0 & ((1 << BAND_SHIFT) - 1);
}

__global__ void __launch_bounds__(256) k_band_count(int nbig, int64_t sort_min,
                                                    const int *__restrict__ span_sb0,
                                                    const int64_t *__restrict__ sb_off,
                                                    int64_t *__restrict__ cnt) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= nbig) return;
    const int lead = sb_off[nbig] / 16 >= sort_min ? band_lead(span_sb0[r]) : 0;
    cnt[r] = (lead + sb_off[r + 1] - sb_off[r] + (1 << BAND_SHIFT) - 1) >> BAND_SHIFT;
}

__global__ void __launch_bounds__(256) k_band_fill(int nbig, const int *__restrict__ span_sb0,
                                                   const int64_t *__restrict__ off,
                                                   int2 *__restrict__ units,
                                                   int *__restrict__ keys) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= nbig) return;
    const int64_t o = off[r], n = off[r + 1] - o;
    for (int u = 0; u < n; u++) {
        units[o + u] = make_int2(r, u);
        keys[o + u] = span_sb0[r] + (u << BAND_SHIFT);   // its band's, less than one off
    }
}

__global__ void __launch_bounds__(256) k_gather_units(int64_t n, const int *__restrict__ order,
                                                      const int2 *__restrict__ units,
                                                      int2 *__restrict__ out) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j < n) out[j] = units[order[j]];
}

// One block per band unit: LDS bitmap over the band, the row's products in
// the band (B rows cut to the band by brows) marked by the 2
// waves, each taking every other A entry; then the band's sub-block
// output counts, its share of the row's output count (rownnz of big rows is
// zero on entry) and, when words is given, the band's bitmap in sparse form:
// per sub-block a mask of its non-empty words (subocc), and the non-empty
// words themselves in column order (the band word list), in the row's region
// [row_off[r], row_off[r + 1]) at a position taken from the row's cursor
// (row_cur[r], starting at row_off[r]) and recorded in
// band_base[band_off[r] + u].  On R-MAT's big rows a fifth of the span's
// words are non-empty, so the lists and masks take a quarter of the bitmap's
// bytes, and no step expands bits.  A band takes its word count rounded up to
// BAND_PAD, so its list starts 16-byte aligned and goes out in whole 16-byte
// stores, staged in the bitmap's LDS once the words are in registers (one
// cursor for all bands had them queue on a single address; the cursor's
// result is first needed after the staging).  A band whose list would pass
// its row's region writes none and sets *overflow, which the host checks.
// Bound by vector instructions, most of them per group of 64 A entries and not
// per product, so the waves share a row by entries (sharing each group's
// batches repeated that work in both: R-MAT 2^20 with 8 draws a row 13.3 ms,
// now 11.8; 2^18 with 4, times its transpose, 0.64 -> 0.47), 8 batches in
// flight (4: 12.0 and 0.54 ms; 2: 12.9 and 0.70).
// 8 waves per SIMD, as with no word lists (the kernel waits on its gathers;
// its arguments alone would take the scalar registers past that).
template <bool DIR>
__global__ void __launch_bounds__(BAND_T) __attribute__((amdgpu_waves_per_eu(8))) k_big_symbolic(
    int64_t nunits, const int2 *__restrict__ units, const int *__restrict__ rows, int k,
    int by_band, const int *__restrict__ ia, const int *__restrict__ ja,
    const int *__restrict__ jb, BRows brows, const int *__restrict__ span_sb0,
    const int64_t *__restrict__ sb_off, uint16_t *__restrict__ subcnt,
    int64_t *__restrict__ rownnz, const int64_t *__restrict__ band_off,
    int64_t *__restrict__ band_base, unsigned long long *__restrict__ row_cur,
    const int64_t *__restrict__ row_off, int64_t *__restrict__ overflow,
    unsigned *__restrict__ subocc, unsigned *__restrict__ words_out) {
    constexpr int NW = BAND_T / 64;
    constexpr int TW = BAND_WORDS / BAND_T;        // words per thread, half a sub-block
    static_assert(TW == 16 && 2 * TW == (1 << (SUB_SHIFT - 5)), "a sub-block is two threads' words");
    __shared__ __align__(16) unsigned bits[BAND_WORDS];
    __shared__ int s_heads[NW][64];
    __shared__ int s_wsum[NW];
    __shared__ long long s_base;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int64_t ui = blockIdx.x; ui < nunits; ui += gridDim.x) {
        const int2 un = units[ui];
        const int r = un.x, u = un.y;
        const int row = rows[r];
        const int lead = by_band ? band_lead(span_sb0[r]) : 0;
        const int j0 = max((u << BAND_SHIFT) - lead, 0);
        const int64_t so = sb_off[r] + j0;
        const int nsb = (int)min((int64_t)((u + 1) << BAND_SHIFT) - lead - j0, sb_off[r + 1] - so);
        const int sb0 = span_sb0[r] + j0;
        const int c0 = sb0 << SUB_SHIFT;
        const int c1 = sub_block_start(sb0 + nsb, k);
        const int words = (c1 - c0 + 31) >> 5;
        for (int i = threadIdx.x; 4 * i < words; i += BAND_T)
            reinterpret_cast<uint4 *>(bits)[i] = make_uint4(0u, 0u, 0u, 0u);
        __syncthreads();
        for_products<BIG_SYM_U, NW, false>(
            ia[row], ia[row + 1], ja, nullptr, ItemRange<DIR>(brows, jb, c0, c1), jb, nullptr,
            s_heads[wave], [&](const Batch &t) {
                if (t.act) {
                    const int cc = t.col - c0;
                    lds_set_bit(&bits[cc >> 5], 1u << (cc & 31));
                }
            },
            wave);
        __syncthreads();
        // thread t takes words [TW t, TW t + TW) (words past the band's end
        // are stale); threads 2s and 2s + 1 hold sub-block s
        unsigned wv[TW];
        int tot = 0;
        unsigned nzm = 0;
        {
            const uint4 *src = reinterpret_cast<const uint4 *>(bits) + threadIdx.x * (TW / 4);
#pragma unroll
            for (int q = 0; q < TW / 4; q++) {
                const uint4 v = src[q];
                wv[4 * q] = v.x;
                wv[4 * q + 1] = v.y;
                wv[4 * q + 2] = v.z;
                wv[4 * q + 3] = v.w;
            }
#pragma unroll
            for (int j = 0; j < TW; j++) {
                if ((int)threadIdx.x * TW + j >= words) wv[j] = 0u;
                tot += __popc(wv[j]);
                nzm |= (wv[j] != 0u ? 1u : 0u) << j;
            }
        }
        const int sbc = tot + __shfl_xor(tot, 1, 64);
        const unsigned occ = nzm | (__shfl_xor(nzm, 1, 64) << TW);
        if (!(threadIdx.x & 1) && (int)(threadIdx.x >> 1) < nsb) {
            subcnt[so + (threadIdx.x >> 1)] = (uint16_t)sbc;
            if (words_out) subocc[so + (threadIdx.x >> 1)] = occ;
        }
        // block-wide scans: outputs (for the row's count) and non-empty words
        const int nz = __popc(nzm);
        const int packed_incl = wave_incl_scan(tot | (nz << 16));
        if (lane == 63) s_wsum[wave] = packed_incl;
        __syncthreads();
        int before = (packed_incl >> 16) - nz, total = 0, total_nz = 0;
#pragma unroll
        for (int i = 0; i < NW; i++) {
            const int wsum = s_wsum[i];
            if (i < wave) before += wsum >> 16;
            total += wsum & 0xffff;
            total_nz += wsum >> 16;
        }
        const int padded = (total_nz + BAND_PAD - 1) & -BAND_PAD;
        // thread 0 takes the band's place in its row's region; the result is
        // first needed after the list is staged, so the atomic's round trip
        // overlaps the staging
        unsigned long long ticket = 0;
        if (threadIdx.x == 0) {
            if (total)
                atomicAdd(reinterpret_cast<unsigned long long *>(rownnz + row),
                          (unsigned long long)total);
            if (words_out && padded)
                ticket = atomicAdd(row_cur + r, (unsigned long long)padded);
        }
        if (words_out && total_nz > 0) {
            // the band's <= 2048 non-empty words fit the bitmap's LDS
            int pos = before;
#pragma unroll
            for (int j = 0; j < TW; j++) {
                if (wv[j]) bits[pos] = wv[j];
                pos += wv[j] ? 1 : 0;
            }
            if (threadIdx.x == 0) {
                long long base = (long long)ticket;
                if (base + padded > row_off[r + 1]) {
                    *overflow = 1;
                    base = -1;
                }
                band_base[band_off[r] + u] = base;
                s_base = base;
            }
            __syncthreads();
            const long long base = s_base;
            if (base >= 0) {
                // whole 16-byte stores, the last into the band's padding.
                // Written once, read once by the numeric phase much later:
                // streaming stores keep the L2 for B's rows
                typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
                u32x4 *dst = reinterpret_cast<u32x4 *>(words_out + base);
                const u32x4 *sv = reinterpret_cast<const u32x4 *>(bits);
                for (int i = threadIdx.x; i < padded / 4; i += BAND_T)
                    __builtin_nontemporal_store(sv[i], dst + i);
            }
        }
        __syncthreads();
    }
}

// ------------------------------------------------------ B block pointers
// Row-major table: bptr[t*(nblk+1) + b] = first position of B row t with
// column >= b << bs; one wave per B row, a lane per block.
__global__ void __launch_bounds__(256) k_bptr_rows(int n, const int *__restrict__ ib,
                                                   const int *__restrict__ jb, int nblk, int bs,
                                                   int *__restrict__ bptr) {
    const int l = threadIdx.x & 63;
    for (int64_t t = wave_index(); t < n; t += wave_count()) {
        const int lo = ib[t], hi = ib[t + 1];
        for (int b = l; b <= nblk; b += 64) {
            const int pos = b == nblk ? hi : lower_bound_i32(jb, lo, hi, b << bs);
            bptr[t * (nblk + 1) + b] = pos;
        }
    }
}

// Run directory (RunDir), built in three passes: the cells' bits, the scan of
// their counts, the runs.
//
// Bits: a block takes DIR_ROWS B rows and ranges of DIR_BLK blocks of level 0,
// marks them in LDS and folds each level's pairs of blocks into the next's.
// The bits go out cell-major, DIR_ROWS / 32 consecutive cells a block.  Bound
// by the busiest block, that of the longest rows: 1.2 ms with 512 rows and
// threads a block (R-MAT 2^20, whole rows), 0.5 with 256 and 1024.
// With one range a block goes through its rows' entries.  With more (CUT) it
// has one of them and searches each row's entries in it, so that B is read once
// however many columns it has (B of 1000 rows of 20,000 entries over 2^28
// columns, symbolic phase 857 -> 7.0 ms).  R-MAT with 8 draws a row, whole and
// CUT: 2^16 (one range) 55 and 64 us, 2^18 142 and 163, 2^20 (two) 520 and 436.
constexpr int DIR_ROWS = 256, DIR_GRP = DIR_ROWS / 32, DIR_BLK = 512;

// row (of nr from the first) of the entry at position e: rp ascending
__device__ __forceinline__ int dir_row_of(const int *rp, int nr, int e) {
    int lo = 0, hi = nr;               // rp[lo] <= e < rp[hi]
    while (hi - lo > 1) {
        const int mid = lo + ((hi - lo) >> 1);
        if (rp[mid] <= e) lo = mid;
        else hi = mid;
    }
    return lo;
}

template <bool CUT>
__global__ void __launch_bounds__(1024) k_dir_bits(int n, const int *__restrict__ ib,
                                                  const int *__restrict__ jb, int ngrp, int nblk,
                                                  int shift, int levels,
                                                  unsigned *__restrict__ bits) {
    __shared__ int s_rp[DIR_ROWS + 1];
    __shared__ int s_first[CUT ? DIR_ROWS : 1], s_wave[CUT ? DIR_ROWS / 64 : 1];
    __shared__ unsigned s_bits[2 * DIR_BLK * DIR_GRP];
    const int t = threadIdx.x, t0 = blockIdx.x * DIR_ROWS, g0 = blockIdx.x * DIR_GRP;
    const int nr = min(DIR_ROWS, n - t0), ng = min(DIR_GRP, ngrp - g0);
    if (!CUT)
        for (int i = t; i <= nr; i += blockDim.x) s_rp[i] = ib[t0 + i];
    __syncthreads();
    for (int b0 = blockIdx.y * DIR_BLK; b0 < nblk; b0 += gridDim.y * DIR_BLK) {
        if (CUT) {
            // the rows' entries in the range, back to back: first and count
            int lo = 0, hi = 0, incl = 0;
            if (t < nr) {
                const int end = ib[t0 + t + 1];
                const int64_t past = (int64_t)(b0 + DIR_BLK) << shift;
                lo = lower_bound_i32(jb, ib[t0 + t], end, b0 << shift);
                hi = past <= 0x7fffffff ? lower_bound_i32(jb, lo, end, (int)past) : end;
            }
            if (t < DIR_ROWS) {
                incl = wave_incl_scan(hi - lo);
                if ((t & 63) == 63) s_wave[t >> 6] = incl;
            }
            __syncthreads();
            if (t < DIR_ROWS) {
                for (int w = 0; w < t >> 6; w++) incl += s_wave[w];
                s_rp[t + 1] = incl;
                s_first[t] = lo - (incl - (hi - lo));
                if (t == 0) s_rp[0] = 0;
            }
        }
        for (int i = t; i < DIR_BLK * DIR_GRP; i += blockDim.x) s_bits[i] = 0u;
        __syncthreads();
        for (unsigned e = s_rp[0] + t; e < (unsigned)s_rp[nr]; e += blockDim.x) {
            int r = CUT ? dir_row_of(s_rp, nr, (int)e) : 0;
            const int b = (jb[CUT ? s_first[r] + (int)e : (int)e] >> shift) - b0;
            if (b >= 0 && b < DIR_BLK) {
                if (!CUT) r = dir_row_of(s_rp, nr, (int)e);
                lds_set_bit(&s_bits[b * DIR_GRP + (r >> 5)], 1u << (r & 31));
            }
        }
        __syncthreads();
        unsigned *lev = s_bits;
        int cnt = min(DIR_BLK, nblk - b0);          // a multiple of 1 << (levels - 1)
        for (int v = 0; v < levels; v++, cnt >>= 1) {
            unsigned *out = bits + run_dir_block(nblk, 0, v, b0) * ngrp + g0;
            for (int i = threadIdx.x; i < cnt * DIR_GRP; i += blockDim.x)
                if (i % DIR_GRP < ng) out[(int64_t)(i / DIR_GRP) * ngrp + i % DIR_GRP] = lev[i];
            unsigned *up = lev + cnt * DIR_GRP;
            for (int i = threadIdx.x; i < (cnt >> 1) * DIR_GRP; i += blockDim.x) {
                const int a = (i / DIR_GRP) * 2 * DIR_GRP + i % DIR_GRP;
                up[i] = lev[a] | lev[a + DIR_GRP];
            }
            lev = up;
            __syncthreads();
        }
    }
}

// Scan of the cells' counts: chunks of DIR_CHUNK cells, a total each (then
// scanned), and the cells {bits, runs before}.
constexpr int DIR_CHUNK = 8192;

__global__ void __launch_bounds__(256) k_dir_sums(int64_t ncells, const unsigned *__restrict__ bits,
                                                  int64_t *__restrict__ sums) {
    __shared__ int s_sum[4];
    int64_t i = (int64_t)blockIdx.x * DIR_CHUNK + threadIdx.x * 4;
    int c = 0;
#pragma unroll
    for (int q = 0; q < DIR_CHUNK / 1024; q++, i += 1024) {
        // (the array is whole chunks)
        const uint4 v = *reinterpret_cast<const uint4 *>(bits + i);
        c += i < ncells ? __popc(v.x) : 0;
        c += i + 1 < ncells ? __popc(v.y) : 0;
        c += i + 2 < ncells ? __popc(v.z) : 0;
        c += i + 3 < ncells ? __popc(v.w) : 0;
    }
    c = wave_sum(c);
    if (__lane_id() == 0) s_sum[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) sums[blockIdx.x] = s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3];
}

__global__ void __launch_bounds__(256) k_dir_cells(int64_t ncells,
                                                   const unsigned *__restrict__ bits,
                                                   const int64_t *__restrict__ sums,
                                                   uint2 *__restrict__ cells) {
    __shared__ int s_sum[4];
    const int w = threadIdx.x >> 6;
    int before = (int)sums[blockIdx.x];
    for (int q = 0; q < DIR_CHUNK / 1024; q++) {
        const int64_t i = (int64_t)blockIdx.x * DIR_CHUNK + q * 1024 + threadIdx.x * 4;
        uint4 v = *reinterpret_cast<const uint4 *>(bits + i);
        if (i >= ncells) v.x = 0;
        if (i + 1 >= ncells) v.y = 0;
        if (i + 2 >= ncells) v.z = 0;
        if (i + 3 >= ncells) v.w = 0;
        const int a = __popc(v.x), b = a + __popc(v.y), c = b + __popc(v.z), d = c + __popc(v.w);
        const int incl = wave_incl_scan(d);
        if (__lane_id() == 63) s_sum[w] = incl;
        __syncthreads();
        int at = before + incl - d;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if (k < w) at += s_sum[k];
            before += s_sum[k];
        }
        __syncthreads();
        uint4 *out = reinterpret_cast<uint4 *>(cells + i);
        out[0] = make_uint4(v.x, (unsigned)at, v.y, (unsigned)(at + a));
        out[1] = make_uint4(v.z, (unsigned)(at + b), v.w, (unsigned)(at + c));
    }
}

// Runs: a thread per entry, which at each level stores its run's first
// position if it is the first and the end if it is the last.  Bound by the
// latency of a cell's read and the store behind it, so the levels' reads are
// issued together; blocks take entries, not rows, which hub rows make uneven
// (R-MAT 2^20
// with 8 draws a row: blocks of 512 rows 6.6 ms, of 64 rows 3.2, of entries
// 0.6).
constexpr int RUN_ENT = 512;

__global__ void __launch_bounds__(256) k_dir_runs(int n, int nnz, const int *__restrict__ ib,
                                                  const int *__restrict__ jb, int ngrp, int nblk,
                                                  int shift, int levels,
                                                  const uint2 *__restrict__ cells,
                                                  int2 *__restrict__ runs) {
    __shared__ int s_r[2];
    const int e0 = blockIdx.x * RUN_ENT, e1 = e0 + min(RUN_ENT, nnz - e0);
    if (threadIdx.x < 2) {
        // row of the block's first and last entry: the last t with ib[t] <= e
        const int e = threadIdx.x ? e1 - 1 : e0;
        s_r[threadIdx.x] = lower_bound_i32(ib, 0, n, e + 1) - 1;
    }
    __syncthreads();
    for (unsigned q = threadIdx.x; q < (unsigned)(e1 - e0); q += blockDim.x) {
        const int e = e0 + (int)q;
        const int r = lower_bound_i32(ib, s_r[0], s_r[1] + 1, e + 1) - 1;
        const int c = jb[e];
        // level-0 blocks of the entry and of its neighbours (-1: none)
        const int b = c >> shift;
        const int pb = e > ib[r] ? jb[e - 1] >> shift : -1;
        const int nb = e + 1 < ib[r + 1] ? jb[e + 1] >> shift : -1;
        const uint2 *mine = cells + (r >> 5);
        const unsigned below = (1u << (r & 31)) - 1u;
        bool first[BAND_SHIFT + 1], last[BAND_SHIFT + 1];
        uint2 w[BAND_SHIFT + 1];
#pragma unroll
        for (int v = 0; v <= BAND_SHIFT; v++) {
            first[v] = v < levels && (pb < 0 || (pb >> v) != (b >> v));
            last[v] = v < levels && (nb < 0 || (nb >> v) != (b >> v));
            w[v] = first[v] || last[v] ? mine[run_dir_block(nblk, shift, v, c) * ngrp]
                                       : make_uint2(0u, 0u);
        }
#pragma unroll
        for (int v = 0; v <= BAND_SHIFT; v++) {
            int2 *run = runs + w[v].y + __popc(w[v].x & below);
            if (first[v] && last[v])
                *run = make_int2(e, e + 1);
            else if (first[v])
                run->x = e;
            else if (last[v])
                run->y = e + 1;
        }
    }
}

// ------------------------------------------------------------- item plan
// of the sparse classes; items of more outputs are dense
constexpr int ITEM_BOUND[2] = {256, 512};
// Sparse stretches go into wide items of up to this many outputs.  R-MAT 2^20
// with 8 draws a row, both sparse kernels: 31.7 ms without wide items (its
// 30M items of <= 256 outputs hold 45 each, and each costs its A entries, two
// lookups an entry and its tables), 20.2 up to 256, 19.2 up to 384,
// 19.3 up to 512; R-MAT 2^18 with 4: 1.27, 1.01, 0.98, 0.96; ER batch of 512:
// 6.0, 5.9, 5.1, 4.3.
constexpr int WIDE_CAP = 512;
static_assert(WIDE_CAP <= ITEM_BOUND[1], "wide items run in the sparse kernels");

// Split of each big row into items: the row's span is cut into windows of
// WSB sub-blocks (at most ITEM_WBITS columns); inside a window, runs of
// sub-blocks with at most ITEM_CAP outputs, empty sub-blocks at their ends left
// out; with by_band aligned runs of 8, 4, 2 or 1 sub-blocks, which the run
// directory of B has blocks for.
// One wave per big row, one lane per window (64 windows per pass): a lane
// loads its window's counts at once and splits them in registers, and wave
// scans place the items and their outputs.  FILL=false counts items per
// row; FILL=true (item_cnt = exclusive item offsets) writes each item's
// record -- {row, c0, c1}, its first output position -- and output count, and,
// in rank mode (band_base given), where its first
// non-empty word is in the band word lists of the symbolic phase (from the
// sub-blocks' masks of non-empty words); the record's fourth field then
// holds the item's first sub-block's index in subcnt and subocc (< 2^31 in
// that mode), so the numeric phase finds the item's masks with no other
// lookup.  Windows lie inside bands, and a
// band's windows inside one pass of 64 windows, so the item's place in its
// band's list is its count of non-empty words before it less that of the
// band's first window.
// Wide items: an aligned run of 2, 4 or 8 windows of one band whose outputs
// number at most wide_cap becomes one item (the longest such run).
template <bool FILL, int WSB>
__global__ void __launch_bounds__(256) k_items(int nbig, const int *__restrict__ rows, int k,
                                               int by_band, int wide_cap,
                                               const int *__restrict__ span_sb0,
                                               const int64_t *__restrict__ sb_off,
                                               const uint16_t *__restrict__ subcnt,
                                               const int64_t *__restrict__ ic,
                                               int64_t *__restrict__ item_cnt,
                                               ItemRec *__restrict__ items,
                                               int *__restrict__ item_n,
                                               const unsigned *__restrict__ subocc,
                                               const int64_t *__restrict__ band_off,
                                               const int64_t *__restrict__ band_base) {
    static_assert(WSB <= (1 << (ITEM_WBITS_SHIFT - SUB_SHIFT)), "item wider than its LDS");
    constexpr int WPB = (1 << BAND_SHIFT) / WSB;   // windows per band
    static_assert(WPB * WSB == (1 << BAND_SHIFT) && 64 % WPB == 0, "windows tile the bands");
    const bool words = band_base != nullptr;   // rank mode: word-list positions
    const int r = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int l = threadIdx.x & 63;
    if (r >= nbig) return;
    const int row = rows[r];
    const uint16_t *sc = subcnt + sb_off[r];
    const int nsb = (int)(sb_off[r + 1] - sb_off[r]);
    // windows are cut from the first band's start with by_band
    const int lead = by_band ? band_lead(span_sb0[r]) : 0;
    const int first = span_sb0[r];
    const int nwin = (lead + nsb + WSB - 1) / WSB;
    int64_t wbase = FILL ? item_cnt[r] : 0;
    int64_t obase = FILL ? ic[row] : 0;
    for (int w0 = 0; w0 < nwin; w0 += 64) {
        const int win = w0 + l;
        const int j0 = win * WSB - lead;
        const int len = win < nwin ? min(WSB, nsb - j0) : 0;
        int cs[WSB], os[WSB];
        int nzt = 0;
#pragma unroll
        for (int q = 0; q < WSB; q++) {
            const bool in = q < len && j0 + q >= 0;
            cs[q] = in ? (int)sc[j0 + q] : 0;
            os[q] = FILL && words && in ? __popc(subocc[sb_off[r] + j0 + q]) : 0;
            nzt += os[q];
        }
        int nit = 0, tot = 0, firstq = WSB, lastq = -1;
#pragma unroll
        for (int q = 0; q < WSB; q++) {
            tot += cs[q];
            if (cs[q] != 0) {
                firstq = min(firstq, q);
                lastq = q;
            }
        }
        // ends[q]: an item ends with sub-block q
        bool ends[WSB];
        if (by_band) {
            // halves, quarters, ... until a part has at most ITEM_CAP outputs
            int part[WSB];
#pragma unroll
            for (int q = 0; q < WSB; q++) {
                part[q] = cs[q];
                ends[q] = true;
            }
#pragma unroll
            for (int z = 2; z <= WSB; z <<= 1) {
#pragma unroll
                for (int q = 0; q < WSB; q += z) {
                    // both halves are whole (their sums fit) and so is the sum
                    part[q] += part[q + z / 2];
                    ends[q + z / 2 - 1] = part[q] > ITEM_CAP;
                }
            }
        } else {
            int cnt = 0;
#pragma unroll
            for (int q = 0; q < WSB; q++) {
                cnt += cs[q];
                ends[q] = q + 1 == WSB || cnt + cs[q + 1 < WSB ? q + 1 : q] > ITEM_CAP;
                if (ends[q]) cnt = 0;
            }
        }
        {
            int cnt = 0;
#pragma unroll
            for (int q = 0; q < WSB; q++) {
                cnt += cs[q];
                if (ends[q]) {
                    nit += cnt > 0;
                    cnt = 0;
                }
            }
        }
        // the run of windows this one is in: its length, outputs, first and
        // last sub-block with outputs
        int run = 1, run_tot = tot;
        int sb_first = lastq >= 0 ? j0 + firstq : 0x7fffffff;
        int sb_last = lastq >= 0 ? j0 + lastq : -1;
        {
            int g_tot = tot, g_first = sb_first, g_last = sb_last;
#pragma unroll
            for (int g = 2; g <= WPB; g <<= 1) {
                g_tot += __shfl_xor(g_tot, g >> 1, 64);
                g_first = min(g_first, __shfl_xor(g_first, g >> 1, 64));
                g_last = max(g_last, __shfl_xor(g_last, g >> 1, 64));
                if (g_tot <= wide_cap) {
                    run = g;
                    run_tot = g_tot;
                    sb_first = g_first;
                    sb_last = g_last;
                }
            }
        }
        if (run > 1) nit = (l & (run - 1)) == 0 && run_tot > 0 ? 1 : 0;
        const int it_incl = wave_incl_scan(nit);
        const int out_incl = wave_incl_scan(tot);
        // non-empty words of this pass before this window, and before the
        // first window of this lane's band
        const int nz_excl = FILL ? wave_incl_scan(nzt) - nzt : 0;
        const int band_nz = FILL ? __shfl(nz_excl, (l / WPB) * WPB, 64) : 0;
        if (FILL && nit > 0) {
            int64_t w = wbase + it_incl - nit;
            int64_t out = obase + out_incl - tot;
            const int cbase = first + j0;
            // this window's first non-empty word in the band word lists
            const int64_t wb =
                words ? band_base[band_off[r] + win / WPB] + (nz_excl - band_nz) : 0;
            if (run > 1) {
                items[w] = ItemRec{make_int4(row, (first + sb_first) << SUB_SHIFT,
                                             sub_block_start(first + sb_last + 1, k),
                                             words ? (int)(sb_off[r] + sb_first) : 0),
                                   out, wb};
                item_n[w] = run_tot;
            }
            // an item's columns: from its first sub-block with outputs to its last
            int start = -1, stop = 0, cnt = 0, nzrun = 0, nzs = 0;
#pragma unroll
            for (int q = 0; q < WSB; q++) {
                if (run > 1) break;
                if (cs[q] != 0) {
                    if (start < 0) {
                        start = q;
                        nzs = nzrun;
                    }
                    stop = q + 1;
                    cnt += cs[q];
                }
                nzrun += os[q];
                if (ends[q] && cnt > 0) {
                    items[w] = ItemRec{make_int4(row, (cbase + start) << SUB_SHIFT,
                                                 sub_block_start(cbase + stop, k),
                                                 words ? (int)(sb_off[r] + j0 + start) : 0),
                                       out, wb + nzs};
                    item_n[w] = cnt;
                    w++;
                    out += cnt;
                    start = -1;
                    cnt = 0;
                }
            }
        }
        wbase += group_last<64>(it_incl);
        obase += group_last<64>(out_incl);
    }
    if (!FILL && l == 0) item_cnt[r] = wbase;
}

// Items in order of their first column: keys, then the gather of the items
// and their output offsets into the sorted order.  The numeric phase takes
// items in this order, so the items in flight at any time gather B entries
// of one narrow column band, which the L2 caches keep, instead of bands
// spread over all of B.
// Items sort by size class (ITEM_BOUND), then by first column, after those of
// rows of LONG_ROW entries or more: an item is one wave's work, so a class ends
// no sooner than its longest item, which had better start first (R-MAT 2^18
// times its transpose, items of <= 512 outputs 0.69 -> 0.56 ms; its numeric
// phase at LONG_ROW 256, 1024 and 4096 1.44, 1.43 and 1.49 ms, 1.57 without).
// key = class << class_bit + 1 | 1 << class_bit | first sub-block (a long
// row's without the 1; class_bit < 0: the sub-block only).  The numeric phase
// runs each class with tables that hold just that class's items: the waves an
// LDS holds set its speed.  Class 1 is the dense one.  R-MAT 2^20 with 8 draws a row: <= 256
// outputs 5.8 -> 4.2 ms (4 batches in flight, 8 waves per SIMD; 6 batches: 4.7),
// <= 512 12.8 -> 11.8 (at 4 waves).  Finer classes gained nothing there (384:
// 4.2 + 7.5 ms; 768: 7.8 + 7.9 against 15.9) and cost R-MAT 2^18 a tail each.
// class_cnt counts the items of each class but the last.
__global__ void __launch_bounds__(256) k_item_keys(int64_t n, const ItemRec *__restrict__ items,
                                                   const int *__restrict__ item_n,
                                                   const int *__restrict__ ia, int class_bit,
                                                   int *__restrict__ keys,
                                                   unsigned long long *__restrict__ class_cnt) {
    constexpr int PER = 16, LONG_ROW = 1024;
    __shared__ int s_cnt[ITEM_CLASSES - 1];
    if (threadIdx.x < ITEM_CLASSES - 1) s_cnt[threadIdx.x] = 0;
    __syncthreads();
    int cnt[ITEM_CLASSES - 1] = {};
    for (int q = 0; q < PER; q++) {
        const int64_t i = ((int64_t)blockIdx.x * PER + q) * 256 + threadIdx.x;
        int cls = ITEM_CLASSES - 1;
        if (i < n) {
            if (class_bit >= 0) {
                const int outputs = item_n[i];
                cls = outputs <= ITEM_BOUND[0] ? 0 : outputs > ITEM_BOUND[1] ? 1 : 2;
            }
            const int4 d = items[i].d;
            int key = d.y >> SUB_SHIFT;
            if (class_bit >= 0) {
                const bool other = ia[d.x + 1] - ia[d.x] < LONG_ROW;
                key |= (2 * cls + (other ? 1 : 0)) << class_bit;
            }
            keys[i] = key;
        }
#pragma unroll
        for (int c = 0; c < ITEM_CLASSES - 1; c++) cnt[c] += __popcll(__ballot(cls == c));
    }
    if (__lane_id() == 0)
        for (int c = 0; c < ITEM_CLASSES - 1; c++) atomicAdd(&s_cnt[c], cnt[c]);
    __syncthreads();
    if (threadIdx.x < ITEM_CLASSES - 1 && s_cnt[threadIdx.x])
        atomicAdd(class_cnt + threadIdx.x, (unsigned long long)s_cnt[threadIdx.x]);
}

__global__ void __launch_bounds__(256) k_gather_items(int64_t n, const int *__restrict__ order,
                                                      const ItemRec *__restrict__ items,
                                                      ItemRec *__restrict__ items_out) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j < n) items_out[j] = items[order[j]];
}

// --------------------------------------------------------- big rows: numeric
// One wave per item (grid-stride over items).  LDS per wave: a key hash with
// a 16-bit id per slot, values compacted by insertion id (only the item's
// <= ITEM_CAP outputs are stored), the item's column bitmap (emission order)
// and the tag table of the ordered accumulation.
struct ItemSmem {
    double vals[ITEM_CAP];
    int keys[ITEM_SLOTS];
    unsigned short ids[ITEM_SLOTS];
    unsigned bits[ITEM_WORDS];
    unsigned tags[ITEM_TAGS];
    int heads[64];                // start bits of the product expansion
    int nid;
};

template <bool FUSED, bool DIR>
__global__ void __launch_bounds__(64 * ITEM_WAVES) k_big_numeric(
    int64_t nitems, const ItemRec *__restrict__ items,
    const int *__restrict__ ia, const int *__restrict__ ja, const double *__restrict__ a,
    const int *__restrict__ jb, const double *__restrict__ b, BRows brows, int *__restrict__ jc,
    double *__restrict__ c, int b_strict) {
    extern __shared__ __align__(16) unsigned char smem[];
    ItemSmem &S = reinterpret_cast<ItemSmem *>(smem)[threadIdx.x >> 6];
    const int l = __lane_id();
    for (int i = l; i < ITEM_TAGS; i += 64) S.tags[i] = 0xffffffffu;
    const int64_t wave_id = (int64_t)blockIdx.x * ITEM_WAVES + (threadIdx.x >> 6);
    const int64_t nwaves = (int64_t)gridDim.x * ITEM_WAVES;
    for (int64_t it = wave_id; it < nitems; it += nwaves) {
        const int4 item = items[it].d;
        const int row = item.x, c0 = item.y, c1 = item.z;
        const int nwords = (c1 - c0 + 31) >> 5;
        for (int i = l; i < ITEM_SLOTS; i += 64) S.keys[i] = -1;
        for (int i = l; i < nwords; i += 64) S.bits[i] = 0u;
        if (l == 0) S.nid = 0;
        wave_lds_fence();
        for_products<ITEM_U, 1, true>(
            ia[row], ia[row + 1], ja, a, ItemRange<DIR>(brows, jb, c0, c1), jb, b, S.heads,
            [&](const Batch &t) {
                int slot = -1;
                if (t.act) {
                    bool created;
                    slot = hash_insert<ITEM_SLOTS>(S.keys, t.col, created);
                    if (created) {
                        const int id = atomicAdd(&S.nid, 1);
                        S.ids[slot] = (unsigned short)id;
                        S.vals[id] = 0.0;
                        const int cc = t.col - c0;
                        atomicOr(&S.bits[cc >> 5], 1u << (cc & 31));
                    }
                }
                wave_lds_fence();
                const int id = slot >= 0 ? (int)S.ids[slot] : -1;
                ordered_accumulate<FUSED, ITEM_TAGS>(t.act, id, t.a, t.b, S.vals, S.tags,
                                                     (unsigned)l, t.nseg == 1 && b_strict);
            });
        wave_lds_fence();
        // emit in column order: bitmap words -> ranks -> hash lookups
        int64_t o = items[it].off;
        for (int w0 = 0; w0 < nwords; w0 += 64) {
            const int w = w0 + l;
            unsigned word = w < nwords ? S.bits[w] : 0u;
            const int pc = __popc(word);
            const int incl = wave_incl_scan(pc);
            int64_t pos = o + incl - pc;
            while (word) {
                const int bit = __ffs(word) - 1;
                word &= word - 1;
                const int col = c0 + (w << 5) + bit;
                const int slot = hash_find<ITEM_SLOTS>(S.keys, col);
                jc[pos] = col;
                c[pos] = slot >= 0 ? S.vals[S.ids[slot]] : 0.0;
                pos++;
            }
            o += __shfl(incl, 63, 64);
        }
        wave_lds_fence();
    }
}

// Entries of a batch added one after the other.  Numeric phase at 4, 8 and 16:
// ER 65536 with 24 a row, all rows big, 691, 685 and 766 us; R-MAT 2^16 with 8
// draws a row 1.39, 1.26 and 1.20 ms, 2^20 31.6, 31.7 and 32.6 ms.
constexpr int RANK_SEGS = 8;
constexpr int RANK_TAGS = 128;         // tag buckets of the rank-indexed kernel

// Rank-indexed variant: the symbolic phase stored every big row's column
// bitmap (in sparse form: per sub-block a mask of its non-empty words, and
// those words), so an item's outputs are known before its products are
// visited.  The rank of column j inside the item is pre[w] + popc(bits[w]
// below j), and values accumulate
// in a dense rank-ordered array that is written out coalesced.
// WORDS: bitmap words of the widest item (256 or 512: items of 8192 or
// 16384 columns).
// 10048 bytes at 8192 columns: 16 waves a CU.  Their number sets the kernel's
// speed, the latency of a group's loads and LDS turns its bound: R-MAT 2^20
// with 8 draws a row, 26.8 ms at 10 waves, 22.5 at 12, 18.6 at 14 (pairs of
// words and prefixes, 256 tags), 16.5 now, with both reads of a tag round in
// one wait.
template <int WORDS>
struct RankSmem {
    double vals[ITEM_CAP];
    uint2 bits[WORDS / 2];        // 64 columns each
    uint16_t pre[WORDS / 2];      // outputs before them
    unsigned tags[RANK_TAGS];     // bucketed by rank
    int heads[2 * RANK_U];        // start bits of the product expansion
};

// Rank table of one item, in two parts so that other loads can be issued
// between them: item_words loads the item's bitmap words (<= ITEM_WORDS,
// every load issued before the first is used); item_rank_build clears bits
// at or past c1, stores {word, outputs before it} pairs in S.words, writes
// the item's columns to jc at offset o (expanded into S.vals, then stored
// coalesced; the stores drain while the products are processed), zeroes the
// item's first cnt values and returns cnt, the item's output count.
// item_words rebuilds the words from the band word list: lane l takes words
// l, l + 64, ..., and word w of sub-block s (lanes 0..15 of occ hold the
// item's sub-block masks, of pre their exclusive popcount prefix) is there
// when its bit of occ[s] is set, at list + pre[s] + popc(occ[s] below it).
template <int WCH>
__device__ __forceinline__ void item_words(const unsigned *__restrict__ list, unsigned occ,
                                           int pre, int c0, int c1, unsigned (&wv)[WCH]) {
    static_assert(2 * WCH <= 16, "an item's sub-block masks sit in lanes 0..15");
    const int l = __lane_id();
    const int nwords = (c1 - c0 + 31) >> 5;
    const unsigned below = (1u << (l & 31)) - 1u;
#pragma unroll
    for (int j = 0; j < WCH; j++) {
        const int w = j * 64 + l;
        // word w is in sub-block 2j (lanes 0..31) or 2j + 1 (lanes 32..63)
        const unsigned o0 = __builtin_amdgcn_readlane(occ, 2 * j);
        const unsigned o1 = __builtin_amdgcn_readlane(occ, 2 * j + 1);
        const int p0 = __builtin_amdgcn_readlane(pre, 2 * j);
        const int p1 = __builtin_amdgcn_readlane(pre, 2 * j + 1);
        const unsigned om = l < 32 ? o0 : o1;
        const int pm = l < 32 ? p0 : p1;
        const bool present = w < nwords && ((om >> (l & 31)) & 1u);
        // read once: a streaming load keeps the L2 for B's rows.  A 32-bit
        // offset from the wave's scalar base keeps one address register
        // per load
        const unsigned off = (unsigned)pm + (unsigned)__popc(om & below);
        wv[j] = present ? __builtin_nontemporal_load(list + off) : 0u;
    }
}

template <int WORDS, int WCH = WORDS / 64>
__device__ __forceinline__ int item_rank_build(RankSmem<WORDS> &S, unsigned (&wv)[WCH],
                                               int c0, int c1, int64_t o, int *__restrict__ jc) {
    const int l = __lane_id();
    const int nwords = (c1 - c0 + 31) >> 5;
    // the 64-word chunks are scanned independently
    int incl[WCH], tot[WCH];
#pragma unroll
    for (int j = 0; j < WCH; j++) {
        const int w = j * 64 + l;
        const int lastbits = (c1 - c0) - (w << 5);
        if (w < nwords && lastbits < 32) wv[j] &= (1u << lastbits) - 1u;
        incl[j] = wave_incl_scan(__popc(wv[j]));
        tot[j] = group_last<64>(incl[j]);
    }
    int cnt = 0;
    int *cols = reinterpret_cast<int *>(S.vals);
#pragma unroll
    for (int j = 0; j < WCH; j++) {
        const int w = j * 64 + l;
        const int base = cnt + incl[j] - __popc(wv[j]);
        if (w < nwords) {
            reinterpret_cast<unsigned *>(S.bits)[w] = wv[j];
            if (!(w & 1)) S.pre[w >> 1] = (uint16_t)base;
        }
        unsigned word = wv[j];
        int pos = base;
        while (word) {
            const int bit = __ffs(word) - 1;
            word &= word - 1;
            cols[pos++] = c0 + (w << 5) + bit;
        }
        cnt += tot[j];
    }
    wave_lds_fence();
    for (int i = l; i < cnt; i += 64) __builtin_nontemporal_store(cols[i], jc + o + i);
    wave_lds_fence();
    for (int i = l; i < cnt; i += 64) S.vals[i] = 0.0;
    wave_lds_fence();
    return cnt;
}

// Accumulates one batch of products into the item's rank-ordered values:
// a batch from one A entry (distinct columns when B's rows are strictly
// ascending) adds directly, one from a few A entries one entry after the
// other, any other by tag rounds in lane order.
template <bool FUSED, int WORDS>
__device__ __forceinline__ void item_accumulate(RankSmem<WORDS> &S, int c0, const Batch &t,
                                                int b_strict) {
    int rank = -1;
    if (t.act) {
        const int cc = t.col - c0;
        const uint2 wd = S.bits[cc >> 6];
        const unsigned below = (1u << (cc & 31)) - 1u;
        rank = (int)S.pre[cc >> 6] + __popc(wd.x & (cc & 32 ? ~0u : below)) +
               __popc(wd.y & (cc & 32 ? below : 0u));
    }
    if (b_strict && t.nseg <= RANK_SEGS) {
        for (int s = 1; s <= t.nseg; s++) {
            if (rank >= 0 && t.seg == s) S.vals[rank] = acc_step<FUSED>(S.vals[rank], t.a, t.b);
            wave_lds_fence();
        }
        return;
    }
    ordered_accumulate<FUSED, RANK_TAGS>(rank >= 0, rank, t.a, t.b, S.vals, S.tags,
                                         (unsigned)__lane_id(), false);
}

// What the item kernels work on, but for the items.
struct ItemArgs {
    const unsigned *wlist, *subocc;
    const int *ia, *ja;
    const double *a;
    const int *jb;
    const int4 *bpk;
    int *jc;
    double *c;
    int b_strict;
};

template <bool FUSED, int WORDS, bool DIR>
__device__ __forceinline__ void dense_item(RankSmem<WORDS> &S, const ItemRec &rec,
                                           const ItemArgs &T, const BRows &brows) {
    const int l = __lane_id();
    for (int i = l; i < RANK_TAGS; i += 64) S.tags[i] = 0xffffffffu;
    const int4 item = rec.d;
    const int64_t o = rec.off;
    const unsigned *list = T.wlist + rec.wpos;
    const int c0 = item.y, c1 = item.z;
    // the rank table is built after the first groups' A entries and cells are
    // issued, so the word loads and that chain of loads overlap
    const ItemRange<DIR> range(brows, T.jb, c0, c1);
    EntryPipe<true, 1> pipe;
    pipe.ja = T.ja;
    pipe.aval = T.a;
    pipe.part = 0;
    pipe.load(T.ia[item.x], T.ia[item.x + 1]);
    // item.w: the item's first sub-block in subocc
    const int nsb = min((c1 - c0 + (1 << SUB_SHIFT) - 1) >> SUB_SHIFT, 2 * (WORDS / 64));
    const unsigned occ = l < nsb ? T.subocc[(int64_t)item.w + l] : 0u;
    pipe.cells(range);
    const int pc = __popc(occ);
    const int pre = dpp_incl_scan<16>(pc) - pc;
    unsigned wv[WORDS / 64];
    item_words(list, occ, pre, c0, c1, wv);
    pipe.first(range);
    const int cnt = item_rank_build(S, wv, c0, c1, o, T.jc);
    auto f = [&](const Batch &t) { item_accumulate<FUSED>(S, c0, t, T.b_strict); };
    for (unsigned g = pipe.pa; g < pipe.pe; g += 64) {
        pipe.ahead(g, range);
        expand_group<RANK_U, true, true>(pipe.lo, max(pipe.hi - pipe.lo, 0), pipe.a, T.jb, nullptr,
                                         S.heads, f, T.bpk);
        pipe.take();
    }
    wave_lds_fence();
    for (int i = l; i < cnt; i += 64) __builtin_nontemporal_store(S.vals[i], T.c + o + i);
    wave_lds_fence();
}

// Items of at most CAP outputs, however wide up to a band: the rank of a
// column goes through the item's sub-blocks (mask of non-empty words, words
// before it) to its word (bits, outputs before it), so table and work follow
// the outputs and not the columns.  The outputs' columns are noted by the
// products (as offsets in the item) instead of expanded from the words.
//
// The dense tables it replaces for these items cost ~500 vector instructions
// an item whatever its products (the issue rate bound them: 25 of 29 ms of
// R-MAT 2^20 with 8 draws a row); with the sparse tables those and the items of
// 257..512 outputs went from 37.7 to 18.5 ms, and to 16.0 with the run directory
// and tables of half the size.  Bound by latency, so by the waves an LDS holds.
// Larger items keep the dense table: one lookup a product.
template <int CAP, int U>
struct SparseSmem {
    double vals[CAP];
    unsigned words[CAP];          // the item's words
    uint16_t pre[CAP];            // outputs before them
    uint2 sub[1 << BAND_SHIFT];   // {mask of non-empty words, words before}
    uint16_t cols[CAP];
    unsigned tags[CAP / 4];       // a byte per output, or tag buckets
    int heads[2 * U];
};

template <bool FUSED, int CAP, int U, bool DIR>
__device__ __forceinline__ void sparse_item(SparseSmem<CAP, U> &S, const ItemRec &rec,
                                            const ItemArgs &T, const BRows &brows) {
    constexpr int NT = CAP / 4;
    const int l = __lane_id();
    uint8_t *own = reinterpret_cast<uint8_t *>(S.tags);
    const int4 item = rec.d;
    const int64_t o = rec.off;
    const unsigned *list = T.wlist + rec.wpos;
    const int c0 = item.y, c1 = item.z;
    const ItemRange<DIR> range(brows, T.jb, c0, c1);
    EntryPipe<true, 1> pipe;
    pipe.ja = T.ja;
    pipe.aval = T.a;
    pipe.part = 0;
    pipe.load(T.ia[item.x], T.ia[item.x + 1]);
    const int nsb = min((c1 - c0 + (1 << SUB_SHIFT) - 1) >> SUB_SHIFT, 1 << BAND_SHIFT);
    const unsigned occ = l < nsb ? T.subocc[(int64_t)item.w + l] : 0u;
    pipe.cells(range);
    const int pc = __popc(occ);
    const int incl = wave_incl_scan(pc);
    // every non-empty word has an output
    const int nw = min(__builtin_amdgcn_readlane(incl, 63), CAP);
    unsigned wv[CAP / 64];
#pragma unroll
    for (int j = 0; j < CAP / 64; j++)
        wv[j] = j * 64 + l < nw ? __builtin_nontemporal_load(list + j * 64 + l) : 0u;
    pipe.first(range);
    S.sub[l] = make_uint2(occ, (unsigned)(incl - pc));
    int cnt = 0;
#pragma unroll
    for (int j = 0; j < CAP / 64; j++) {
        if (j * 64 < nw) {
            const int p = __popc(wv[j]);
            const int in = wave_incl_scan(p);
            if (j * 64 + l < nw) {
                S.words[j * 64 + l] = wv[j];
                S.pre[j * 64 + l] = (uint16_t)(cnt + in - p);
            }
            cnt += __builtin_amdgcn_readlane(in, 63);
        }
    }
    cnt = min(cnt, CAP);
    for (int i = l; i < cnt; i += 64) S.vals[i] = 0.0;
    wave_lds_fence();
    auto f = [&](const Batch &t) {
        int rank = -1;
        if (t.act) {
            const int cc = t.col - c0;
            const uint2 sb = S.sub[(cc >> SUB_SHIFT) & ((1 << BAND_SHIFT) - 1)];
            const int w = min(
                (int)sb.y + (int)__popc(sb.x & ((1u << ((cc >> 5) & 31)) - 1u)), CAP - 1);
            rank = min((int)S.pre[w] + (int)__popc(S.words[w] & ((1u << (cc & 31)) - 1u)),
                       CAP - 1);
            S.cols[rank] = (uint16_t)cc;
        }
        bool clash = t.nseg > 1 || !T.b_strict;
        if (T.b_strict && t.nseg > 2) {
            if (t.act) own[rank] = (uint8_t)l;
            wave_lds_fence();
            clash = __ballot(t.act && own[rank] != (uint8_t)l) != 0;
            wave_lds_fence();
        }
        if (!clash) {
            if (t.act) S.vals[rank] = acc_step<FUSED>(S.vals[rank], t.a, t.b);
            wave_lds_fence();
        } else if (T.b_strict && t.nseg <= FLAT_SEGS) {
            for (int s = 1; s <= t.nseg; s++) {
                if (t.act && t.seg == s) S.vals[rank] = acc_step<FUSED>(S.vals[rank], t.a, t.b);
                wave_lds_fence();
            }
        } else {
            for (int i = l; i < NT; i += 64) S.tags[i] = 0xffffffffu;
            wave_lds_fence();
            ordered_accumulate<FUSED, NT>(t.act, rank, t.a, t.b, S.vals, S.tags, (unsigned)l,
                                          false);
        }
    };
    for (unsigned g = pipe.pa; g < pipe.pe; g += 64) {
        pipe.ahead(g, range);
        expand_group<U, true, true>(pipe.lo, max(pipe.hi - pipe.lo, 0), pipe.a, T.jb, nullptr,
                                    S.heads, f, T.bpk);
        pipe.take();
    }
    wave_lds_fence();
    for (int i = l; i < cnt; i += 64) {
        __builtin_nontemporal_store(c0 + (int)S.cols[i], T.jc + o + i);
        __builtin_nontemporal_store(S.vals[i], T.c + o + i);
    }
    wave_lds_fence();
}

// The items of at most 256 outputs: 32 waves a CU.
template <bool FUSED, bool DIR>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(8))) k_big_numeric_small(
    int64_t nitems, const ItemRec *__restrict__ items, ItemArgs T, BRows brows) {
    __shared__ __align__(16) SparseSmem<ITEM_BOUND[0], 4> S;
    for (int64_t it = blockIdx.x; it < nitems; it += gridDim.x)
        sparse_item<FUSED, ITEM_BOUND[0], 4, DIR>(S, items[it], T, brows);
}

// The others, the first ndense in dense tables (all items in rows' order): in
// one launch, so the other class runs beside the longest items, which a wave
// each works on for most of a small product's time (R-MAT 2^18 with 4, times
// its transpose: 0.91 + 0.54 ms in two launches, 1.03 in one; R-MAT 2^20 with 8
// draws a row 27.1 ms either way).  Teams of 2 to 4 waves on an item, in turns
// by group of A entries, took 1.2 to 2 times as long: the turns are most of a
// group's time.
template <bool FUSED, int WORDS, bool DIR>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4))) k_big_numeric_rank(
    int64_t nitems, int64_t ndense, const ItemRec *__restrict__ items, ItemArgs T, BRows brows) {
    union Smem {
        RankSmem<WORDS> dense;
        SparseSmem<ITEM_BOUND[1], 6> sparse;
    };
    __shared__ __align__(16) Smem S;
    for (int64_t it = blockIdx.x; it < nitems; it += gridDim.x) {
        if (it < ndense)
            dense_item<FUSED, WORDS, DIR>(S.dense, items[it], T, brows);
        else
            sparse_item<FUSED, ITEM_BOUND[1], 6, DIR>(S.sparse, items[it], T, brows);
    }
}

// B's entries as 16-byte {column, 0, value lo, value hi} records for the
// big-row numeric kernel's gathers.
__global__ void __launch_bounds__(256) k_pack_b(int64_t nnz, const int *__restrict__ jb,
                                                const double *__restrict__ b,
                                                int4 *__restrict__ bpk) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= nnz) return;
    const double v = b[q];
    bpk[q] = make_int4(jb[q], 0, __double2loint(v), __double2hiint(v));
}

// The same for the B rows that big rows name (rows named more than once are
// written with the same records): with few big rows that is less than all of
// B.  A block takes PACK_ENT of the big rows' A entries, whichever rows they
// are of (ent_off: entries of the rows before each), and blockIdx.y its share
// of their B entries, flat, so neither a long row of A nor long B rows are one
// wave's work (a wave per big row took 25 ms for one of 50,000 entries).
//
// All of B takes 4.3 ps an entry, named rows 1.2 to 2 ns an A entry as they
// lie apart, from 5 us up: 7.4M entries of B 32 us, or 5 us with 1000 A entries,
// 20 with 16,000, 103 with 50,000; 32.5M entries 136 us, or 62 with 50,000; ER
// batch of 512 matrices 670 us, or 32.
constexpr int PACK_ENT = 64, PACK_ENT_COST = 256, PACK_PROD_COST = 4;

__global__ void __launch_bounds__(256) k_pack_rows(int64_t nent, int nbig,
                                                   const int64_t *__restrict__ ent_off,
                                                   const int *__restrict__ rows,
                                                   const int *__restrict__ ia,
                                                   const int *__restrict__ ja,
                                                   const int *__restrict__ ib,
                                                   const int *__restrict__ jb,
                                                   const double *__restrict__ b,
                                                   int4 *__restrict__ bpk) {
    __shared__ int s_end[PACK_ENT], s_first[PACK_ENT];
    static_assert(PACK_ENT == 64, "a lane per entry");
    if (threadIdx.x < PACK_ENT) {
        const int64_t e = (int64_t)blockIdx.x * PACK_ENT + threadIdx.x;
        int lo = 0, cnt = 0;
        if (e < nent) {
            int r = 0, hi = nbig;              // ent_off[r] <= e < ent_off[hi]
            while (hi - r > 1) {
                const int mid = r + ((hi - r) >> 1);
                if (ent_off[mid] <= e) r = mid;
                else hi = mid;
            }
            const int row = rows[r], p = ia[row] + (int)(e - ent_off[r]);
            if (p < ia[row + 1]) {
                const int t = ja[p];
                lo = ib[t];
                cnt = max(ib[t + 1] - lo, 0);
            }
        }
        const int incl = wave_incl_scan(cnt);
        s_end[threadIdx.x] = incl;
        s_first[threadIdx.x] = lo - (incl - cnt);
    }
    __syncthreads();
    const unsigned total = (unsigned)s_end[PACK_ENT - 1];
    for (unsigned q = blockIdx.y * 256 + threadIdx.x; q < total; q += gridDim.y * 256) {
        int i = 0;                             // the first entry that ends past q
#pragma unroll
        for (int z = PACK_ENT / 2; z > 0; z >>= 1)
            if ((unsigned)s_end[i + z - 1] <= q) i += z;
        const int p = s_first[i] + (int)q;
        const double v = b[p];
        bpk[p] = make_int4(jb[p], 0, __double2loint(v), __double2hiint(v));
    }
}

// The plan's run directory or block pointers; without either, B's row pointers
// b_ptr (of the call at hand) as a one-block table.
static BRows b_rows(const RowPlan &p, const int *b_ptr) {
    BRows r;
    r.dir = p.dir;
    r.bp.p = p.bptr ? p.bptr : b_ptr;
    r.bp.tstride = p.bptr ? p.nblk + 1 : 1;
    r.bp.bs = p.bptr ? p.blk_shift : 30;
    return r;
}

// One block per item (the hardware dispatcher hands the next item to
// whichever CU frees a slot first, so no CU idles behind a long tail); the
// item kernels keep a grid-stride loop for item counts beyond the grid limit.
static unsigned item_grid(int64_t nitems) {
    return grid_for((size_t)nitems, ITEM_WAVES, MAX_GRID * 4 / ITEM_WAVES);
}

// Raises a kernel's dynamic LDS limit once per process (later calls, e.g.
// inside a captured numeric phase, touch no runtime state).
template <class K>
void set_smem(K kernel, size_t bytes) {
    static std::mutex mu;
    static std::map<const void *, size_t> done;
    const void *key = reinterpret_cast<const void *>(kernel);
    std::lock_guard<std::mutex> lk(mu);
    auto it = done.find(key);
    if (it != done.end() && it->second >= bytes) return;
    TSG_HIP_TRY(hipFuncSetAttribute(key, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
    done[key] = bytes;
}

}  // namespace

// =================================================================== host
void row_symbolic(RowPlan &p, const CsrIn &A, const CsrIn &B, int64_t *d_ic, int64_t *nnz_c,
                  const RowFront &front, HostBox *box, Arena &ws, hipStream_t s, StageTimer &tm,
                  const RowTuning &tune) {
    const int m = A.rows, n = A.cols, k = B.cols;
    TSG_CHECK(tune.bin1 >= 0 && tune.bin1 <= 64 && tune.bin1 <= tune.bin2 && tune.bin2 <= 256 &&
                  tune.bin2 <= tune.bin3 && tune.bin3 <= ROW_SMALL_PROD,
              TSG_ERR_INVALID, "row bins out of range");
    p = RowPlan();
    p.m = m;
    p.n = n;
    p.k = k;
    p.front = front;
    int64_t *scan_tmp = ws.alloc_n<int64_t>(scan_tmp_elems((size_t)m + 1));

    // small rows
    tm.begin("row.small_symbolic");
    {
        auto launch = [&](auto kern, int rpb, int threads, int bin) {
            in_launches(front.count[bin], rpb, threads, [&](int64_t r0, int nr) {
                hipLaunchKernelGGL(kern, dim3(grid_for(nr, rpb)), dim3(threads), 0, s, nr,
                                   front.rows(bin) + r0, A.ptr, A.idx, B.ptr, B.idx, front.rownnz);
                TSG_LAUNCH_CHECK();
            });
        };
        launch(k_flat_symbolic<16, 4, 64, 64, 256>, 16, 256, 1);
        launch(k_flat_symbolic<64, 4, 64, 512, 64>, 1, 64, 2);
        launch(k_flat_symbolic<64, 8, 64, 512, 64>, 1, 64, 3);
        launch(k_flat_symbolic<64, 16, 64, 512, 64, 6>, 1, 64, 4);
        launch(k_flat_symbolic<64, 16, 1024, 512, 64>, 1, 64, ROW_BIN_MANY);
        launch(k_flat_symbolic<64, 24, 64, 512, 64>, 1, 64, ROW_BIN_MED);
    }
    tm.end();

    // big rows
    p.nbig = front.count[ROW_BIN_BIG];
    int64_t *band_off = nullptr, *band_base = nullptr, *row_loff = nullptr;
    unsigned long long *row_cur = nullptr;
    int64_t *d_overflow = nullptr;
    if (p.nbig > 0) {
        const int *rowsb = front.rows(ROW_BIN_BIG);
        tm.begin("row.big_symbolic");
        // column span of every big row, in sub-blocks, span offsets and the
        // band units over the spans
        p.span_sb0 = ws.alloc_n<int>((size_t)p.nbig + 1);
        p.sb_off = ws.alloc_n<int64_t>((size_t)p.nbig + 1);
        band_off = ws.alloc_n<int64_t>((size_t)p.nbig + 1);
        int64_t *tmp_sb = ws.alloc_n<int64_t>(scan_tmp_elems((size_t)p.nbig + 1));
        int64_t *a_ent = p.ent_off = ws.alloc_n<int64_t>((size_t)p.nbig + 1);
        int64_t *a_prod = ws.alloc_n<int64_t>((size_t)p.nbig + 1);
        row_loff = ws.alloc_n<int64_t>((size_t)p.nbig + 1);
        hipLaunchKernelGGL(k_big_span, dim3(grid_for((size_t)p.nbig, 4, MAX_GRID)), dim3(256), 0, s,
                           p.nbig, rowsb, A.ptr, A.idx, B.ptr, B.idx, front.rowprod, p.span_sb0,
                           p.sb_off, a_ent, a_prod, row_loff);
        TSG_LAUNCH_CHECK();
        exclusive_scan_i64(p.sb_off, p.sb_off, (size_t)p.nbig, tmp_sb, s);
        hipLaunchKernelGGL(k_band_count, dim3(grid_for((size_t)p.nbig, 256)), dim3(256), 0, s,
                           p.nbig, tune.item_sort_min, p.span_sb0, p.sb_off, band_off);
        TSG_LAUNCH_CHECK();
        exclusive_scan_i64(band_off, band_off, (size_t)p.nbig, tmp_sb, s);
        exclusive_scan_i64(a_ent, a_ent, (size_t)p.nbig, tmp_sb, s);
        exclusive_scan_i64(a_prod, a_prod, (size_t)p.nbig, tmp_sb, s);
        exclusive_scan_i64(row_loff, row_loff, (size_t)p.nbig, tmp_sb, s);
        publish_i64({{p.sb_off + p.nbig, band_off + p.nbig, a_ent + p.nbig, a_prod + p.nbig,
                      row_loff + p.nbig}},
                    5, box, s);
        TSG_HIP_TRY(hipStreamSynchronize(s));
        int64_t tot2[5];
        std::copy(box->v, box->v + 5, tot2);
        const int64_t nsb_total = tot2[0], nunits = tot2[1];
        p.nsb_total = nsb_total;
        p.big_ent = tot2[2];
        p.big_prod = tot2[3];
        p.subcnt = ws.alloc_n<uint16_t>((size_t)nsb_total + 1);
        // keep every big row's bitmap in sparse form (masks of non-empty
        // words per sub-block, and band word lists: each row's region sized
        // by the bound min(products, span words) plus its bands' padding) for
        // the rank-indexed numeric phase when they fit a budget of device
        // memory; else the numeric phase uses per-item hash tables
        p.words_cap = tot2[4];
        const size_t cols_bytes =
            ((size_t)p.words_cap + (size_t)nsb_total) * sizeof(unsigned);
        size_t free_b = 0, total_b = 0;
        if (hipMemGetInfo(&free_b, &total_b) != hipSuccess) { (void)hipGetLastError(); free_b = 0; }
        const size_t budget = tune.bitmap_budget >= 0
                                  ? (size_t)tune.bitmap_budget
                                  : std::min<size_t>(size_t(48) << 30, free_b / 10 * 4);
        p.use_rank = cols_bytes <= budget && nsb_total < (int64_t(1) << 31);
        p.bandwords = p.use_rank ? ws.alloc_n<unsigned>((size_t)p.words_cap + 1) : nullptr;
        p.subocc = p.use_rank ? ws.alloc_n<unsigned>((size_t)nsb_total + 1) : nullptr;
        if (p.use_rank) {
            band_base = ws.alloc_n<int64_t>((size_t)nunits + 1);
            row_cur = ws.alloc_n<unsigned long long>((size_t)p.nbig + 1);
            d_overflow = ws.alloc_n<int64_t>(1);
            TSG_HIP_TRY(hipMemcpyAsync(row_cur, row_loff, sizeof(int64_t) * (size_t)p.nbig,
                                       hipMemcpyDeviceToDevice, s));
            TSG_HIP_TRY(hipMemsetAsync(d_overflow, 0, sizeof(int64_t), s));
        }
        // B as {column, value} records for the rank kernel's gathers
        p.bpk = p.use_rank ? ws.alloc_n<int4>((size_t)B.nnz + 1) : nullptr;
        // Spans this wide (at least item_sort_min windows of 16 sub-blocks)
        // make enough bands and items for them to run in column order, which
        // a radix sort arranges; B is then cut by its run directory and the
        // items are at most 8 sub-blocks wide, or sparse.
        p.column_order = nsb_total / 16 >= tune.item_sort_min;
        tm.end();

        // Column order: the run directory of B (R-MAT 2^20 with 8 draws a row:
        // 1.4 ms to build and 1.5 GB; the block pointers it replaces 3.3 ms
        // and 4.3 GB, and the numeric phase waited for them half its time, on
        // 390M of its 800M L2 misses in items of more than 512 outputs).  Rows'
        // order: B block pointers at the sub-block width (item and band
        // boundaries then need no search).  Either with finest blocks of 1024
        // columns while it stays <= 6 GiB, coarser beyond (a directory that
        // does not fit at all: a search).  Neither when building it would cost
        // more than the searches it saves -- more than 8 max(1, log2(L / 16)) entries per (A entry,
        // window of 16 sub-blocks) pair of the big rows, with the pairs
        // estimated from their A entries and average span and L, the mean
        // length of the B rows they reference, from their products per A
        // entry (measured on batches: an entry costs ~5 ps to build, a search
        // ~26 ps in B rows of ~30 entries, which span one or two cache lines,
        // and several times that in rows of hundreds, where each step misses;
        // the rule is the pointers', but holds for the directory.  Whole
        // products with it and with searches: R-MAT with 8 draws a row 2^16
        // 1.82 and 1.95 ms, 2^18 6.4 and 11.5, 2^20 48 and 136; rows of 500 and
        // 5000 entries, 1000 and 64 of them, in 2^20 columns of 8 entries 2.2
        // and 1.6, 2.4 and 1.7, and searched; it is off for few long rows, whose
        // waves wait on each search: one of 50,000 entries 2.6 and 3.9, four of
        // 100,000 5.6 and 7.1, and searched)
        // -- or when the budget is 0: B's row pointers then act as a one-block
        // table (block width 2^30 >= k) and every range comes from a search
        // inside its B row.
        tm.begin("row.bptr");
        const size_t bptr_cap = tune.bptr_budget >= 0 ? (size_t)tune.bptr_budget
                                                      : (size_t(6) << 30);
        const double fine_entries =
            (double)n * (double)((((size_t)k + (1u << SUB_SHIFT) - 1) >> SUB_SHIFT) + 1);
        const double pairs = (double)tot2[2] * ((double)nsb_total / (16.0 * p.nbig) + 1.0);
        const double brow = tot2[2] > 0 ? (double)tot2[3] / (double)tot2[2] : 1.0;
        const bool rowptr = k <= (1 << 30) &&
                        (tune.bptr_budget == 0 ||
                         (tune.bptr_budget < 0 &&
                          fine_entries > 8.0 * pairs * std::max(1.0, std::log2(brow / 16.0))));
        p.dir = RunDir();
        p.bptr = nullptr;
        bool table = !rowptr && n > 0;
        if (table && p.column_order) {
            // finest blocks of 1 << shift columns, coarser until cells (12
            // bytes each with the bits they are built from) and runs fit
            const int ngrp = (n + 31) / 32;
            const int nband = (int)(((size_t)k + (1u << (SUB_SHIFT + BAND_SHIFT)) - 1) >>
                                    (SUB_SHIFT + BAND_SHIFT));
            for (int c = 0; c <= BAND_SHIFT && !p.dir.cells; c++) {
                const int levels = BAND_SHIFT + 1 - c;
                const int64_t nblk = (int64_t)nband << (BAND_SHIFT - c);
                const int64_t ncells = (2 * nblk - (2 * nblk >> levels)) * ngrp;
                const int64_t chunks = (ncells + DIR_CHUNK - 1) / DIR_CHUNK;
                const int64_t max_runs = levels * (int64_t)B.nnz;
                const size_t bytes = (size_t)chunks * (DIR_CHUNK * 12 + 8) + (size_t)max_runs * 8;
                if (bytes > bptr_cap || max_runs >= (int64_t(1) << 31) ||
                    nblk >= (int64_t(1) << 30) || chunks >= (int64_t(1) << 31))
                    continue;
                unsigned *bits = ws.alloc_n<unsigned>((size_t)chunks * DIR_CHUNK);
                uint2 *cells = ws.alloc_n<uint2>((size_t)chunks * DIR_CHUNK);
                int2 *runs = ws.alloc_n<int2>((size_t)max_runs + 1);
                int64_t *sums = ws.alloc_n<int64_t>((size_t)chunks + 1);
                int64_t *tmp = ws.alloc_n<int64_t>(scan_tmp_elems((size_t)chunks + 1));
                p.dir.cells = cells;
                p.dir.runs = runs;
                p.dir.ngrp = ngrp;
                p.dir.nblk = (int)nblk;
                p.dir.shift = SUB_SHIFT + c;
                p.dir.coarse = c > 0;
                const unsigned ranges = grid_for((size_t)nblk, DIR_BLK, 65535);
                const bool cut = ranges > 1;
                hipLaunchKernelGGL(cut ? k_dir_bits<true> : k_dir_bits<false>,
                                   dim3(grid_for((size_t)n, DIR_ROWS), cut ? ranges : 1),
                                   dim3(1024), 0, s, n, B.ptr, B.idx, ngrp, p.dir.nblk,
                                   p.dir.shift, levels, bits);
                TSG_LAUNCH_CHECK();
                hipLaunchKernelGGL(k_dir_sums, dim3((unsigned)chunks), dim3(256), 0, s, ncells,
                                   bits, sums);
                TSG_LAUNCH_CHECK();
                exclusive_scan_i64(sums, sums, (size_t)chunks, tmp, s);
                hipLaunchKernelGGL(k_dir_cells, dim3((unsigned)chunks), dim3(256), 0, s, ncells,
                                   bits, sums, cells);
                TSG_LAUNCH_CHECK();
                hipLaunchKernelGGL(k_dir_runs, dim3(grid_for((size_t)B.nnz, RUN_ENT)), dim3(256), 0,
                                   s, n, (int)B.nnz, B.ptr, B.idx, ngrp, p.dir.nblk, p.dir.shift, levels,
                                   cells, runs);
                TSG_LAUNCH_CHECK();
            }
            table = !p.dir.cells && k > (1 << 30);
        }
        if (table) {
            int bs = SUB_SHIFT;
            while (bs < 30) {
                size_t nblk = ((size_t)k + (1u << bs) - 1) >> bs;
                if ((size_t)n * (nblk + 1) * sizeof(int) <= bptr_cap) break;
                bs++;
            }
            p.blk_shift = bs;
            p.nblk = (int)(((size_t)k + (1u << bs) - 1) >> bs);
            p.bptr = ws.alloc_n<int>((size_t)n * (p.nblk + 1));
            hipLaunchKernelGGL(k_bptr_rows, dim3(grid_for((size_t)n, 4, MAX_GRID)), dim3(256), 0,
                               s, n, B.ptr, B.idx, p.nblk, bs, p.bptr);
            TSG_LAUNCH_CHECK();
        }
        tm.end();

        tm.begin("row.big_symbolic");
        int2 *units = ws.alloc_n<int2>((size_t)nunits + 1);
        int *ukeys = ws.alloc_n<int>((size_t)nunits + 1);
        hipLaunchKernelGGL(k_band_fill, dim3(grid_for((size_t)p.nbig, 256)), dim3(256), 0, s,
                           p.nbig, p.span_sb0, band_off, units, ukeys);
        TSG_LAUNCH_CHECK();
        if (p.column_order && nunits > 1 && nunits < (int64_t(1) << 31)) {
            int *order = ws.alloc_n<int>((size_t)nunits);
            int end_bit = 1;
            while (end_bit < 31 && (int64_t(1) << end_bit) <= ((int64_t)k >> SUB_SHIFT)) end_bit++;
            sort_order_i32(ukeys, nunits, end_bit, order, ws, s);
            int2 *sorted = ws.alloc_n<int2>((size_t)nunits + 1);
            hipLaunchKernelGGL(k_gather_units, dim3(grid_for((size_t)nunits, 256)), dim3(256), 0,
                               s, nunits, order, units, sorted);
            TSG_LAUNCH_CHECK();
            units = sorted;
        }
        auto symbolic = p.dir.cells ? k_big_symbolic<true> : k_big_symbolic<false>;
        hipLaunchKernelGGL(symbolic,
                           dim3(grid_for((size_t)nunits, 1, MAX_GRID * 256 / BAND_T)), dim3(BAND_T),
                           0, s, nunits, units, rowsb, k, (int)p.column_order, A.ptr, A.idx, B.idx,
                           b_rows(p, B.ptr), p.span_sb0, p.sb_off, p.subcnt, front.rownnz, band_off,
                           band_base, row_cur, row_loff, d_overflow, p.subocc, p.bandwords);
        TSG_LAUNCH_CHECK();
        tm.end();
    }

    tm.begin("row.scan");
    exclusive_scan_i64(front.rownnz, d_ic, (size_t)m, scan_tmp, s, &box->v[7]);
    tm.end();

    int64_t h_tot[2] = {0, 0};
    if (p.nbig > 0) {
        tm.begin("row.items");
        const int *rowsb = front.rows(ROW_BIN_BIG);
        p.item_cnt = ws.alloc_n<int64_t>((size_t)p.nbig + 1);
        int64_t *tmp2 = ws.alloc_n<int64_t>(scan_tmp_elems((size_t)p.nbig + 1));
        // Narrow (8-sub-block) windows when the spans are wide enough that
        // the items will be run in column order: the items in flight then
        // read a band of B half as wide, which the L2 holds better; wide
        // windows otherwise (fewer items, fewer (A entry, item) pairs).
        const bool narrow = p.column_order;
        p.narrow_items = narrow;
        // sparse stretches in wide items, for the kernel whose work and LDS
        // follow the outputs, not the columns (rank mode, by size class)
        int wide_cap = narrow && p.use_rank ? WIDE_CAP : 0;
        auto items_kernel = [&](auto kern, int64_t *cnt, ItemRec *it, int *itn) {
            in_launches(p.nbig, 4, 256, [&](int64_t r0, int nr) {
                hipLaunchKernelGGL(kern, dim3(grid_for(nr, 4)), dim3(256), 0, s, nr, rowsb + r0, k,
                                   (int)narrow, wide_cap, p.span_sb0 + r0, p.sb_off + r0, p.subcnt,
                                   d_ic, cnt + r0, it, itn, p.subocc, band_off + r0, band_base);
                TSG_LAUNCH_CHECK();
            });
        };
        while (true) {
            if (narrow)
                items_kernel(k_items<false, 8>, p.item_cnt, nullptr, nullptr);
            else
                items_kernel(k_items<false, 16>, p.item_cnt, nullptr, nullptr);
            exclusive_scan_i64(p.item_cnt, p.item_cnt, (size_t)p.nbig, tmp2, s);
            publish_i64({{p.item_cnt + p.nbig, d_overflow}}, d_overflow ? 2 : 1, box, s);
            TSG_HIP_TRY(hipStreamSynchronize(s));
            // more than can be sorted by class: none for the sparse kernels
            if (wide_cap == 0 || box->v[0] < (int64_t(1) << 31)) break;
            wide_cap = 0;
        }
        h_tot[0] = box->v[7];
        h_tot[1] = box->v[0];
        const int64_t h_overflow = d_overflow ? box->v[1] : 0;
        // the lists are sized by a bound on the outputs, so this holds unless
        // the symbolic phase itself went wrong
        TSG_CHECK(h_overflow == 0, TSG_ERR_OVERFLOW, "big-row word lists exceed their bound");
        p.nitems = h_tot[1];
        p.items = ws.alloc_n<ItemRec>((size_t)p.nitems + 1);
        int *item_n = ws.alloc_n<int>((size_t)p.nitems + 1);
        if (narrow)
            items_kernel(k_items<true, 8>, p.item_cnt, p.items, item_n);
        else
            items_kernel(k_items<true, 16>, p.item_cnt, p.items, item_n);
        p.class_end[0] = 0;
        p.class_end[1] = p.nitems;
        if (p.column_order && p.nitems > 0 && p.nitems < (int64_t(1) << 31)) {
            const size_t ni = (size_t)p.nitems;
            int *keys = ws.alloc_n<int>(ni);
            int *order = ws.alloc_n<int>(ni);
            unsigned long long *class_cnt = ws.alloc_n<unsigned long long>(ITEM_CLASSES);
            TSG_HIP_TRY(hipMemsetAsync(class_cnt, 0, sizeof(int64_t) * ITEM_CLASSES, s));
            int end_bit = 1;
            while (end_bit < 27 && (int64_t(1) << end_bit) <= ((int64_t)k >> SUB_SHIFT)) end_bit++;
            // the size class splits the rank path's items only
            hipLaunchKernelGGL(k_item_keys, dim3(grid_for(ni, 256 * 16)), dim3(256), 0, s,
                               p.nitems, p.items, item_n, A.ptr, p.use_rank ? end_bit : -1, keys,
                               class_cnt);
            TSG_LAUNCH_CHECK();
            sort_order_i32(keys, p.nitems, p.use_rank ? end_bit + 4 : end_bit, order, ws, s);
            ItemRec *items_s = ws.alloc_n<ItemRec>(ni + 1);
            hipLaunchKernelGGL(k_gather_items, dim3(grid_for(ni, 256)), dim3(256), 0, s,
                               p.nitems, order, p.items, items_s);
            TSG_LAUNCH_CHECK();
            p.items = items_s;
            if (p.use_rank) {
                const int64_t *cc = reinterpret_cast<const int64_t *>(class_cnt);
                publish_i64({{cc, cc + 1}}, ITEM_CLASSES - 1, box, s);
                TSG_HIP_TRY(hipStreamSynchronize(s));
                int64_t end = 0;
                for (int c = 0; c < ITEM_CLASSES - 1; c++) p.class_end[c] = end += box->v[c];
            }
        }
        tm.end();
    } else {
        TSG_HIP_TRY(hipStreamSynchronize(s));
        h_tot[0] = box->v[7];
    }
    *nnz_c = h_tot[0];
    p.valid = true;
}

template <bool FUSED>
static void row_numeric_t(RowPlan &p, const CsrIn &A, const CsrIn &B, const int64_t *d_ic,
                          int *d_jc, double *d_c, hipStream_t s, StageTimer &tm) {
    const RowFront &front = p.front;
    tm.begin("row.small_numeric");
    {
        auto launch = [&](auto kern, int rpb, int threads, int bin) {
            in_launches(front.count[bin], rpb, threads, [&](int64_t r0, int nr) {
                hipLaunchKernelGGL(kern, dim3(grid_for(nr, rpb)), dim3(threads), 0, s, nr,
                                   front.rows(bin) + r0, A.ptr, A.idx, A.val, B.ptr, B.idx, B.val,
                                   d_ic, d_jc, d_c, (int)p.b_strict);
                TSG_LAUNCH_CHECK();
            });
        };
        launch(k_flat_numeric<FUSED, 16, 4, 64, 64, 64, 256>, 16, 256, 1);
        launch(k_flat_numeric<FUSED, 64, 4, 64, 512, 256, 64>, 1, 64, 2);
        launch(k_flat_numeric<FUSED, 64, 8, 64, 512, 512, 64>, 1, 64, 3);
        launch(k_flat_numeric<FUSED, 64, 16, 64, 512, 512, 64>, 1, 64, 4);
        launch(k_flat_numeric<FUSED, 64, 16, 1024, 512, 512, 64>, 1, 64, ROW_BIN_MANY);
        launch(k_flat_numeric<FUSED, 64, 24, 64, 512, 512, 64, 4>, 1, 64, ROW_BIN_MED);
    }
    tm.end();
    if (p.nitems > 0 && p.use_rank) {
        tm.begin("row.big_numeric");
        if (p.big_ent * PACK_ENT_COST < B.nnz && p.big_prod * PACK_PROD_COST < B.nnz) {
            const unsigned groups = grid_for((size_t)p.big_ent, PACK_ENT);
            const unsigned share = std::min(std::max(4096u / groups, 4u), 64u);
            hipLaunchKernelGGL(k_pack_rows, dim3(groups, share), dim3(256), 0, s, p.big_ent, p.nbig,
                               p.ent_off, front.rows(ROW_BIN_BIG), A.ptr, A.idx, B.ptr, B.idx,
                               B.val, p.bpk);
            TSG_LAUNCH_CHECK();
        } else if (B.nnz > 0) {
            hipLaunchKernelGGL(k_pack_b, dim3(grid_for((size_t)B.nnz, 256)), dim3(256), 0, s,
                               B.nnz, B.idx, B.val, p.bpk);
            TSG_LAUNCH_CHECK();
        }
        const ItemArgs T{p.bandwords, p.subocc, A.ptr, A.idx,  A.val,
                         B.idx,       p.bpk,    d_jc,  d_c,    (int)p.b_strict};
        const BRows brows = b_rows(p, B.ptr);
        const int64_t ns = p.class_end[0], nd = p.class_end[1] - ns;
        if (ns > 0) {
            auto kern = p.dir.cells ? k_big_numeric_small<FUSED, true>
                                    : k_big_numeric_small<FUSED, false>;
            hipLaunchKernelGGL(kern, dim3(item_grid(ns)), dim3(64), 0, s, ns, p.items, T, brows);
            TSG_LAUNCH_CHECK();
        }
        if (p.nitems > ns) {
            constexpr int W = ITEM_WORDS;
            auto kern = !p.narrow_items ? k_big_numeric_rank<FUSED, W, false>
                        : p.dir.cells   ? k_big_numeric_rank<FUSED, W / 2, true>
                                        : k_big_numeric_rank<FUSED, W / 2, false>;
            hipLaunchKernelGGL(kern, dim3(item_grid(p.nitems - ns)), dim3(64), 0, s,
                               p.nitems - ns, nd, p.items + ns, T, brows);
            TSG_LAUNCH_CHECK();
        }
        tm.end();
    } else if (p.nitems > 0) {
        tm.begin("row.big_numeric");
        constexpr size_t sm = sizeof(ItemSmem) * ITEM_WAVES;
        auto kern = p.dir.cells ? k_big_numeric<FUSED, true> : k_big_numeric<FUSED, false>;
        set_smem(kern, sm);
        const unsigned grid = item_grid(p.nitems);
        hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * ITEM_WAVES), sm, s, p.nitems, p.items,
                           A.ptr, A.idx, A.val, B.idx, B.val, b_rows(p, B.ptr), d_jc, d_c, (int)p.b_strict);
        TSG_LAUNCH_CHECK();
        tm.end();
    }
}

void row_numeric(RowPlan &p, const CsrIn &A, const CsrIn &B, const int64_t *d_ic, int *d_jc,
                 double *d_c, int fused, hipStream_t s, StageTimer &tm) {
    TSG_CHECK(p.valid && p.m == A.rows && p.n == A.cols && p.k == B.cols, TSG_ERR_STATE,
              "row numeric phase without a matching symbolic phase");
    if (fused)
        row_numeric_t<true>(p, A, B, d_ic, d_jc, d_c, s, tm);
    else
        row_numeric_t<false>(p, A, B, d_ic, d_jc, d_c, s, tm);
}
