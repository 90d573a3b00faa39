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
//   * Small rows (<= SMALL_PROD products): one lane group per row with all its
//     products in registers (tsg_flat.h); an output's place is its column's
//     rank in a two-level bitmap, so C comes out sorted with no hash or sort.
//   * Big rows: the symbolic phase cuts each row's column span into bands of
//     65536 columns, marks the row's columns of a band in an LDS bitmap and
//     records the count of every 1024-column sub-block (and, when memory
//     allows, the band's bitmap in sparse form: a mask of non-empty words per
//     sub-block, and those words); the numeric phase splits the row into
//     items of <= ITEM_CAP outputs and <= 16384 columns, each accumulated by
//     one wave into a rank-ordered LDS array (rank from the stored bitmap)
//     and written in column order.  A B block pointer table gives each B row's
//     sub-range of a band or item without a search; bands and items run in
//     order of their first column, so those in flight share a band of B.
#include "tsg_internal.h"

#include <cmath>
#include "tsg_device.h"
#include "tsg_expand.h"
#include "tsg_flat.h"

#include <algorithm>
#include <map>
#include <mutex>

namespace {

constexpr int SMALL_PROD = 1024;       // rows up to this many products: small path

constexpr int SUB_SHIFT = 10;          // sub-block = 1024 columns
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
    const int r = blockIdx.x * RPB + grp;
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
// one B row after the other; past that, tag rounds take fewer steps.
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
    const int r = blockIdx.x * RPB + grp;
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
    const int r = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int l = threadIdx.x & 63;
    if (r >= nbig) return;
    const int row = rows[r];
    int lo = 0x7fffffff, hi = -1;
    for (int p = ia[row] + l; p < ia[row + 1]; p += 64) {
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
                    BAND_PAD * ((ns + (1 << BAND_SHIFT) - 1) >> BAND_SHIFT);
    }
}

// -------------------------------------------------------- big rows: symbolic
// A big row's span is cut into bands of 64 sub-blocks; a band unit {r, u}
// covers span sub-blocks [64u, 64u + 64) of big row r.  Units are run in
// order of their first column (like the numeric items), so the units in
// flight read B columns of one narrow band, which the L2 caches keep.
__global__ void __launch_bounds__(256) k_band_count(int nbig, const int64_t *__restrict__ nsb,
                                                    int64_t *__restrict__ cnt) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < nbig) cnt[r] = (nsb[r] + (1 << BAND_SHIFT) - 1) >> BAND_SHIFT;
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
        keys[o + u] = span_sb0[r] + (u << BAND_SHIFT);
    }
}

__global__ void __launch_bounds__(256) k_gather_units(int64_t n, const int *__restrict__ order,
                                                      const int2 *__restrict__ units,
                                                      int2 *__restrict__ out) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j < n) out[j] = units[order[j]];
}

// One block per band unit: LDS bitmap over the band, the row's products in
// the band (B rows restricted through the block pointers) marked by the 2
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
__global__ void __launch_bounds__(BAND_T) __attribute__((amdgpu_waves_per_eu(8))) k_big_symbolic(
    int64_t nunits, const int2 *__restrict__ units, const int *__restrict__ rows, int k,
    const int *__restrict__ ia, const int *__restrict__ ja, const int *__restrict__ ib,
    const int *__restrict__ jb, BlockPtrs bp, const int *__restrict__ span_sb0,
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
        const int64_t so = sb_off[r] + ((int64_t)u << BAND_SHIFT);
        const int nsb = (int)min((int64_t)1 << BAND_SHIFT, sb_off[r + 1] - so);
        const int sb0 = span_sb0[r] + (u << BAND_SHIFT);
        const int c0 = sb0 << SUB_SHIFT;
        const int c1 = (int)min((int64_t)k, (int64_t)(sb0 + nsb) << SUB_SHIFT);
        const int words = (c1 - c0 + 31) >> 5;
        for (int i = threadIdx.x; 4 * i < words; i += BAND_T)
            reinterpret_cast<uint4 *>(bits)[i] = make_uint4(0u, 0u, 0u, 0u);
        __syncthreads();
        for_products<BIG_SYM_U, NW, true, false>(
            ia[row], ia[row + 1], ja, nullptr, ib, jb, nullptr, bp, c0, c1, s_heads[wave],
            [&](const Batch &t) {
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
    const int t = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int l = threadIdx.x & 63;
    if (t >= n) return;
    const int lo = ib[t], hi = ib[t + 1];
    for (int b = l; b <= nblk; b += 64) {
        const int pos = b == nblk ? hi : lower_bound_i32(jb, lo, hi, b << bs);
        bptr[(size_t)t * (nblk + 1) + b] = pos;
    }
}

// Block-major table: bptr[b*n + t] = first position of B row t with column
// >= b << bs.  A block of 4 waves takes 64 B rows; for each range of 64 blocks
// the waves fill an LDS tile [block][row], a lane per block searching inside
// its row, then write it out as 64 consecutive rows per block (256-byte runs).
// The 64 rows' columns are one contiguous range of jb: when it holds at most
// BPT_STAGE entries (R-MAT 2^20's B averages ~940 per 64 rows) it is staged
// in LDS once and every search runs there; otherwise the searches read jb.
// The searches wait on their loads, so residency mattered with global
// searches (a 128-block tile took 6.2 ms instead of 4.5 ms for R-MAT 2^20's
// 16,385 x 2^20 table, a 32-block one 7.1 ms), and still does with staged
// ones: blocks of 128 or 256 rows (512- or 1024-byte runs) took 6.6 and
// 8.4 ms instead of 4.5.
constexpr int BPT_ROWS = 64, BPT_BLK = 64, BPT_STAGE = 2048;

__device__ __forceinline__ int lds_lower_bound(const int *a, int lo, int hi, int key) {
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (a[mid] < key) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

__global__ void __launch_bounds__(256) k_bptr(int n, const int *__restrict__ ib,
                                              const int *__restrict__ jb, int nblk, int bs,
                                              int *__restrict__ bptr) {
    __shared__ int tile[BPT_BLK][BPT_ROWS + 1];
    __shared__ int s_col[BPT_STAGE];
    __shared__ int s_rp[BPT_ROWS + 1];
    const int t0 = blockIdx.x * BPT_ROWS;
    const int nr = min(BPT_ROWS, n - t0);
    for (int i = threadIdx.x; i <= nr; i += blockDim.x) s_rp[i] = ib[t0 + i];
    __syncthreads();
    const int e0 = s_rp[0];
    const bool staged = s_rp[nr] - e0 <= BPT_STAGE;
    if (staged)
        for (int i = threadIdx.x; i < s_rp[nr] - e0; i += blockDim.x) s_col[i] = jb[e0 + i];
    __syncthreads();
    for (int b0 = 0; b0 <= nblk; b0 += BPT_BLK) {
        // (row, block) pairs, a thread each: a row's blocks in consecutive lanes
        for (int i = threadIdx.x; i < nr * BPT_BLK; i += blockDim.x) {
            const int r = i / BPT_BLK, bb = i % BPT_BLK;
            const int b = b0 + bb;
            if (b > nblk) continue;
            const int lo = s_rp[r], hi = s_rp[r + 1];
            int pos = hi;
            if (b < nblk)
                pos = staged ? e0 + lds_lower_bound(s_col, lo - e0, hi - e0, b << bs)
                             : lower_bound_i32(jb, lo, hi, b << bs);
            tile[bb][r] = pos;
        }
        __syncthreads();
        // a block's rows in consecutive lanes: runs of 4 * BPT_ROWS bytes
        for (int i = threadIdx.x; i < BPT_BLK * BPT_ROWS; i += blockDim.x) {
            const int bb = i / BPT_ROWS, r = i % BPT_ROWS;
            const int b = b0 + bb;
            if (b <= nblk && r < nr) bptr[(size_t)b * n + t0 + r] = tile[bb][r];
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------- item plan
constexpr int SMALL_ITEM = 256;
constexpr int MID_ITEM = 512;
// Sparse stretches go into wide items of up to this many outputs.  R-MAT 2^20
// with 8 draws a row, both sparse kernels: 31.7 ms without wide items (its
// 30M items of <= 256 outputs hold 45 each, and each costs its A entries, two
// block pointers an entry and its tables), 20.2 up to 256, 19.2 up to 384,
// 19.3 up to 512; R-MAT 2^18 with 4: 1.27, 1.01, 0.98, 0.96; ER batch of 512:
// 6.0, 5.9, 5.1, 4.3.
constexpr int WIDE_CAP = 512;
static_assert(WIDE_CAP <= MID_ITEM, "wide items run in the sparse kernels");

// Split of each big row into items: the row's span is cut into windows of
// WSB sub-blocks (at most ITEM_WBITS columns); inside a window, runs of
// sub-blocks with at most ITEM_CAP outputs, leading empty sub-blocks skipped.
// One wave per big row, one lane per window (64 windows per pass): a lane
// loads its window's counts at once and splits them in registers, and wave
// scans place the items and their outputs.  FILL=false counts items per
// row; FILL=true (item_cnt = exclusive item offsets) writes each item's
// record -- {row, c0, c1, big-row index}, its first output position -- and
// output count, and, in rank mode (band_base given), where its first
// non-empty word is in the band word lists of the symbolic phase (from the
// sub-blocks' masks of non-empty words); the record's fourth field then
// holds the item's first sub-block's index in subcnt and subocc (< 2^31 in
// that mode) instead of the big-row index, so the numeric phase finds the
// item's masks with no other lookup.  Windows lie inside bands, and a
// band's windows inside one pass of 64 windows, so the item's place in its
// band's list is its count of non-empty words before it less that of the
// band's first window.
// Wide items: an aligned run of 2, 4 or 8 windows of one band whose outputs
// number at most wide_cap becomes one item (the longest such run).
template <bool FILL, int WSB>
__global__ void __launch_bounds__(256) k_items(int nbig, const int *__restrict__ rows, int k,
                                               int wide_cap,
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
    const int first = span_sb0[r];
    const int nwin = (nsb + WSB - 1) / WSB;
    int64_t wbase = FILL ? item_cnt[r] : 0;
    int64_t obase = FILL ? ic[row] : 0;
    for (int w0 = 0; w0 < nwin; w0 += 64) {
        const int win = w0 + l;
        const int j0 = win * WSB;
        const int len = win < nwin ? min(WSB, nsb - j0) : 0;
        int cs[WSB], os[WSB];
        int nzt = 0;
#pragma unroll
        for (int q = 0; q < WSB; q++) {
            cs[q] = q < len ? (int)sc[j0 + q] : 0;
            os[q] = FILL && words && q < len ? __popc(subocc[sb_off[r] + j0 + q]) : 0;
            nzt += os[q];
        }
        int nit = 0, tot = 0, firstq = WSB, lastq = -1;
        {
            int start = -1, cnt = 0;
#pragma unroll
            for (int q = 0; q < WSB; q++) {
                if (start >= 0 && cnt + cs[q] > ITEM_CAP) {
                    nit++;
                    start = -1;
                    cnt = 0;
                }
                if (cs[q] != 0 || start >= 0) {
                    if (start < 0) start = q;
                    cnt += cs[q];
                }
                tot += cs[q];
                if (cs[q] != 0) {
                    firstq = min(firstq, q);
                    lastq = q;
                }
            }
            if (start >= 0 && cnt > 0) nit++;
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
                                             min(k, (first + sb_last + 1) << SUB_SHIFT),
                                             words ? (int)(sb_off[r] + sb_first) : r),
                                   out, wb};
                item_n[w] = run_tot;
            }
            int start = -1, cnt = 0, nzrun = 0, nzs = 0;
#pragma unroll
            for (int q = 0; q < WSB; q++) {
                if (run > 1) break;
                if (start >= 0 && cnt + cs[q] > ITEM_CAP) {
                    items[w] = ItemRec{make_int4(row, (cbase + start) << SUB_SHIFT,
                                                 min(k, (cbase + q) << SUB_SHIFT),
                                                 words ? (int)(sb_off[r] + j0 + start) : r),
                                       out, wb + nzs};
                    item_n[w] = cnt;
                    w++;
                    out += cnt;
                    start = -1;
                    cnt = 0;
                }
                if (cs[q] != 0 || start >= 0) {
                    if (start < 0) {
                        start = q;
                        nzs = nzrun;
                    }
                    cnt += cs[q];
                }
                nzrun += os[q];
            }
            if (run == 1 && start >= 0 && cnt > 0) {
                items[w] = ItemRec{make_int4(row, (cbase + start) << SUB_SHIFT,
                                             min(k, (cbase + len) << SUB_SHIFT),
                                             words ? (int)(sb_off[r] + j0 + start) : r),
                                   out, wb + nzs};
                item_n[w] = cnt;
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
// Items sort by size class -- at most SMALL_ITEM outputs, at most MID_ITEM,
// more -- then by first column: key = class << class_bit | first sub-block
// (class_bit < 0: no classes).  The numeric phase runs each class in a
// kernel whose value array holds just that class's items, so smaller items
// take less LDS and more of them are resident.  block_small[b] and
// block_mid[b] count block b's items of the first two classes.
// Product batches in flight per lane and waves per SIMD of the two sparse
// item kernels.  R-MAT 2^20 (8 draws a row), <= 256 outputs: 6.0 ms at (4, 6),
// 5.8 at (6, 5) and (4, 7), 6.2 at (8, 5); <= 512: 13.3 at (6, 5), 12.7 at
// (6, 4), 12.9 at (8, 4), 13.0 at (4, 5).
constexpr int SMALL_RANK_U = 6;
constexpr int SMALL_MINW = 5;
constexpr int MID_RANK_U = 6;
constexpr int MID_MINW = 4;

__global__ void __launch_bounds__(256) k_item_keys(int64_t n, const ItemRec *__restrict__ items,
                                                   const int *__restrict__ item_n, int class_bit,
                                                   int *__restrict__ keys,
                                                   int *__restrict__ block_small,
                                                   int *__restrict__ block_mid) {
    __shared__ int s_cnt[2][4];
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int cls = 0;
    if (i < n && class_bit >= 0) cls = item_n[i] <= SMALL_ITEM ? 0 : item_n[i] <= MID_ITEM ? 1 : 2;
    if (i < n) keys[i] = (cls << max(class_bit, 0)) | (items[i].d.y >> SUB_SHIFT);
    const unsigned long long b0 = __ballot(i < n && class_bit >= 0 && cls == 0);
    const unsigned long long b1 = __ballot(i < n && class_bit >= 0 && cls == 1);
    if (__lane_id() == 0) {
        s_cnt[0][threadIdx.x >> 6] = __popcll(b0);
        s_cnt[1][threadIdx.x >> 6] = __popcll(b1);
    }
    __syncthreads();
    if (threadIdx.x < 2)
        (threadIdx.x ? block_mid : block_small)[blockIdx.x] =
            s_cnt[threadIdx.x][0] + s_cnt[threadIdx.x][1] + s_cnt[threadIdx.x][2] +
            s_cnt[threadIdx.x][3];
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

template <bool FUSED>
__global__ void __launch_bounds__(64 * ITEM_WAVES) k_big_numeric(
    int64_t nitems, const ItemRec *__restrict__ items,
    const int *__restrict__ ia, const int *__restrict__ ja, const double *__restrict__ a,
    const int *__restrict__ ib, const int *__restrict__ jb, const double *__restrict__ b,
    BlockPtrs bp, int *__restrict__ jc,
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
        for_products<ITEM_U, 1, true, true>(
            ia[row], ia[row + 1], ja, a, ib, jb, b, bp, c0, c1, S.heads, [&](const Batch &t) {
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

// Rank-indexed variant: the symbolic phase stored every big row's column
// bitmap (in sparse form: per sub-block a mask of its non-empty words, and
// those words), so an item's outputs are known before its products are
// visited.  The rank of column j inside the item is prefix[w] + popc(bits[w]
// below j) -- one LDS read of a {bits, prefix} pair -- and values accumulate
// in a dense rank-ordered array that is written out coalesced.
// WORDS: bitmap words of the widest item (256 or 512: items of 8192 or
// 16384 columns).
template <int WORDS>
struct RankSmem {
    uint2 words[WORDS];           // {bitmap word, outputs before it}
    double vals[ITEM_CAP];
    unsigned tags[ITEM_TAGS];     // bucketed by rank
    int heads[64];                // start bits of the product expansion
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
__device__ __forceinline__ int item_rank_build(RankSmem<WORDS> &S, unsigned (&wv)[WCH], int c0,
                                               int c1, int64_t o, int *__restrict__ jc) {
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
        if (w < nwords) S.words[w] = make_uint2(wv[j], (unsigned)base);
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

// Writes an item's cnt values to C at offset o, straight from LDS.
template <int WORDS>
__device__ __forceinline__ void item_store_values(RankSmem<WORDS> &S, int cnt, int64_t o,
                                                  double *__restrict__ c) {
    const int l = __lane_id();
    wave_lds_fence();
    for (int i = l; i < cnt; i += 64) __builtin_nontemporal_store(S.vals[i], c + o + i);
    wave_lds_fence();
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
        const uint2 wd = S.words[cc >> 5];
        rank = (int)wd.y + __popc(wd.x & ((1u << (cc & 31)) - 1u));
    }
    if (b_strict && t.nseg <= FLAT_SEGS) {
        for (int s = 1; s <= t.nseg; s++) {
            if (rank >= 0 && t.seg == s) S.vals[rank] = acc_step<FUSED>(S.vals[rank], t.a, t.b);
            wave_lds_fence();
        }
        return;
    }
    ordered_accumulate<FUSED, ITEM_TAGS>(rank >= 0, rank, t.a, t.b, S.vals, S.tags,
                                         (unsigned)__lane_id(), false);
}

template <bool FUSED, int WORDS>
__global__ void __launch_bounds__(64 * ITEM_WAVES) k_big_numeric_rank(
    int64_t nitems, const ItemRec *__restrict__ items, const unsigned *__restrict__ wlist,
    const unsigned *__restrict__ subocc, const int *__restrict__ ia, const int *__restrict__ ja,
    const double *__restrict__ a, const int *__restrict__ jb, const double *__restrict__ b,
    const int4 *__restrict__ bpk, BlockPtrs bp, int *__restrict__ jc, double *__restrict__ c,
    int b_strict) {
    extern __shared__ __align__(16) unsigned char smem[];
    RankSmem<WORDS> &S = reinterpret_cast<RankSmem<WORDS> *>(smem)[threadIdx.x >> 6];
    const int l = __lane_id();
    for (int i = l; i < ITEM_TAGS; i += 64) S.tags[i] = 0xffffffffu;
    const int64_t wave_id = (int64_t)blockIdx.x * ITEM_WAVES + (threadIdx.x >> 6);
    const int64_t nwaves = (int64_t)gridDim.x * ITEM_WAVES;
    // the next item's descriptor is loaded when an item starts, and its
    // sub-block masks, word-list position and A row bounds while the item's
    // outputs are stored, so an item's first product loads need no chain of
    // dependent loads.  Those and the item's output offset go into one
    // register, a lane each (lanes 0..15 the masks, 16 and 17 the position,
    // 18 and 19 the row bounds, 20 and 21 the offset: one load instruction,
    // and they reach scalar registers at the item's start -- the small-item
    // kernel has no vector registers to spare).
    int4 item = make_int4(0, 0, 0, 0);
    unsigned nx = 0u;
    auto locate = [&](int64_t at) {
        // item.w: the item's first sub-block in subocc
        const int nsb = (item.z - item.y + (1 << SUB_SHIFT) - 1) >> SUB_SHIFT;
        const unsigned *src = nullptr;
        if (l < min(nsb, 2 * (WORDS / 64)))
            src = subocc + ((int64_t)item.w + l);
        else if (l == 16 || l == 17)
            src = reinterpret_cast<const unsigned *>(&items[at].wpos) + (l - 16);
        else if (l == 18 || l == 19)
            src = reinterpret_cast<const unsigned *>(ia + item.x) + (l - 18);
        else if (l == 20 || l == 21)
            src = reinterpret_cast<const unsigned *>(&items[at].off) + (l - 20);
        nx = src ? *src : 0u;
    };
    // (streaming loads of the item descriptors and A entries, read once per
    // item, were measured slower: 158 -> 166 ms on R-MAT 2^20 A*A^T)
    if (wave_id < nitems) {
        item = items[wave_id].d;
        locate(wave_id);
    }
    for (int64_t it = wave_id; it < nitems; it += nwaves) {
        const int c0 = __builtin_amdgcn_readfirstlane(item.y);
        const int c1 = __builtin_amdgcn_readfirstlane(item.z);
        const unsigned iocc = l < 16 ? nx : 0u;
        const int ipa = __builtin_amdgcn_readlane((int)nx, 18);
        const int ipe = __builtin_amdgcn_readlane((int)nx, 19);
        const int64_t iwpos =
            (int64_t)(((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)nx, 17) << 32) |
                      (uint32_t)__builtin_amdgcn_readlane((int)nx, 16));
        const unsigned *ilist = wlist + iwpos;
        const int64_t o =
            (int64_t)(((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)nx, 21) << 32) |
                      (uint32_t)__builtin_amdgcn_readlane((int)nx, 20));
        const int64_t next = it + nwaves;
        if (next < nitems) item = items[next].d;
        // the product pipeline of for_products, with the rank table built
        // after the first groups' A entries and B ranges are issued, so the
        // word loads and that chain of dependent loads overlap
        auto load_t = [&](int g, int &t, double &av) {
            const int p = g + l;
            t = -1;
            av = 0.0;
            if (g < ipe && p < ipe) {
                t = ja[p];
                av = a[p];
            }
        };
        auto load_range = [&](int t, int &lo, int &hi) {
            lo = 0;
            hi = 0;
            if (t >= 0) {
                lo = brange_lo(bp, jb, t, c0);
                hi = brange_lo(bp, jb, t, c1);
            }
        };
        int t0, t1;
        double a0, a1;
        load_t(ipa, t0, a0);
        load_t(ipa + 64, t1, a1);
        const int pc = __popc(iocc);
        const int pre = dpp_incl_scan<16>(pc) - pc;
        unsigned wv[WORDS / 64];
        item_words(ilist, iocc, pre, c0, c1, wv);
        int lo, hi;
        load_range(t0, lo, hi);
        const int cnt = item_rank_build<WORDS>(S, wv, c0, c1, o, jc);
        auto f = [&](const Batch &t) {
            item_accumulate<FUSED, WORDS>(S, c0, t, b_strict);
        };
        for (int g = ipa; g < ipe; g += 64) {
            const double ag = a0;
            int lo_n, hi_n, t2;
            double a2;
            load_range(t1, lo_n, hi_n);
            load_t(g + 128, t2, a2);
            expand_group<RANK_U, true, true>(lo, max(hi - lo, 0), ag, jb, b, S.heads, f, bpk);
            lo = lo_n;
            hi = hi_n;
            t1 = t2;
            a0 = a1;
            a1 = a2;
        }
        if (next < nitems) locate(next);
        item_store_values(S, cnt, o, c);
    }
}

// Items of at most CAP outputs, however wide up to a band: the rank of a
// column goes through the item's sub-blocks (mask of non-empty words, words
// before it) to its word (bits, outputs before it), so table and work follow
// the outputs and not the columns.  The outputs' columns are noted by the
// products (as offsets in the item) instead of expanded from the words.
//
// The dense tables it replaces for these items cost ~500 vector instructions
// an item whatever its products (the issue rate bound them: 25 of 29 ms of
// R-MAT 2^20 with 8 draws a row); now 5.8 ms, with the 257..512-output items
// 37.7 -> 18.5 ms.  Larger items keep the dense table: one lookup a product,
// and they run at the memory's rate (4.65 TB/s).
template <int CAP>
struct SparseSmem {
    uint2 words[CAP];             // {bits, outputs before}
    double vals[CAP];
    uint2 sub[1 << BAND_SHIFT];   // {mask of non-empty words, words before}
    uint16_t cols[CAP];
    unsigned tags[CAP / 4];       // a byte per output, or tag buckets
    int heads[64];
};

template <bool FUSED, int CAP, int U, int MINW>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(MINW)))
k_big_numeric_sparse(int64_t nitems, const ItemRec *__restrict__ items,
                     const unsigned *__restrict__ wlist, const unsigned *__restrict__ subocc,
                     const int *__restrict__ ia, const int *__restrict__ ja,
                     const double *__restrict__ a, const int *__restrict__ jb,
                     const int4 *__restrict__ bpk, BlockPtrs bp, int *__restrict__ jc,
                     double *__restrict__ c, int b_strict) {
    __shared__ __align__(16) SparseSmem<CAP> S;
    constexpr int NT = CAP / 4;
    const int l = threadIdx.x;
    uint8_t *own = reinterpret_cast<uint8_t *>(S.tags);
    for (int64_t it = blockIdx.x; it < nitems; it += gridDim.x) {
        const int4 item = items[it].d;
        const int64_t o = items[it].off;
        const unsigned *list = wlist + items[it].wpos;
        const int c0 = item.y, c1 = item.z;
        const int pa = ia[item.x], pe = ia[item.x + 1];
        const int nsb = min((c1 - c0 + (1 << SUB_SHIFT) - 1) >> SUB_SHIFT, 1 << BAND_SHIFT);
        const unsigned occ = l < nsb ? subocc[(int64_t)item.w + l] : 0u;
        auto load_t = [&](int g, int &t, double &av) {
            const int p = g + l;
            t = -1;
            av = 0.0;
            if (p < pe) {
                t = ja[p];
                av = a[p];
            }
        };
        auto load_range = [&](int t, int &lo, int &hi) {
            lo = 0;
            hi = 0;
            if (t >= 0) {
                lo = brange_lo(bp, jb, t, c0);
                hi = brange_lo(bp, jb, t, c1);
            }
        };
        int t0, lo, hi;
        double a0;
        load_t(pa, t0, a0);
        const int pc = __popc(occ);
        const int incl = wave_incl_scan(pc);
        // every non-empty word has an output
        const int nw = min(__builtin_amdgcn_readlane(incl, 63), CAP);
        unsigned wv[CAP / 64];
#pragma unroll
        for (int j = 0; j < CAP / 64; j++)
            wv[j] = j * 64 + l < nw ? __builtin_nontemporal_load(list + j * 64 + l) : 0u;
        load_range(t0, lo, hi);
        S.sub[l] = make_uint2(occ, (unsigned)(incl - pc));
        int cnt = 0;
#pragma unroll
        for (int j = 0; j < CAP / 64; j++) {
            if (j * 64 < nw) {
                const int p = __popc(wv[j]);
                const int in = wave_incl_scan(p);
                if (j * 64 + l < nw)
                    S.words[j * 64 + l] = make_uint2(wv[j], (unsigned)(cnt + in - p));
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
                const int w = (int)sb.y + (int)__popc(sb.x & ((1u << ((cc >> 5) & 31)) - 1u));
                const uint2 wd = S.words[min(w, CAP - 1)];
                rank = min((int)wd.y + (int)__popc(wd.x & ((1u << (cc & 31)) - 1u)), CAP - 1);
                S.cols[rank] = (uint16_t)cc;
            }
            bool clash = t.nseg > 1 || !b_strict;
            if (b_strict && t.nseg > 2) {
                if (t.act) own[rank] = (uint8_t)l;
                wave_lds_fence();
                clash = __ballot(t.act && own[rank] != (uint8_t)l) != 0;
                wave_lds_fence();
            }
            if (!clash) {
                if (t.act) S.vals[rank] = acc_step<FUSED>(S.vals[rank], t.a, t.b);
                wave_lds_fence();
            } else if (b_strict && t.nseg <= FLAT_SEGS) {
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
        for (int g = pa; g < pe; g += 64) {
            int t1, lo_n, hi_n;
            double a1;
            load_t(g + 64, t1, a1);
            load_range(t1, lo_n, hi_n);
            expand_group<U, true, true>(lo, max(hi - lo, 0), a0, jb, nullptr, S.heads, f, bpk);
            lo = lo_n;
            hi = hi_n;
            a0 = a1;
        }
        wave_lds_fence();
        for (int i = l; i < cnt; i += 64) {
            __builtin_nontemporal_store(c0 + (int)S.cols[i], jc + o + i);
            __builtin_nontemporal_store(S.vals[i], c + o + i);
        }
        wave_lds_fence();
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

// The plan's block pointers in the layout they were built in; without a
// table, B's row pointers b_ptr (of the call at hand) as a one-block table.
static BlockPtrs block_ptrs(const RowPlan &p, const int *b_ptr) {
    BlockPtrs bp;
    bp.p = p.bptr;
    bp.bs = p.blk_shift;
    if (p.bptr_rowptr) {
        bp.p = b_ptr;
        bp.tstride = 1;
        bp.bstride = 1;
    } else if (p.column_order) {
        bp.tstride = 1;
        bp.bstride = p.n;
    } else {
        bp.tstride = p.nblk + 1;
        bp.bstride = 1;
    }
    return bp;
}

// One block per item (the hardware dispatcher hands the next item to
// whichever CU frees a slot first, so no CU idles behind a long tail); the
// item kernels keep a grid-stride loop for item counts beyond the grid limit.
static unsigned item_grid(int64_t nitems) {
    return (unsigned)std::min<int64_t>((nitems + ITEM_WAVES - 1) / ITEM_WAVES, int64_t(1) << 30);
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
                  tune.bin2 <= tune.bin3 && tune.bin3 <= SMALL_PROD,
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
            const int nr = front.count[bin];
            if (nr <= 0) return;
            hipLaunchKernelGGL(kern, dim3(grid_for(nr, rpb)), dim3(threads), 0, s, nr,
                               front.rows(bin), A.ptr, A.idx, B.ptr, B.idx, front.rownnz);
            TSG_LAUNCH_CHECK();
        };
        launch(k_flat_symbolic<16, 4, 64, 64, 256>, 16, 256, 1);
        launch(k_flat_symbolic<64, 4, 64, 512, 64>, 1, 64, 2);
        launch(k_flat_symbolic<64, 8, 64, 512, 64>, 1, 64, 3);
        launch(k_flat_symbolic<64, 16, 64, 512, 64, 6>, 1, 64, 4);
        launch(k_flat_symbolic<64, 16, 1024, 512, 64>, 1, 64, ROW_BIN_MANY);
    }
    tm.end();

    // big rows
    p.nbig = front.count[ROW_BIN_BIG];
    p.sub_shift = SUB_SHIFT;
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
        int64_t *a_ent = ws.alloc_n<int64_t>((size_t)p.nbig + 1);
        int64_t *a_prod = ws.alloc_n<int64_t>((size_t)p.nbig + 1);
        row_loff = ws.alloc_n<int64_t>((size_t)p.nbig + 1);
        hipLaunchKernelGGL(k_big_span, dim3(grid_for((size_t)p.nbig * 64, 256)), dim3(256), 0, s,
                           p.nbig, rowsb, A.ptr, A.idx, B.ptr, B.idx, front.rowprod, p.span_sb0,
                           p.sb_off, a_ent, a_prod, row_loff);
        TSG_LAUNCH_CHECK();
        hipLaunchKernelGGL(k_band_count, dim3(grid_for((size_t)p.nbig, 256)), dim3(256), 0, s,
                           p.nbig, p.sb_off, band_off);
        TSG_LAUNCH_CHECK();
        exclusive_scan_i64(p.sb_off, p.sb_off, (size_t)p.nbig, tmp_sb, s);
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
        // a radix sort arranges; the block pointers are then laid out block
        // major and the items are 8 sub-blocks wide.
        p.column_order = nsb_total / 16 >= tune.item_sort_min;
        tm.end();

        // B block pointers at the sub-block width (item and band boundaries
        // then need no search) while the table stays <= 6 GiB, coarser beyond.
        // No table at all when building it would cost more than the searches
        // it saves -- more than 8 max(1, log2(L / 16)) entries per (A entry,
        // window of 16 sub-blocks) pair of the big rows, with the pairs
        // estimated from their A entries and average span and L, the mean
        // length of the B rows they reference, from their products per A
        // entry (measured on batches: an entry costs ~5 ps to build, a search
        // ~26 ps in B rows of ~30 entries, which span one or two cache lines,
        // and several times that in rows of hundreds, where each step misses)
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
        p.bptr_rowptr = k <= (1 << 30) &&
                        (tune.bptr_budget == 0 ||
                         (tune.bptr_budget < 0 &&
                          fine_entries > 8.0 * pairs * std::max(1.0, std::log2(brow / 16.0))));
        int bs = SUB_SHIFT;
        while (bs < 30) {
            size_t nblk = ((size_t)k + (1u << bs) - 1) >> bs;
            if ((size_t)n * (nblk + 1) * sizeof(int) <= bptr_cap) break;
            bs++;
        }
        if (p.bptr_rowptr) bs = 30;
        p.blk_shift = bs;
        p.nblk = (int)(((size_t)k + (1u << bs) - 1) >> bs);
        p.bptr = p.bptr_rowptr ? nullptr : ws.alloc_n<int>((size_t)n * (p.nblk + 1));
        if (p.bptr_rowptr) {
            // nothing to build
        } else if (n > 0 && p.column_order) {
            hipLaunchKernelGGL(k_bptr, dim3(grid_for((size_t)n, BPT_ROWS)), dim3(256), 0, s, n,
                               B.ptr, B.idx, p.nblk, bs, p.bptr);
            TSG_LAUNCH_CHECK();
        } else if (n > 0) {
            hipLaunchKernelGGL(k_bptr_rows, dim3(grid_for((size_t)n * 64, 256)), dim3(256), 0,
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
        hipLaunchKernelGGL(k_big_symbolic,
                           dim3((unsigned)std::min<int64_t>(nunits, int64_t(1) << 30)),
                           dim3(BAND_T), 0, s, nunits, units, rowsb, k, A.ptr, A.idx, B.ptr,
                           B.idx, block_ptrs(p, B.ptr), p.span_sb0, p.sb_off, p.subcnt, front.rownnz,
                           band_off, band_base, row_cur, row_loff, d_overflow, p.subocc,
                           p.bandwords);
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
        const int wide_cap = narrow && p.use_rank ? WIDE_CAP : 0;
        auto items_kernel = [&](auto kern, int64_t *cnt, ItemRec *it, int *itn) {
            hipLaunchKernelGGL(kern, dim3(grid_for((size_t)p.nbig * 64, 256)), dim3(256), 0, s,
                               p.nbig, rowsb, k, wide_cap, p.span_sb0, p.sb_off, p.subcnt, d_ic, cnt, it,
                               itn, p.subocc, band_off, band_base);
            TSG_LAUNCH_CHECK();
        };
        if (narrow)
            items_kernel(k_items<false, 8>, p.item_cnt, nullptr, nullptr);
        else
            items_kernel(k_items<false, 16>, p.item_cnt, nullptr, nullptr);
        exclusive_scan_i64(p.item_cnt, p.item_cnt, (size_t)p.nbig, tmp2, s);
        publish_i64({{p.item_cnt + p.nbig, d_overflow}}, d_overflow ? 2 : 1, box, s);
        TSG_HIP_TRY(hipStreamSynchronize(s));
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
        p.nitems_small = 0;
        p.nitems_mid = 0;
        if (p.column_order && p.nitems > 1 && p.nitems < (int64_t(1) << 31)) {
            const size_t ni = (size_t)p.nitems;
            int *keys = ws.alloc_n<int>(ni);
            int *order = ws.alloc_n<int>(ni);
            const unsigned kblocks = grid_for(ni, 256);
            int *bsmall = ws.alloc_n<int>((size_t)kblocks + 1);
            int *bmid = ws.alloc_n<int>((size_t)kblocks + 1);
            int64_t *tmpk = ws.alloc_n<int64_t>(scan_tmp_elems((size_t)kblocks + 1));
            int64_t *d_small = ws.alloc_n<int64_t>(2);
            int end_bit = 1;
            while (end_bit < 29 && (int64_t(1) << end_bit) <= ((int64_t)k >> SUB_SHIFT)) end_bit++;
            // the size class splits the rank path's items only
            hipLaunchKernelGGL(k_item_keys, dim3(kblocks), dim3(256), 0, s, p.nitems,
                               p.items, item_n, p.use_rank ? end_bit : -1, keys, bsmall, bmid);
            TSG_LAUNCH_CHECK();
            exclusive_scan_i32(bsmall, bsmall, (size_t)kblocks, tmpk, s, d_small);
            exclusive_scan_i32(bmid, bmid, (size_t)kblocks, tmpk, s, d_small + 1);
            sort_order_i32(keys, p.nitems, p.use_rank ? end_bit + 2 : end_bit, order, ws, s);
            ItemRec *items_s = ws.alloc_n<ItemRec>(ni + 1);
            hipLaunchKernelGGL(k_gather_items, dim3(grid_for(ni, 256)), dim3(256), 0, s,
                               p.nitems, order, p.items, items_s);
            TSG_LAUNCH_CHECK();
            p.items = items_s;
            if (p.use_rank) {
                publish_i64({{d_small, d_small + 1}}, 2, box, s);
                TSG_HIP_TRY(hipStreamSynchronize(s));
                p.nitems_small = box->v[0];
                p.nitems_mid = box->v[0] + box->v[1];
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
            const int nr = front.count[bin];
            if (nr <= 0) return;
            hipLaunchKernelGGL(kern, dim3(grid_for(nr, rpb)), dim3(threads), 0, s, nr,
                               front.rows(bin), A.ptr, A.idx, A.val, B.ptr, B.idx, B.val, d_ic,
                               d_jc, d_c, (int)p.b_strict);
            TSG_LAUNCH_CHECK();
        };
        launch(k_flat_numeric<FUSED, 16, 4, 64, 64, 64, 256>, 16, 256, 1);
        launch(k_flat_numeric<FUSED, 64, 4, 64, 512, 256, 64>, 1, 64, 2);
        launch(k_flat_numeric<FUSED, 64, 8, 64, 512, 512, 64>, 1, 64, 3);
        launch(k_flat_numeric<FUSED, 64, 16, 64, 512, 512, 64>, 1, 64, 4);
        launch(k_flat_numeric<FUSED, 64, 16, 1024, 512, 512, 64>, 1, 64, ROW_BIN_MANY);
    }
    tm.end();
    if (p.nitems > 0 && p.use_rank) {
        tm.begin("row.big_numeric");
        if (B.nnz > 0) {
            hipLaunchKernelGGL(k_pack_b, dim3(grid_for((size_t)B.nnz, 256)), dim3(256), 0, s,
                               B.nnz, B.idx, B.val, p.bpk);
            TSG_LAUNCH_CHECK();
        }
        auto launch_rank = [&](auto kern, size_t sm, int64_t i0, int64_t i1) {
            if (i1 <= i0) return;
            set_smem(kern, sm);
            const unsigned grid = item_grid(i1 - i0);
            hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * ITEM_WAVES), sm, s, i1 - i0,
                               p.items + i0, p.bandwords, p.subocc, A.ptr, A.idx, A.val, B.idx, B.val, p.bpk, block_ptrs(p, B.ptr),
                               d_jc, d_c, (int)p.b_strict);
            TSG_LAUNCH_CHECK();
        };
        // the size classes (sorted in this order) in kernels with value
        // arrays of their size
        const int64_t ns = p.nitems_small, nm = std::max(p.nitems_mid, ns);
        auto launch_sparse = [&](auto kern, int64_t i0, int64_t i1) {
            if (i1 <= i0) return;
            hipLaunchKernelGGL(kern, dim3(item_grid(i1 - i0)), dim3(64), 0, s, i1 - i0,
                               p.items + i0, p.bandwords, p.subocc, A.ptr, A.idx, A.val, B.idx,
                               p.bpk, block_ptrs(p, B.ptr), d_jc, d_c, (int)p.b_strict);
            TSG_LAUNCH_CHECK();
        };
        launch_sparse(k_big_numeric_sparse<FUSED, SMALL_ITEM, SMALL_RANK_U, SMALL_MINW>, 0, ns);
        launch_sparse(k_big_numeric_sparse<FUSED, MID_ITEM, MID_RANK_U, MID_MINW>, ns, nm);
        // the rest: items of more outputs in column order, all in rows' order
        if (p.narrow_items) {
            constexpr int W = ITEM_WORDS / 2;
            launch_rank(k_big_numeric_rank<FUSED, W>, sizeof(RankSmem<W>) * ITEM_WAVES, nm,
                        p.nitems);
        } else {
            constexpr int W = ITEM_WORDS;
            launch_rank(k_big_numeric_rank<FUSED, W>, sizeof(RankSmem<W>) * ITEM_WAVES, nm,
                        p.nitems);
        }
        tm.end();
    } else if (p.nitems > 0) {
        tm.begin("row.big_numeric");
        constexpr size_t sm = sizeof(ItemSmem) * ITEM_WAVES;
        auto kern = k_big_numeric<FUSED>;
        set_smem(kern, sm);
        const unsigned grid = item_grid(p.nitems);
        hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * ITEM_WAVES), sm, s, p.nitems, p.items,
                           A.ptr, A.idx, A.val, B.ptr, B.idx, B.val, block_ptrs(p, B.ptr),
                           d_jc, d_c, (int)p.b_strict);
        TSG_LAUNCH_CHECK();
        tm.end();
    }
}

void row_numeric(RowPlan &p, const CsrIn &A, const CsrIn &B, const int64_t *d_ic, int *d_jc,
                 double *d_c, int fused, Arena & /*ws*/, hipStream_t s, StageTimer &tm,
                 int /*cus*/) {
    TSG_CHECK(p.valid && p.m == A.rows && p.n == A.cols && p.k == B.cols, TSG_ERR_STATE,
              "row numeric phase without a matching symbolic phase");
    if (fused)
        row_numeric_t<true>(p, A, B, d_ic, d_jc, d_c, s, tm);
    else
        row_numeric_t<false>(p, A, B, d_ic, d_jc, d_c, s, tm);
}
