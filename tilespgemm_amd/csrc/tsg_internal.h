// Internal declarations shared by the tsg HIP sources (gfx950, wave64).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stddef.h>
#include <functional>
#include <string>
#include <vector>

#include "../../include/tsg.h"

// ------------------------------------------------------------ error plumbing
struct TsgError {
    int code;
    std::string msg;
};

#define TSG_HIP_TRY(expr)                                                      \
    do {                                                                       \
        hipError_t _e = (expr);                                                \
        if (_e != hipSuccess)                                                  \
            throw TsgError{TSG_ERR_HIP, std::string(#expr) + ": " +            \
                                            hipGetErrorString(_e)};            \
    } while (0)

#define TSG_CHECK(cond, code, text)                                            \
    do {                                                                       \
        if (!(cond)) throw TsgError{(code), (text)};                           \
    } while (0)

// Launch check: surfaces bad launch configurations immediately.
#define TSG_LAUNCH_CHECK() TSG_HIP_TRY(hipGetLastError())

// -------------------------------------------------------------- workspace
// Chunked bump arena over hipMalloc'd blocks.  reset() keeps the blocks, so
// repeated calls of the same size reach a steady state with no allocation.
// An arena attached to an external block (attach) bumps inside that block
// only: it never calls hipMalloc or hipFree, and a request past the block's
// end throws TSG_ERR_ALLOC instead of growing.
class Arena {
public:
    Arena() = default;
    Arena(const Arena &) = delete;
    Arena &operator=(const Arena &) = delete;
    ~Arena();
    void reset();
    void *alloc(size_t bytes);
    template <class T> T *alloc_n(size_t n) {
        return static_cast<T *>(alloc(n * sizeof(T) + 1));
    }
    size_t held() const { return held_; }
    void release();
    // Serve every allocation from [base, base + bytes) (256-byte aligned);
    // what is held is dropped first.
    void attach(void *base, size_t bytes, const char *what);
    size_t used() const;
    // What is allocated after a mark is given back by rewinding to it.
    struct Mark { size_t cur, used; };
    Mark mark() const;
    void rewind(Mark m);

private:
    struct Block { char *base; size_t size; size_t used; };
    std::vector<Block> blocks_;
    size_t cur_ = 0;
    size_t held_ = 0;
    bool external_ = false;
    const char *what_ = "";
};

// -------------------------------------------------------------- scans
// Exclusive scan of n int64 counts in place into out[0..n] (out[n] = total).
// in and out may alias.  tmp must hold scan_tmp_elems(n) int64.
size_t scan_tmp_elems(size_t n);
// With total set, the grand total is written there too (device memory, or
// host memory the device can write).
void exclusive_scan_i64(const int64_t *in, int64_t *out, size_t n, int64_t *tmp,
                        hipStream_t s, int64_t *total = nullptr);
// The int32 scan sums in int64; with total set, the exact int64 grand total
// is written there too (the caller checks it against INT32_MAX).
void exclusive_scan_i32(const int32_t *in, int32_t *out, size_t n, int64_t *tmp,
                        hipStream_t s, int64_t *total = nullptr);

// -------------------------------------------------------------- helpers
static inline unsigned grid_for(size_t work, unsigned per_block, unsigned cap = 1u << 30) {
    size_t g = (work + per_block - 1) / per_block;
    if (g < 1) g = 1;
    if (g > cap) g = cap;
    return (unsigned)g;
}

// A launch holds fewer than 2^32 threads; past them the count wraps, without an
// error.  Work that can take as many either goes through a grid of at most
// MAX_GRID blocks of 256 threads in steps, or in launches of at most 2^31
// threads, per items a block of the threads: f(first item, items).
constexpr unsigned MAX_GRID = 1u << 23;
template <class F>
void in_launches(int64_t items, int per, int threads, F &&f) {
    const int64_t most = (int64_t(1) << 31) / threads * per;
    for (int64_t i = 0; i < items; i += most) f(i, (int)(items - i < most ? items - i : most));
}

// 16x16 tiles that n rows or columns take.
__host__ __device__ __forceinline__ int tiles_of(int n) { return (n >> 4) + ((n & 15) != 0); }
// End of the rows [16 I, 16 I + 16 t) of m (16 I < m).
__host__ __device__ __forceinline__ int tile_rows_end(int I, int t, int m) {
    return m - 16 * I > 16 * t ? 16 * (I + t) : m;
}

// Input description shared by both paths.
struct CsrIn {
    int rows, cols;
    const int *ptr;
    const int *idx;
    const double *val;   // may be null in the symbolic phase
    int64_t nnz;
};

// Stage timer: records (name, start, stop) HIP events on a stream.
struct StageTimer {
    bool enabled = false;
    hipStream_t stream = nullptr;
    std::vector<std::string> names;
    std::vector<hipEvent_t> ev;          // 2 per stage
    std::vector<double> ms;
    void clear();
    void begin(const char *name);
    void end();
    void finalize();                     // synchronizes, fills ms
    ~StageTimer();
};

// ---------------------------------------------------------- host results
// Host memory of a handle that kernels write their small results into: they
// are there once the stream is synchronized, with no copy in between.
constexpr int ROW_BINS = 8;
struct alignas(256) HostBox {
    unsigned flags[2];
    int bins[ROW_BINS];
    unsigned long long sample[2];
    int64_t v[8];
};
// Up to 8 int64 values of device memory into box->v.
struct PublishList { const int64_t *p[8]; };
void publish_i64(const PublishList &src, int n, HostBox *box, hipStream_t s);

// ------------------------------------------------------------ row path
// Row bins by intermediate products: (0, l1] -> 16 lanes a row, (l1, l2],
// (l2, ROW_MID_PROD] and (ROW_MID_PROD, l3] -> a wave a row with 4, 8 and 16
// products a lane (those with more than ROW_FLAT_ENT A entries in a bin of
// their own), (l3, l4] -> 24 a lane if at most ROW_FLAT_ENT entries, the rest
// -> the big-row path.  l4 is ROW_MED_PROD at the full l3, else l3.  ER batch of
// 512 (a tenth of its products in rows of 1025 to 1536): 7.2 ms in the big-row
// path, 3.5 here, at 4 waves per SIMD (3.8 at 3); R-MAT 2^20 with 8 draws a row
// 2.0 and 0.75.
// Each small kernel is exact for
// any row up to its register count, so any limits with l1 <= 64, l2 <= 256,
// l3 <= 1024 (checked on the host) are valid; they are tuning parameters
// (tsg_set_row_bins).
constexpr int ROW_MID_PROD = 512;
constexpr int ROW_FLAT_ENT = 64;
constexpr int ROW_SMALL_PROD = 1024;   // the largest l3
constexpr int ROW_MED_PROD = 1536;
constexpr int ROW_LISTS = ROW_BINS / 2;
constexpr int ROW_BIN_MANY = 5;
constexpr int ROW_BIN_MED = 6;
constexpr int ROW_BIN_BIG = 7;
struct RowBinLimits { int l1, l2, l3, l4; };

__host__ __device__ inline int row_bin_of(int64_t prod, int entries, RowBinLimits lim) {
    if (prod == 0) return 0;
    if (prod <= lim.l1) return 1;
    if (prod > lim.l4) return ROW_BIN_BIG;
    if (prod > lim.l3) return entries <= ROW_FLAT_ENT ? ROW_BIN_MED : ROW_BIN_BIG;
    if (entries > ROW_FLAT_ENT) return ROW_BIN_MANY;
    if (prod <= lim.l2) return 2;
    return prod <= ROW_MID_PROD ? 3 : 4;
}

// The row path's share of the first pass over the operands: products per row
// and the rows of each bin.  Bins 2k + 1 and 2k + 2 share a list, one from its
// front, the other from its back.
struct RowFront {
    int64_t *rowprod = nullptr;      // [m]
    int64_t *rownnz = nullptr;       // [m+1] zero for rows of bin 0 and big rows
    int *list[ROW_LISTS] = {};
    int nlist = 0;                   // ints of each list
    int count[ROW_BINS] = {0};       // (host) rows per bin
    const int *rows(int bin) const {
        return list[(bin - 1) >> 1] + ((bin & 1) ? 0 : nlist - count[bin]);
    }
};

// Tuning parameters of the row path (tsg_set_row_bins): rows with at most
// bin1 products take 16 lanes each, up to bin2 and bin3 a wave each, the rest
// go to the big-row path.
struct RowTuning {
    int bin1 = 64, bin2 = 256, bin3 = 1024;
    int64_t item_sort_min = int64_t(1) << 18;  // big-row items column-ordered from this many
    int64_t bitmap_budget = -1;  // bytes of big-row bitmaps (sparse form) kept; < 0: min(48 GiB, 40% of free)
    int64_t bptr_budget = -1;    // bytes of B's block pointers or run directory; < 0: 6 GiB
};

// One big-row item: d = {row, first column, end column, first sub-block in
// subocc (rank mode)}, the position of its first output in
// C, and of its first word in the band word lists (rank mode).  One record,
// so that gathering the items into column order reads one line per item.
struct ItemRec {
    int4 d;
    int64_t off;
    int64_t wpos;
};
static_assert(sizeof(ItemRec) == 32, "item records are 32 bytes");

// Run directory of B, for work in column order.  The columns are cut in
// blocks of 1 << shift, of 2 << shift and so on, up to a band: level v's
// blocks are 1 << (shift + v) columns wide.  A run is a B row's entries in one
// block; block b of level v has a cell for every 32 B rows: which of them have
// a run there, and the number of runs of earlier cells, so row t's run is
// found in runs[] ({first, end} positions in B) by counting bits.  An item's
// rows then cost a lookup in one block's cells (256 KB for 2^20 rows, which
// stay in L2) and, for rows with a run only, one in its runs; block pointers
// cost two reads from 4 MB each.  Level v's blocks are cells[blocks before v +
// b], blocks before v = 2 nblk - (2 nblk >> v).
struct RunDir {
    const uint2 *cells = nullptr;
    const int2 *runs = nullptr;
    int ngrp = 0;                  // cells a block
    int nblk = 0;                  // blocks of level 0 (whole bands)
    int shift = 0;
    int coarse = 0;                // blocks of level 0 may be wider than items
};

__host__ __device__ __forceinline__ int64_t run_dir_block(int nblk, int shift, int v, int c) {
    return 2ll * nblk - (2ll * nblk >> v) + (c >> (shift + v));
}

// Sub-blocks of the big rows' columns: first column of the sb-th, k past the
// matrix's last (2^31 itself does not fit an int).
constexpr int SUB_SHIFT = 10;          // 1024 columns
__host__ __device__ __forceinline__ int sub_block_start(int sb, int k) {
    return sb <= (k - 1) >> SUB_SHIFT ? sb << SUB_SHIFT : k;
}

// log2 of the finest blocks of the run directory in the handle's plan, 0
// without one (not in the public header: the tests tell the forms apart by it).
extern "C" int tsg_plan_dir_shift(tsg_handle_t handle);

constexpr int ITEM_CLASSES = 3;       // size classes of the row path's items

struct RowPlan {
    bool valid = false;
    bool b_strict = false;           // B rows strictly ascending (no duplicates)
    int m = 0, n = 0, k = 0;
    RowFront front;                  // products per row, rows per bin
    // big-row structures
    int nbig = 0;
    int64_t big_ent = 0, big_prod = 0;   // the big rows' A entries and products
    int64_t *ent_off = nullptr;      // [nbig+1] A entries of the big rows before each
    int *span_sb0 = nullptr;         // [nbig] first sub-block of the row's span
    int64_t *sb_off = nullptr;       // [nbig+1] span offsets (sub-blocks)
    int64_t nsb_total = 0;
    uint16_t *subcnt = nullptr;      // [nsb_total] outputs per span sub-block
    // B's rows cut to big-row bands and items: by the run directory (column
    // order) or the block-pointer table; with neither, B's row pointers serve
    // as a table of one block
    RunDir dir;
    int blk_shift = 0;               // log2 block width (columns)
    int nblk = 0;                    // blocks per B row (+1 stored)
    int *bptr = nullptr;             // [(nblk+1) * n]
    bool column_order = false;       // big-row bands and items run in column order
    // items
    int64_t nitems = 0;
    int64_t class_end[ITEM_CLASSES - 1] = {};   // ends of the items' classes but the last
    int64_t *item_cnt = nullptr;     // [nbig+1] items per big row -> offsets
    ItemRec *items = nullptr;        // by c0 (column order) or by row
    bool narrow_items = false;       // items of <= 8192 columns (else <= 16384)
    // big rows' column bitmaps kept from the symbolic phase (rank mode), in
    // sparse form: per sub-block a mask of its non-empty words, and per
    // 65536-column band those words in column order (a band word list),
    // bands placed in their row's region as they finished
    bool use_rank = false;
    int64_t words_cap = 0;           // words of bandwords (a bound)
    unsigned *bandwords = nullptr;   // [words_cap]
    unsigned *subocc = nullptr;      // [nsb_total] non-empty-word masks

    int4 *bpk = nullptr;             // [nnz(B)] {column, 0, value} records (rank mode)

    // B with rows sorted, when the input's were not (set after row_symbolic):
    // the plan ran on (B.ptr, b_idx); numeric phases gather values by b_perm
    bool b_canon = false;
    int *b_idx = nullptr;
    int *b_perm = nullptr;
    double *b_val = nullptr;
};

void row_symbolic(RowPlan &p, const CsrIn &A, const CsrIn &B, int64_t *d_ic,
                  int64_t *nnz_c, const RowFront &front, HostBox *box, Arena &ws, hipStream_t s,
                  StageTimer &tm, const RowTuning &tune);
void row_numeric(RowPlan &p, const CsrIn &A, const CsrIn &B, const int64_t *d_ic,
                 int *d_jc, double *d_c, int fused, hipStream_t s, StageTimer &tm);

// ------------------------------------------------------------ tile path
// One tile's numeric-phase metadata in 64 bytes (one aligned half line), so
// a matched pair's two tiles cost two reads.  A tiles: row masks (bit 15-c)
// and row starts of the row-major payload; B tiles: column masks (bit 15-k)
// and column starts of the column-major payload.
struct TileRec {
    uint16_t mask[16];
    uint8_t start[16];
    int off;                     // payload offset of the tile
    int pad[3];
};
static_assert(sizeof(TileRec) == 64, "tile records are 64 bytes");

struct TileMat {
    int rows = 0, cols = 0, blkm = 0, blkn = 0, numblk = 0;
    int *tile_ptr = nullptr;     // [blkm+1]
    int *tile_col = nullptr;     // [numblk]
    int *tile_off = nullptr;     // [numblk+1]
    uint16_t *mask = nullptr;    // [16*numblk]
    uint8_t *rowptr = nullptr;   // [16*numblk]
    uint8_t *idx = nullptr;      // [nnz]
    double *val = nullptr;       // [nnz]
    int64_t nnz = 0;
    // tile-CSC index (B only)
    int *csc_ptr = nullptr;      // [blkn+1]
    int *csc_row = nullptr;      // [numblk]
    int *csc_tile = nullptr;     // [numblk]
    TileRec *rec = nullptr;      // [numblk] A: row layout; B: column layout
    // entry -> payload position permutation (values refreshed per numeric)
    int *perm = nullptr;         // [nnz] CSR position -> tile payload position
    int *permc = nullptr;        // [nnz] CSR position -> column-major payload position (B only)
    double *valc = nullptr;      // [nnz] values column-major inside each tile (B only)
};

struct TilePlan {
    bool valid = false;
    bool b_is_a = false;         // B has A's structure (same index arrays)
    TileMat A, B;
    int numblkC = 0;
    int *tptrC = nullptr;        // [blkm+1]
    int *tcolC = nullptr;        // [numblkC]
    int *trowC = nullptr;        // [numblkC]
    uint16_t *maskC = nullptr;   // [16*numblkC]
    uint8_t *rowptrC = nullptr;  // [16*numblkC]
    int64_t *offC = nullptr;     // [numblkC+1] payload offsets (tile order)
    int *rowoffC = nullptr;      // [numblkC*16] start of (tile,row) inside CSR row
    int64_t *rownnz = nullptr;   // [m+1] CSR row counts
    int64_t nnzC = 0;
    // matched (A tile, B tile) pairs of every C tile in ascending K
    int64_t *tpair = nullptr;    // [numblkC+1] offsets into pairs, or counts with tslot
    int64_t *tslot = nullptr;    // [numblkC] first pair of each C tile (pairs in slots)
    int2 *pairs = nullptr;       // [npairs] {A tile position, B tile position}
    int64_t npairs = 0;
    // numeric work units (tile * 4 + part) by C tile output count: bins 0..3
    // (<= 16, <= 32, <= 64, 64-output parts of larger tiles) back to back,
    // tiles without outputs left out
    int4 *tbin_units = nullptr;      // [units] {tile, part | pairs << 2, first pair (lo, hi)}
    int tbin_start[5] = {0, 0, 0, 0, 0};
};

// Throws TSG_ERR_OVERFLOW unless 0 <= n_c_tiles <= INT32_MAX.
void check_tile_count(int64_t n_c_tiles);
// A matrix's tile count per tile row, scanned, enqueued ahead of the tile
// path (beside the input's validation, whose host round trip then brings
// the total back into nt): the count clamps every index, so it is safe on
// unchecked input.  tile_ptr and nt are used only once the input is valid.
struct EarlyTileCount {
    int *tile_ptr = nullptr;     // [blkm+1] device
    int nt = -1;                 // host, after the round trip
};
void tile_count_early(const CsrIn &X, EarlyTileCount &e, int64_t *total, Arena &ws,
                      hipStream_t s);
void tile_symbolic(TilePlan &p, const CsrIn &A, const CsrIn &B, bool b_is_a,
                   int64_t *d_ic, int64_t *nnz_c, HostBox *box, Arena &ws, hipStream_t s,
                   StageTimer &tm, const EarlyTileCount *earlyA = nullptr,
                   const EarlyTileCount *earlyB = nullptr);
void tile_numeric(TilePlan &p, const CsrIn &A, const CsrIn &B, const int64_t *d_ic,
                  int *d_jc, double *d_c, int fused, hipStream_t s, StageTimer &tm);

// ------------------------------------------------------------ batches
// A batch laid out as one block-diagonal product (tsg_batch.hip).
struct BatchState {
    bool valid = false;
    int count = 0;
    bool b_is_a = false;
    bool local_cols = false;                   // B (and so C) keeps each product's own columns
    int rows = 0, cols_a = 0, cols_b = 0;     // sum m, sum n; columns of C (see local_cols)
    int64_t nnz_a = 0, nnz_b = 0;
    void *desc = nullptr;                      // device descriptors
    int64_t *row_off = nullptr;                // [count+1] C/A row offsets
    int *ia = nullptr, *ja = nullptr, *ib = nullptr, *jb = nullptr;
    double *a = nullptr, *b = nullptr;
    std::vector<tsg_product_t> host;           // structure identity check
};

// ------------------------------------------------------------ handle
struct tsg_handle_s {
    int device = 0;
    hipStream_t stream = nullptr;
    hipStream_t own_stream = nullptr;
    int method = TSG_METHOD_AUTO;
    int fp_mode = TSG_FP_FUSED;
    int method_used = TSG_METHOD_AUTO;
    double tile_density = 32.0;  // AUTO: tile path from this many entries per tile
    RowTuning row_tune;
    Arena ws;       // plan of the last symbolic phase
    Arena bws;      // batch layout (outlives the plan's reset)
    Arena aux;      // scratch of utility calls (transpose, product counts)
    HostBox *box = nullptr;   // pinned; results of the phases' kernels
    RowPlan row;
    TilePlan tile;
    BatchState batch;
    StageTimer tm;
    std::string err;
};

void batch_symbolic(tsg_handle_t h, int count, const tsg_product_t *prods, int64_t *d_ic,
                    int64_t *nnz_c_total, int64_t *nnz_c);
void batch_numeric(tsg_handle_t h, int count, const tsg_product_t *prods, const int64_t *d_ic,
                   int *d_jc, double *d_c);
// Row pointers of every product of the last batch rebased to start at 0,
// m_i + 1 entries each, back to back (rows + count entries).
void batch_rebase(tsg_handle_t h, const int64_t *d_ic, int64_t *d_out);

// CSR utilities
// First pass over the operands (tsg_front.hip): checks of A and B on the
// device, one host round trip (flags: A in bits 0-7, B in bits 8-15; 1 bad row
// pointers, 2 column out of range, 4 not strictly ascending).  With
// density_sample, the {tiles, entries} of a sample of A's tile rows; with rows
// (and tune), the row path's products and bins.  before_sync enqueues more
// work (and read-backs) ahead of the round trip.
int front_pass(const CsrIn &A, const CsrIn &B, Arena &ws, hipStream_t s, HostBox *box,
               unsigned long long *density_sample = nullptr, RowFront *rows = nullptr,
               const RowTuning *tune = nullptr, const std::function<void()> &before_sync = {});
// entries per non-empty 16x16 tile of X (tsg_tile.hip; a sample of every
// tile_sample_step-th tile row decides when clear of the threshold)
int tile_sample_step(int blkm);
double tile_density(const CsrIn &X, double threshold, Arena &ws, hipStream_t s,
                    const unsigned long long *sample = nullptr);
void csr_transpose(int m, int n, const int *ia, const int *ja, const double *a,
                   int64_t nnz, int *tp, int *ti, double *tv, Arena &ws,
                   hipStream_t s, int *tpos = nullptr);
// Row-sorted copy of X's columns (stable: equal columns keep their order) and
// the original position of every sorted entry; temporaries from tmp.
void csr_sort_rows(int m, int n, const int *ia, const int *ja, int64_t nnz, int *sorted_ja,
                   int *perm, Arena &tmp, hipStream_t s);
void gather_values(int64_t n, const int *perm, const double *src, double *dst, hipStream_t s);
void sort_order_i32(const int *keys, int64_t n, int end_bit, int *order, Arena &ws,
                    hipStream_t s);
void csr_row_products(int m, const int *ia, const int *ja, int64_t nnz, const int *ib,
                      int64_t *rowprod, Arena &ws, hipStream_t s);
