// Utilities: workspace arena, device-wide scans, stage timer, CSR transpose,
// intermediate-product counts.
#include "tsg_internal.h"
#include "tsg_device.h"

#include <algorithm>
#include <cstring>
#include <rocprim/rocprim.hpp>

// ================================================================= arena
Arena::~Arena() { release(); }

void Arena::release() {
    if (!external_)
        for (auto &b : blocks_) (void)hipFree(b.base);
    blocks_.clear();
    cur_ = 0;
    held_ = 0;
    external_ = false;
}

void Arena::attach(void *base, size_t bytes, const char *what) {
    release();
    external_ = true;
    what_ = what;
    blocks_.push_back(Block{static_cast<char *>(base), bytes & ~size_t(255), 0});
}

size_t Arena::used() const {
    size_t u = 0;
    for (const auto &b : blocks_) u += b.used;
    return u;
}

void Arena::reset() {
    for (auto &b : blocks_) b.used = 0;
    cur_ = 0;
}

Arena::Mark Arena::mark() const {
    return Mark{cur_, cur_ < blocks_.size() ? blocks_[cur_].used : 0};
}

void Arena::rewind(Mark m) {
    for (size_t i = m.cur + 1; i < blocks_.size(); i++) blocks_[i].used = 0;
    if (m.cur < blocks_.size()) blocks_[m.cur].used = m.used;
    cur_ = m.cur;
}

void *Arena::alloc(size_t bytes) {
    bytes = (bytes + 255) & ~size_t(255);
    while (cur_ < blocks_.size()) {
        Block &b = blocks_[cur_];
        if (b.size - b.used >= bytes) {
            void *p = b.base + b.used;
            b.used += bytes;
            return p;
        }
        cur_++;
    }
    if (external_)
        throw TsgError{TSG_ERR_ALLOC, std::string(what_) + " of " +
                                          std::to_string(blocks_.empty() ? 0 : blocks_[0].size) +
                                          " bytes exhausted: " + std::to_string(used()) +
                                          " bytes in use, " + std::to_string(bytes) +
                                          " more needed"};
    size_t sz = std::max(bytes, size_t(64) << 20);
    void *p = nullptr;
    hipError_t e = hipMalloc(&p, sz);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        throw TsgError{TSG_ERR_ALLOC, "workspace hipMalloc of " + std::to_string(sz) +
                                          " bytes failed: " + hipGetErrorString(e)};
    }
    blocks_.push_back(Block{static_cast<char *>(p), sz, bytes});
    cur_ = blocks_.size() - 1;
    held_ += sz;
    return p;
}

// ================================================================= scans
// Exclusive scan: per-block totals, then a rescan of each block with its
// offset, which up to SCAN_FLAT blocks add up themselves from the totals (a
// launch less: whole ER products of 16,000 rows 97.0 -> 94.0 us, of 2^20 840 ->
// 826; at 512 or 8192 blocks the same); past that the totals are scanned first, recursively.  1024
// elements per 256-thread block (4 per thread).
namespace {
constexpr int SCAN_T = 256;
constexpr int SCAN_PER = 4;
constexpr int SCAN_BLK = SCAN_T * SCAN_PER;
constexpr size_t SCAN_FLAT = 2048;

template <class T>
__device__ __forceinline__ long long block_excl_scan(long long x, long long *total) {
    __shared__ long long wsum[SCAN_T / 64];
    long long inc = wave_incl_scan64(x);
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    if (l == 63) wsum[w] = inc;
    __syncthreads();
    long long off = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < SCAN_T / 64; i++) {
        if (i < w) off += wsum[i];
        tot += wsum[i];
    }
    __syncthreads();
    *total = tot;
    return off + inc - x;
}

template <class T>
__global__ void __launch_bounds__(SCAN_T) k_scan_reduce(const T *in, size_t n, long long *sums) {
    size_t base = (size_t)blockIdx.x * SCAN_BLK + threadIdx.x * SCAN_PER;
    long long s = 0;
#pragma unroll
    for (int i = 0; i < SCAN_PER; i++)
        if (base + i < n) s += (long long)in[base + i];
    long long tot;
    (void)block_excl_scan<T>(s, &tot);
    if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

template <class T>
__global__ void __launch_bounds__(SCAN_T) k_scan_apply(const T *in, T *out, size_t n,
                                                        const long long *offs, int has_offs,
                                                        long long *total) {
    size_t base = (size_t)blockIdx.x * SCAN_BLK + threadIdx.x * SCAN_PER;
    T v[SCAN_PER];
    long long s = 0;
#pragma unroll
    for (int i = 0; i < SCAN_PER; i++) {
        v[i] = base + i < n ? in[base + i] : T(0);
        s += (long long)v[i];
    }
    long long tot;
    long long ex = block_excl_scan<T>(s, &tot);
    long long before = 0;              // of earlier blocks: 1 scanned, 2 totals
    if (has_offs == 1) before = offs[blockIdx.x];
    if (has_offs == 2) {
        long long part = 0;
        for (unsigned i = threadIdx.x; i < blockIdx.x; i += SCAN_T) part += offs[i];
        (void)block_excl_scan<T>(part, &before);
    }
    long long run = ex + before;
#pragma unroll
    for (int i = 0; i < SCAN_PER; i++) {
        if (base + i < n) out[base + i] = (T)run;
        run += (long long)v[i];
    }
    // out[n] = grand total, written by the thread that owns element n-1; the
    // exact 64-bit total also goes to *total when asked for (T may be narrower)
    if (n > 0 && base <= n - 1 && n - 1 < base + SCAN_PER) {
        out[n] = (T)run;
        if (total) *total = run;
    }
    if (n == 0 && blockIdx.x == 0 && threadIdx.x == 0) {
        out[0] = T(0);
        if (total) *total = 0;
    }
}

size_t level_elems(size_t n) { return (n + SCAN_BLK - 1) / SCAN_BLK; }

template <class T>
void scan_rec(const T *in, T *out, size_t n, long long *tmp, hipStream_t s,
              long long *total = nullptr) {
    size_t nb = level_elems(n);
    if (nb <= 1) {
        hipLaunchKernelGGL(k_scan_apply<T>, dim3(1), dim3(SCAN_T), 0, s, in, out, n,
                           (const long long *)nullptr, 0, total);
        TSG_LAUNCH_CHECK();
        return;
    }
    long long *sums = tmp;
    long long *rest = tmp + nb + 1;
    hipLaunchKernelGGL(k_scan_reduce<T>, dim3((unsigned)nb), dim3(SCAN_T), 0, s, in, n, sums);
    TSG_LAUNCH_CHECK();
    const bool flat = nb <= SCAN_FLAT;
    if (!flat) scan_rec<long long>(sums, sums, nb, rest, s);
    hipLaunchKernelGGL(k_scan_apply<T>, dim3((unsigned)nb), dim3(SCAN_T), 0, s, in, out, n,
                       (const long long *)sums, flat ? 2 : 1, total);
    TSG_LAUNCH_CHECK();
}
}  // namespace

size_t scan_tmp_elems(size_t n) {
    size_t total = 0;
    size_t nb = level_elems(n);
    while (nb > 1) {
        total += nb + 1;
        nb = level_elems(nb);
    }
    return total + 8;
}

// The apply pass reads in[] before any block writes out[] only within its own
// block range, so in == out is safe: every block reads its elements before
// writing them, and out[n] lies outside every block's input range.
void exclusive_scan_i64(const int64_t *in, int64_t *out, size_t n, int64_t *tmp, hipStream_t s,
                        int64_t *total) {
    scan_rec<long long>((const long long *)in, (long long *)out, n, (long long *)tmp, s,
                        (long long *)total);
}

__global__ void __launch_bounds__(64) k_publish(PublishList src, int n,
                                                int64_t *__restrict__ out) {
    const int t = threadIdx.x;
    if (t < n) out[t] = *src.p[t];
}

void publish_i64(const PublishList &src, int n, HostBox *box, hipStream_t s) {
    hipLaunchKernelGGL(k_publish, dim3(1), dim3(64), 0, s, src, n, box->v);
    TSG_LAUNCH_CHECK();
}

void exclusive_scan_i32(const int32_t *in, int32_t *out, size_t n, int64_t *tmp, hipStream_t s,
                        int64_t *total) {
    scan_rec<int>(in, out, n, (long long *)tmp, s, (long long *)total);
}

// ================================================================= timer
void StageTimer::clear() {
    for (auto e : ev) (void)hipEventDestroy(e);
    ev.clear();
    names.clear();
    ms.clear();
}

void StageTimer::begin(const char *name) {
    if (!enabled) return;
    hipEvent_t a, b;
    TSG_HIP_TRY(hipEventCreate(&a));
    TSG_HIP_TRY(hipEventCreate(&b));
    TSG_HIP_TRY(hipEventRecord(a, stream));
    names.emplace_back(name);
    ev.push_back(a);
    ev.push_back(b);
}

void StageTimer::end() {
    if (!enabled || ev.empty()) return;
    TSG_HIP_TRY(hipEventRecord(ev.back(), stream));
}

void StageTimer::finalize() {
    if (!enabled) return;
    ms.assign(names.size(), 0.0);
    for (size_t i = 0; i < names.size(); i++) {
        TSG_HIP_TRY(hipEventSynchronize(ev[2 * i + 1]));
        float t = 0.f;
        TSG_HIP_TRY(hipEventElapsedTime(&t, ev[2 * i], ev[2 * i + 1]));
        ms[i] = t;
    }
}

StageTimer::~StageTimer() { clear(); }

// The kernels below run between kernels that stream gigabytes, so their
// operands are cold in every cache: each keeps its chain of dependent loads
// to two or three (no searches, no per-row loops), which is what sets their
// duration.

// ======================================================= row products
// rowprod[i] = sum over A's entries a_ik in row i of |row k of B|
// (main_spgemm-col.cu:4950-4955), as P[ia[i+1]] - P[ia[i]] with P the
// exclusive scan of the per-entry counts |row ja[p] of B|.  A must be a valid
// CSR with columns indexing rows of B.
__global__ void __launch_bounds__(256) k_entry_products(int64_t nnz, const int *__restrict__ ja,
                                                        const int *__restrict__ ib,
                                                        int64_t *__restrict__ ep) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= nnz) return;
    const int k = ja[p];
    ep[p] = ib[k + 1] - ib[k];
}

__global__ void __launch_bounds__(256) k_row_diff(int m, const int *__restrict__ ia,
                                                  const int64_t *__restrict__ P,
                                                  int64_t *__restrict__ rowprod) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < m) rowprod[i] = P[ia[i + 1]] - P[ia[i]];
}

__global__ void k_zero_i64(int64_t n, int64_t *__restrict__ v) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) v[i] = 0;
}

void csr_row_products(int m, const int *ia, const int *ja, int64_t nnz, const int *ib,
                      int64_t *rowprod, Arena &ws, hipStream_t s) {
    if (m <= 0) return;
    if (nnz <= 0) {
        hipLaunchKernelGGL(k_zero_i64, dim3(grid_for((size_t)m, 256)), dim3(256), 0, s,
                           (int64_t)m, rowprod);
        TSG_LAUNCH_CHECK();
        return;
    }
    int64_t *P = ws.alloc_n<int64_t>((size_t)nnz + 1);
    int64_t *tmp = ws.alloc_n<int64_t>(scan_tmp_elems((size_t)nnz + 1));
    hipLaunchKernelGGL(k_entry_products, dim3(grid_for((size_t)nnz, 256)), dim3(256), 0, s, nnz,
                       ja, ib, P);
    TSG_LAUNCH_CHECK();
    exclusive_scan_i64(P, P, (size_t)nnz, tmp, s);
    hipLaunchKernelGGL(k_row_diff, dim3(grid_for((size_t)m, 256)), dim3(256), 0, s, m, ia, P,
                       rowprod);
    TSG_LAUNCH_CHECK();
}

// ============================================================ transpose
// Stable CSR transpose: a radix sort of (column, position) pairs keeps equal
// columns in position order, i.e. ascending source row (utils.h:158-195).
// Row and position of every entry, 8 lanes a row.
__global__ void k_row_pos(int m, const int *__restrict__ ia, int *__restrict__ rowidx,
                          int *__restrict__ pos) {
    const int l = threadIdx.x & 7;
    for (int64_t row = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 3; row < m;
         row += (int64_t)gridDim.x * blockDim.x >> 3) {
        const unsigned pe = (unsigned)ia[row + 1];
        for (unsigned p = (unsigned)ia[row] + l; p < pe; p += 8) {
            rowidx[p] = (int)row;
            pos[p] = (int)p;
        }
    }
}

__global__ void k_iota(int64_t n, int *__restrict__ v) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) v[i] = (int)i;
}

// First position of every column c in [0, n] among the sorted columns.
__global__ void k_col_ptr(int n, int nnz, const int *__restrict__ sorted, int *__restrict__ tp) {
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c <= n) tp[c] = lower_bound_i32(sorted, 0, nnz, (int)c);
}

__global__ void k_gather_t(int64_t nnz, const int *__restrict__ pos, const int *__restrict__ rowidx,
                           const double *__restrict__ a, int *__restrict__ ti,
                           double *__restrict__ tv, int *__restrict__ tpos) {
    int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= nnz) return;
    int p = pos[q];
    ti[q] = rowidx[p];
    if (a) tv[q] = a[p];
    if (tpos) tpos[q] = p;
}

// Stable sort of n (key, value) pairs by the low end_bit bits.  From
// SORT_RADIX pairs on by radix passes: the library's own choice up to 2^20
// pairs, merge passes, takes 158 us for 10^6 keys of 20 bits against 102 (70
// for 9 bits), 112 against 93 for 300,000; below, merging is faster (51 us
// against 89 for 100,000).
constexpr size_t SORT_RADIX = 200 * 1024;
using SortConfig = rocprim::radix_sort_config<rocprim::default_config, rocprim::default_config,
                                              rocprim::default_config, SORT_RADIX>;

static void sort_pairs(const int *keys, int *keys_out, const int *vals, int *vals_out, size_t n,
                       int end_bit, Arena &ws, hipStream_t s) {
    size_t tbytes = 0;
    TSG_HIP_TRY(rocprim::radix_sort_pairs<SortConfig>(nullptr, tbytes, keys, keys_out, vals,
                                                      vals_out, n, 0u, (unsigned)end_bit, s));
    void *tstore = ws.alloc(tbytes);
    TSG_HIP_TRY(rocprim::radix_sort_pairs<SortConfig>(tstore, tbytes, keys, keys_out, vals,
                                                      vals_out, n, 0u, (unsigned)end_bit, s));
}

// The column pointers come from the sorted columns, by a search per column
// (R-MAT 2^18: 8 us; counting with an atomic per entry took 192 us, its hub
// columns' entries queueing on one address).
void csr_transpose(int m, int n, const int *ia, const int *ja, const double *a, int64_t nnz,
                   int *tp, int *ti, double *tv, Arena &ws, hipStream_t s, int *tpos) {
    if (nnz <= 0) {
        TSG_HIP_TRY(hipMemsetAsync(tp, 0, sizeof(int) * ((size_t)n + 1), s));
        return;
    }
    int *rowidx = ws.alloc_n<int>((size_t)nnz);
    int *pos_in = ws.alloc_n<int>((size_t)nnz);
    int *pos_out = ws.alloc_n<int>((size_t)nnz);
    int *keys_out = ws.alloc_n<int>((size_t)nnz);
    hipLaunchKernelGGL(k_row_pos, dim3(grid_for((size_t)m, 32, MAX_GRID)), dim3(256), 0, s, m, ia,
                       rowidx, pos_in);
    TSG_LAUNCH_CHECK();
    int end_bit = 1;
    while (end_bit < 31 && (1ll << end_bit) < (long long)n) end_bit++;
    sort_pairs(ja, keys_out, pos_in, pos_out, (size_t)nnz, end_bit, ws, s);
    hipLaunchKernelGGL(k_col_ptr, dim3(grid_for((size_t)n + 1, 256)), dim3(256), 0, s, n,
                       (int)nnz, keys_out, tp);
    TSG_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_gather_t, dim3(grid_for((size_t)nnz, 256)), dim3(256), 0, s, nnz,
                       pos_out, rowidx, a, ti, tv, tpos);
    TSG_LAUNCH_CHECK();
}

// ====================================================== stable key order
// order[j] = index of the j-th smallest of keys[0..n) (each in [0, 2^end_bit)),
// equal keys in index order.
void sort_order_i32(const int *keys, int64_t n, int end_bit, int *order, Arena &ws,
                    hipStream_t s) {
    if (n <= 0) return;
    TSG_CHECK(n < ((int64_t)1 << 31), TSG_ERR_OVERFLOW, "sort_order_i32: more than 2^31 keys");
    int *iota = ws.alloc_n<int>((size_t)n);
    int *keys_out = ws.alloc_n<int>((size_t)n);
    hipLaunchKernelGGL(k_iota, dim3(grid_for((size_t)n, 256)), dim3(256), 0, s, n, iota);
    TSG_LAUNCH_CHECK();
    sort_pairs(keys, keys_out, iota, order, (size_t)n, end_bit, ws, s);
}

// ================================================== stable row sort of B
// Row-sorted copy of a CSR matrix whose rows may be unsorted or hold
// duplicates: two stable transposes (each a stable radix sort of columns by
// position) give every row ascending columns with equal columns in their
// original order; perm[q] is the original position of sorted entry q.  The
// row pointers are unchanged.
__global__ void k_compose_pos(int64_t n, const int *__restrict__ outer,
                              const int *__restrict__ inner, int *__restrict__ perm) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q < n) perm[q] = inner[outer[q]];
}

__global__ void k_gather_vals(int64_t n, const int *__restrict__ perm,
                              const double *__restrict__ src, double *__restrict__ dst) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q < n) dst[q] = src[perm[q]];
}

void csr_sort_rows(int m, int n, const int *ia, const int *ja, int64_t nnz, int *sorted_ja,
                   int *perm, Arena &tmp, hipStream_t s) {
    if (nnz <= 0) return;
    int *tp = tmp.alloc_n<int>((size_t)n + 1);
    int *ti = tmp.alloc_n<int>((size_t)nnz);
    int *pos1 = tmp.alloc_n<int>((size_t)nnz);
    int *tp2 = tmp.alloc_n<int>((size_t)m + 1);
    int *pos2 = tmp.alloc_n<int>((size_t)nnz);
    csr_transpose(m, n, ia, ja, nullptr, nnz, tp, ti, nullptr, tmp, s, pos1);
    csr_transpose(n, m, tp, ti, nullptr, nnz, tp2, sorted_ja, nullptr, tmp, s, pos2);
    hipLaunchKernelGGL(k_compose_pos, dim3(grid_for((size_t)nnz, 256)), dim3(256), 0, s, nnz,
                       pos2, pos1, perm);
    TSG_LAUNCH_CHECK();
}

void gather_values(int64_t n, const int *perm, const double *src, double *dst, hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_gather_vals, dim3(grid_for((size_t)n, 256)), dim3(256), 0, s, n, perm,
                       src, dst);
    TSG_LAUNCH_CHECK();
}
