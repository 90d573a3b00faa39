// The first pass over the operands of a product: input checks, AUTO's tile
// density sample, and the row path's products per row and row bins, in one
// launch and one host round trip.
#include "tsg_internal.h"
#include "tsg_device.h"
#include "tsg_sample.h"

#include <algorithm>
#include <cstring>

namespace {

constexpr int FT = 256;                  // threads
constexpr int FRONT_LINE = 32;           // ints between counters (a line each)
constexpr int SAMPLE_SLOTS = 64;         // the sample's sums, spread over lines

// Device counters, zero on entry: one line each, as blocks queue up on an
// address (~8 ns an atomic: 1280 blocks adding two counts to one line had
// been most of the checks' 20 us on a 2D mesh of 65536 rows).
struct FrontCounters {
    unsigned flags[2][FRONT_LINE];       // A, B
    int bins[ROW_BINS][FRONT_LINE];
    unsigned long long sample[SAMPLE_SLOTS][FRONT_LINE / 2];
};

// Products of a row that crosses blocks, by the block it starts in.
struct FrontSlot {
    unsigned long long sum;
    unsigned done;                       // entries added, and 1 for the row's end
    unsigned pad;
};

// One matrix to check (and, prod set, to count products of).
struct FrontMat {
    int rows, cols;
    const int *ptr, *idx;
    int64_t nnz;
    int nblk;                            // blocks of its own
};

struct FrontBins {
    const int *ib;                       // B's row pointers
    int64_t *rowprod, *rownnz;
    int *list[ROW_LISTS];                // bins 1 and 2, 3 and 4, ...: front, back
    int nlist;
    FrontSlot *slots;
    RowBinLimits lim;
};

// Largest r in [0, m] with r + ia[r] <= d, by a wave: 64 probes a step.
// Ends whatever ia holds (the range shrinks by 64 each step).
__device__ __forceinline__ int front_row(const int *__restrict__ ia, int m, int64_t d) {
    int lo = 0, hi = m;
    const int l = __lane_id();
    while (lo < hi) {
        const int step = (int)(((int64_t)hi - lo + 63) >> 6);
        const int64_t r = lo + (int64_t)step * (l + 1);
        const bool ok = r <= hi && r + (int64_t)ia[r <= hi ? r : hi] <= d;
        const unsigned long long b = __ballot(ok);
        const int c = b == ~0ull ? 64 : __builtin_ctzll(~b);
        lo = (int)min((int64_t)hi, lo + (int64_t)step * c);
        hi = (int)min((int64_t)hi, lo + (int64_t)step - 1);
    }
    return lo;
}

// Places a row in its bin's list at pos.
__device__ __forceinline__ void front_place(const FrontBins &P, int bin, int64_t pos, int row) {
    if (bin < 1 || pos < 0 || pos >= P.nlist) return;
    int *list = P.list[(bin - 1) >> 1];
    list[(bin & 1) ? pos : P.nlist - 1 - pos] = row;
}

// A's rows and entries laid out as one list -- a row's entries, then its end
// -- cut into blocks of FT * PER items, so that every block has the same
// work whatever the rows' lengths.  A block checks its share of the row
// pointers (every pointer is some block's) and its entries' columns; an
// entry must be above the one before it unless it starts a row, and the row
// starts among the block's entries are a bit each in LDS.  Then the entries'
// products -- the lengths of the B rows they name -- are summed per row by a
// prefix over the block's entries, and the rows that end here go to their
// bins: positions by a ballot per wave, an LDS atomic per wave and a global
// one per block and bin.  A row that crosses blocks is summed in the slot of
// the block it starts in; whoever adds its last part bins it.
//
// Reads stay inside the arrays whatever they hold: row pointers and columns
// are clamped, and a block takes at most its items.
//
// Bound: a chain of about ten dependent steps per block (17 us on a 2D mesh
// of 65536 rows, 9 us on 1000 rows), then the gathers of B's row lengths
// (20M items of random columns: 43 us of checks, 174 us with products; the
// ER batch's 276M items: 1.2 ms).  In place of checks, sample, product
// counts, their scan, differences and two bin passes -- ten launches, two
// round trips: 2D mesh 70 us of kernels -> 24, 27-point 64^3 145 -> 70 us,
// ER batch 3.4 -> 1.2 ms.
template <int PER>
__global__ void __launch_bounds__(FT) k_front(FrontMat A, FrontMat B, int prod, FrontBins P,
                                              FrontCounters *__restrict__ C, int nsample,
                                              int sample_step) {
    constexpr int W = FT * PER;
    struct Lists {
        unsigned pre[W];                 // products before each entry of a wave's part
        unsigned start[W / 32];          // entries that start a row
        uint16_t slot[W];                // a row's bin and its place among the block's
    };
    __shared__ __align__(16) union {
        Lists L;
        unsigned sample[TS_WORDS];
    } S;
    __shared__ int s_r[2];
    __shared__ unsigned s_woff[5];
    __shared__ unsigned long long s_w64[4];
    __shared__ int s_cnt[ROW_BINS], s_base[ROW_BINS];
    int blk = blockIdx.x;
    if (blk < nsample) {
        tile_sample_row(blk * sample_step, A.rows, A.cols, A.nnz, A.ptr, A.idx,
                        C->sample[blk % SAMPLE_SLOTS], S.sample);
        return;
    }
    blk -= nsample;
    const bool second = blk >= A.nblk;
    if (second) blk -= A.nblk;
    const FrontMat M = second ? B : A;
    const bool count = prod && !second;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int m = M.rows, n = M.cols;
    const int64_t nnz = M.nnz;
    int f = 0;
    // the block's share of the row pointers
    {
        const int64_t per = ((int64_t)m + M.nblk - 1) / M.nblk;
        const int64_t r_end = min((int64_t)m, (blk + 1) * per);
        for (int64_t r = blk * per + t; r < r_end; r += FT) {
            const int64_t lo = M.ptr[r], hi = M.ptr[r + 1];
            if (lo > hi || lo < 0 || hi > nnz) f |= 1;
            if (r == 0 && lo != 0) f |= 1;
            if (r == m - 1 && hi != nnz) f |= 1;
        }
    }
    // its items: rows that end in [r0, r1), entries [e0, e0 + ne)
    const int64_t d0 = (int64_t)blk * W, d1 = min((int64_t)m + nnz, d0 + W);
    if (w < 2) {
        const int r = front_row(M.ptr, m, w ? d1 : d0);
        if (lane == 0) s_r[w] = r;
    }
    for (int i = t; i < W / 32; i += FT) S.L.start[i] = 0u;
    if (t < ROW_BINS) s_cnt[t] = 0;
    __syncthreads();
    const int r0 = s_r[0];
    const int nr = min(max(s_r[1] - r0, 0), W);
    const int64_t e0 = min(max(d0 - r0, (int64_t)0), nnz);
    const int ne = (int)min(max(min(d1 - (r0 + nr), nnz) - e0, (int64_t)0), (int64_t)W);
    for (int i = t; i <= nr; i += FT) {
        const int64_t s = (int64_t)M.ptr[r0 + i] - e0;
        if (s >= 0 && s < ne) atomicOr(&S.L.start[s >> 5], 1u << (s & 31));
    }
    __syncthreads();
    // entries, a wave 64 * PER of them in chunks of 64
    {
        int col[PER], cnt[PER];
#pragma unroll
        for (int j = 0; j < PER; j++) {
            const int i = (w * PER + j) * 64 + lane;
            const bool act = i < ne;
            col[j] = act ? M.idx[e0 + i] : 0;
            const int prev = act && e0 + i > 0 ? M.idx[e0 + i - 1] : -1;
            if (act && (col[j] < 0 || col[j] >= n)) f |= 2;
            if (act && prev >= col[j] && !((S.L.start[i >> 5] >> (i & 31)) & 1u)) f |= 4;
        }
        if (count) {
            unsigned run = 0;
            unsigned long long sum = 0;
#pragma unroll
            for (int j = 0; j < PER; j++) {
                const bool act = (w * PER + j) * 64 + lane < ne && n > 0;
                const int k = min(max(col[j], 0), max(n - 1, 0));
                cnt[j] = act ? max(P.ib[k + 1] - P.ib[k], 0) : 0;
            }
#pragma unroll
            for (int j = 0; j < PER; j++) {
                sum += (unsigned)cnt[j];
                const unsigned incl = (unsigned)wave_incl_scan(cnt[j]);
                S.L.pre[(w * PER + j) * 64 + lane] = run + incl - (unsigned)cnt[j];
                run += (unsigned)__builtin_amdgcn_readlane((int)incl, 63);
            }
            sum = group_sum<64>(sum);
            if (lane == 0) {
                s_woff[w + 1] = run;
                s_w64[w] = sum;
            }
        }
    }
    // one atomic per wave and matrix, for what is wrong only
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) f |= __shfl_xor(f, d, 64);
    if (lane == 0 && f && (C->flags[second][0] & f) != (unsigned)f)
        atomicOr(&C->flags[second][0], (unsigned)f);
    if (!count) return;
    __syncthreads();
    if (t == 0) {
        s_woff[0] = 0;
        for (int i = 1; i < 5; i++) s_woff[i] += s_woff[i - 1];
    }
    const bool wide = s_w64[0] + s_w64[1] + s_w64[2] + s_w64[3] >> 32 != 0;
    __syncthreads();
    // products of the block's entries [x, y)
    auto products = [&](int x, int y) -> int64_t {
        if (wide) {
            // 2^32 products or more in this block: its 32-bit sums wrap
            int64_t s = 0;
            for (int i = x; i < y; i++) {
                const int k = min(max(M.idx[e0 + i], 0), max(n - 1, 0));
                s += max(P.ib[k + 1] - P.ib[k], 0);
            }
            return s;
        }
        auto at = [&](int i) {
            return i < W ? S.L.pre[i] + s_woff[i / (64 * PER)] : s_woff[4];
        };
        return (int64_t)(at(y) - at(x));
    };
    // rows that end here, all but a first one that began in an earlier block
    for (int i0 = 0; i0 < nr; i0 += FT) {
        const int i = i0 + t;
        int bin = -1, pos = 0;
        if (i < nr) {
            const int64_t p0 = M.ptr[r0 + i], p1 = M.ptr[r0 + i + 1];
            const int x = (int)min(max(p0 - e0, (int64_t)0), (int64_t)ne);
            const int y = (int)min(max(p1 - e0, (int64_t)x), (int64_t)ne);
            if (p0 >= e0) {
                const int64_t s = products(x, y);
                P.rowprod[r0 + i] = s;
                bin = row_bin_of(s, (int)(p1 - p0), P.lim);
                if (bin == 0 || bin == ROW_BINS - 1) P.rownnz[r0 + i] = 0;
            }
        }
        const unsigned long long below = (1ull << lane) - 1;
#pragma unroll
        for (int q = 1; q < ROW_BINS; q++) {
            const unsigned long long mask = __ballot(bin == q);
            if (!mask) continue;
            int base = 0;
            if (lane == 0) base = atomicAdd(&s_cnt[q], __popcll(mask));
            base = __builtin_amdgcn_readlane(base, 0);
            if (bin == q) pos = base + __popcll(mask & below);
        }
        if (i < nr) S.L.slot[i] = (uint16_t)(max(bin, 0) | (pos << 3));
    }
    __syncthreads();
    if (t > 0 && t < ROW_BINS && s_cnt[t]) s_base[t] = atomicAdd(&C->bins[t][0], s_cnt[t]);
    __syncthreads();
    for (int i = t; i < nr; i += FT) {
        const int v = S.L.slot[i], bin = v & 7;
        if (bin) front_place(P, bin, (int64_t)s_base[bin] + (v >> 3), r0 + i);
    }
    // the parts of rows that cross blocks: the first row's (thread 0), ended
    // here, and the last one's (thread 1), which goes on
    if (t < 2) {
        const int r = t == 0 ? r0 : r0 + nr;
        if (t == 0 ? nr > 0 : r < m) {
            const int64_t p0 = M.ptr[r], p1 = M.ptr[r + 1];
            const int x = (int)min(max(p0 - e0, (int64_t)0), (int64_t)ne);
            const int y = t == 0 ? (int)min(max(p1 - e0, (int64_t)0), (int64_t)ne) : ne;
            const bool part = t == 0 ? p0 < e0 : x < ne;
            const int64_t home = (p0 + r) / W;
            if (part && home >= 0 && home < M.nblk && x <= y) {
                const unsigned add = (unsigned)(y - x) + (t == 0 ? 1u : 0u);
                FrontSlot *slot = P.slots + home;
                // the sum's old value is waited for, so it is in before the
                // count goes up (a device-wide fence instead wrote back the
                // L2 for every block: 400 us of this kernel on 20M items)
                const unsigned long long was =
                    atomicAdd(&slot->sum, (unsigned long long)products(x, y));
                asm volatile("" ::"v"(was) : "memory");
                const unsigned old = atomicAdd(&slot->done, add);
                if (old + add == (unsigned)(p1 - p0) + 1u) {
                    const int64_t s = (int64_t)atomicAdd(&slot->sum, 0ull);
                    P.rowprod[r] = s;
                    const int bin = row_bin_of(s, (int)(p1 - p0), P.lim);
                    if (bin == 0 || bin == ROW_BINS - 1) P.rownnz[r] = 0;
                    if (bin) front_place(P, bin, atomicAdd(&C->bins[bin][0], 1), r);
                }
            }
        }
    }
}

// The counters into the handle's host memory.
__global__ void __launch_bounds__(64) k_front_publish(const FrontCounters *__restrict__ C,
                                                      HostBox *__restrict__ box) {
    const int t = threadIdx.x;
    static_assert(SAMPLE_SLOTS == 64, "a lane per slot");
    const unsigned long long a = group_sum<64>(C->sample[t][0]);
    const unsigned long long b = group_sum<64>(C->sample[t][1]);
    if (t == 0) {
        box->sample[0] = a;
        box->sample[1] = b;
    }
    if (t < 2) box->flags[t] = C->flags[t][0];
    if (t < ROW_BINS) box->bins[t] = C->bins[t][0];
}

}  // namespace

int front_pass(const CsrIn &A, const CsrIn &B, Arena &ws, hipStream_t s, HostBox *box,
               unsigned long long *density_sample, RowFront *rows, const RowTuning *tune,
               const std::function<void()> &before_sync) {
    const bool two = B.rows > 0 && (B.ptr != A.ptr || B.idx != A.idx || B.cols != A.cols);
    const int64_t items = std::max((int64_t)A.rows + A.nnz, two ? (int64_t)B.rows + B.nnz : 0);
    // small inputs in more, smaller blocks: 1024 of 1024 items at most
    const int per = items <= (1 << 20) ? 4 : 16;
    auto blocks = [&](const CsrIn &X) {
        return X.rows > 0 ? (int)(((int64_t)X.rows + X.nnz + FT * per - 1) / (FT * per)) : 0;
    };
    FrontMat MA{A.rows, A.cols, A.ptr, A.idx, A.nnz, blocks(A)};
    FrontMat MB{B.rows, B.cols, B.ptr, B.idx, B.nnz, two ? blocks(B) : 0};
    FrontBins P{};
    const size_t nslots = rows ? (size_t)MA.nblk + 1 : 0;
    char *zero = static_cast<char *>(ws.alloc(sizeof(FrontCounters) + nslots * sizeof(FrontSlot)));
    FrontCounters *C = reinterpret_cast<FrontCounters *>(zero);
    P.slots = reinterpret_cast<FrontSlot *>(zero + sizeof(FrontCounters));
    if (rows) {
        // a row in a bin has an entry
        rows->nlist = (int)std::min<int64_t>(A.rows, A.nnz);
        rows->rowprod = ws.alloc_n<int64_t>((size_t)A.rows + 1);
        rows->rownnz = ws.alloc_n<int64_t>((size_t)A.rows + 1);
        for (int i = 0; i < ROW_LISTS; i++) {
            rows->list[i] = ws.alloc_n<int>((size_t)rows->nlist + 1);
            P.list[i] = rows->list[i];
        }
        P.ib = B.ptr;
        P.rowprod = rows->rowprod;
        P.rownnz = rows->rownnz;
        P.nlist = rows->nlist;
        P.lim = RowBinLimits{tune->bin1, tune->bin2, tune->bin3,
                             tune->bin3 == ROW_SMALL_PROD ? ROW_MED_PROD : tune->bin3};
    }
    TSG_HIP_TRY(hipMemsetAsync(zero, 0, sizeof(FrontCounters) + nslots * sizeof(FrontSlot), s));
    int nsample = 0, step = 1;
    if (density_sample && A.rows > 0 && A.nnz > 0) {
        const int blkm = tiles_of(A.rows);
        step = tile_sample_step(blkm);
        nsample = (blkm + step - 1) / step;
    }
    const int64_t grid = (int64_t)nsample + MA.nblk + MB.nblk;
    if (grid > 0) {
        if (per == 4)
            hipLaunchKernelGGL(k_front<4>, dim3((unsigned)grid), dim3(FT), 0, s, MA, MB,
                               rows ? 1 : 0, P, C, nsample, step);
        else
            hipLaunchKernelGGL(k_front<16>, dim3((unsigned)grid), dim3(FT), 0, s, MA, MB,
                               rows ? 1 : 0, P, C, nsample, step);
        TSG_LAUNCH_CHECK();
    }
    if (before_sync) before_sync();
    hipLaunchKernelGGL(k_front_publish, dim3(1), dim3(64), 0, s, C, box);
    TSG_LAUNCH_CHECK();
    TSG_HIP_TRY(hipStreamSynchronize(s));
    if (density_sample) {
        density_sample[0] = box->sample[0];
        density_sample[1] = box->sample[1];
    }
    if (rows)
        for (int b = 0; b < ROW_BINS; b++) rows->count[b] = box->bins[b];
    int fa = (int)box->flags[0], fb = (int)box->flags[1];
    if (A.rows == 0 && A.nnz != 0) fa |= 1;
    if (B.rows == 0 && B.nnz != 0) fb |= 1;
    return fa | (fb << 8);
}
