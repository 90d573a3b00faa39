// Tile columns of a range of CSR entries (gfx950, wave64): the marking of
// an LDS bitmap shared by the tile counts and AUTO's density sample.
#pragma once

#include <limits.h>

#include "tsg_device.h"

constexpr int TC_U = 4;

// Row pointers are clamped to [0, nnz] and columns to [0, ncols): every
// access stays in bounds (and the tile-column loop bounded) whatever the
// entries hold.  A bit already set is not set again (power-law rows repeat a
// few tile columns, whose words would serialise the LDS atomics); TC_U
// entries per lane and pass have their loads issued together.
template <int NT>
struct TileCols {
    int p1, cmax;
    const int *ja;
    // (positions are unsigned: a pass ends past 2^31 at the end of 2^31 - 1
    // entries)
    __device__ void load(unsigned p, int (&J)[TC_U]) const {
#pragma unroll
        for (int q = 0; q < TC_U; q++) {
            const unsigned pq = p + (unsigned)(q * NT);
            J[q] = pq < (unsigned)p1 ? min(max(ja[pq], 0), cmax) >> 4 : -1;
        }
    }
    // tile-column range of the entries [p0 + t, p1) taken by thread t
    __device__ void range(int p0, int t, int &lo, int &hi) const {
        lo = INT_MAX;
        hi = -1;
        for (unsigned p = (unsigned)p0 + t; p < (unsigned)p1; p += NT * TC_U) {
            int J[TC_U];
            load(p, J);
#pragma unroll
            for (int q = 0; q < TC_U; q++)
                if (J[q] >= 0) {
                    lo = min(lo, J[q]);
                    hi = max(hi, J[q]);
                }
        }
    }
    __device__ void mark(int p0, int t, int w0, int w1, unsigned *bits) const {
        for (unsigned p = (unsigned)p0 + t; p < (unsigned)p1; p += NT * TC_U) {
            int J[TC_U];
            load(p, J);
#pragma unroll
            for (int q = 0; q < TC_U; q++)
                if (J[q] >= w0 && J[q] < w1) {
                    const unsigned bit = 1u << ((J[q] - w0) & 31);
                    unsigned *word = &bits[(J[q] - w0) >> 5];
                    if (!(*word & bit)) atomicOr(word, bit);
                }
        }
    }
};

// AUTO's density sample: a 256-thread block takes tile row I and adds its
// tiles and entries to sums[0] and sums[1].  The block shares a bitmap of
// TS_WORDS * 32 tile columns per pass -- a power-law matrix puts most of its
// entries in its first tile rows, and one wave per row left the sample
// waiting on those.
constexpr int TS_WORDS = 4096;

__device__ __forceinline__ void tile_sample_row(int I, int m, int ncols, int64_t nnz,
                                                const int *__restrict__ ia,
                                                const int *__restrict__ ja,
                                                unsigned long long *__restrict__ sums,
                                                unsigned *bits) {
    __shared__ int s_lo[4], s_hi[4];
    __shared__ int s_cnt[4];
    const int t = threadIdx.x, l = t & 63, w = t >> 6;
    const int p0 = (int)min((int64_t)max(ia[I * 16], 0), nnz);
    const int p1 = (int)min((int64_t)max(ia[tile_rows_end(I, 1, m)], p0), nnz);
    const TileCols<256> tc{p1, max(ncols - 1, 0), ja};
    int lo, hi;
    tc.range(p0, t, lo, hi);
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) {
        lo = min(lo, __shfl_xor(lo, d, 64));
        hi = max(hi, __shfl_xor(hi, d, 64));
    }
    if (l == 0) {
        s_lo[w] = lo;
        s_hi[w] = hi;
    }
    __syncthreads();
    lo = min(min(s_lo[0], s_lo[1]), min(s_lo[2], s_lo[3]));
    hi = max(max(s_hi[0], s_hi[1]), max(s_hi[2], s_hi[3]));
    int count = 0;
    // lo and hi are the block's: every thread takes every pass and barrier
    for (int w0 = lo; w0 <= hi; w0 += TS_WORDS * 32) {
        const int w1 = min(hi + 1, w0 + TS_WORDS * 32);
        const int nwords = (w1 - w0 + 31) >> 5;
        for (int i = t; i < nwords; i += 256) bits[i] = 0u;
        __syncthreads();
        tc.mark(p0, t, w0, w1, bits);
        __syncthreads();
        for (int i = t; i < nwords; i += 256) count += __popc(bits[i]);
        __syncthreads();
    }
    count = wave_sum(count);
    if (l == 0) s_cnt[w] = count;
    __syncthreads();
    if (t == 0) {
        atomicAdd(&sums[0], (unsigned long long)(s_cnt[0] + s_cnt[1] + s_cnt[2] + s_cnt[3]));
        atomicAdd(&sums[1], (unsigned long long)(p1 - p0));
    }
}
