// tpamd_sort.hip -- the bin sums of the adjoint's dL/dB records (with hipCUB's
// block scan) and the radix sort (hipCUB over rocPRIM) for grids with more
// bins than the reverse kernel's counters hold, kept in their own translation
// unit so that the pusher source does not carry rocPRIM's templates.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <hipcub/hipcub.hpp>

#include "tpamd_adjoint.h"

namespace tpamd {

// Sorts (key, record) pairs on key bits [begin_bit, end_bit).  With
// d_temp == nullptr only the temporary storage size is written.
template <typename R>
hipError_t adj_sort_records(void* d_temp, size_t& temp_bytes, const unsigned* keys_in,
                            unsigned* keys_out, const AdjRec<R>* vals_in, AdjRec<R>* vals_out,
                            long long n, int begin_bit, int end_bit, hipStream_t stream)
{
    return hipcub::DeviceRadixSort::SortPairs(d_temp, temp_bytes, keys_in, keys_out, vals_in,
                                              vals_out, (size_t)n, begin_bit, end_bit, stream);
}

namespace {

// Index of the f-th record of a bin's concatenated segments within a chunk
// of blocks starting at block c0: pre[] is the exclusive scan of the
// segment counts and beg[] the segments' block-local starts (nb entries).
template <int P>
__device__ __forceinline__ long long seg_record(const unsigned* pre, const unsigned* beg, int nb, int c0,
                                                unsigned f)
{
    int lo = 0, hi = nb - 1;                  // the last segment starting at or before f
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (pre[mid] <= f) lo = mid;
        else hi = mid - 1;
    }
    return (long long)(c0 + lo) * P + beg[lo] + (f - pre[lo]);
}

// The sums of k_adj_bins, over block-sorted records: bin b's records are the
// segments [blk * P + start, + count) of every block (seg[b][blk]).
// The bin's row of segment counts is scanned in LDS, kChunk blocks at a time,
// and thread f takes the f-th record of the concatenated segments, so
// neighbouring threads read neighbouring records of a segment.
//
// Each batch of RB records is grouped by cell in LDS with a counting sort (one
// ds_add_u32 per record for its rank in the cell, a block scan of the cell
// counts), and one owner thread per cell sums the cell's records into 24
// double registers.  A cell with more than kLim records in the batch is summed
// by the whole workgroup instead, a lane for each of the 24 sums and 16
// records at a time: particles from one point fill a few cells.  Each float
// product is formed in float and converted to double (its scale is a power of
// two); only the order of the double sums differs from one launch to the next.
//
// What bounds it: reading 32 or 52 B a record, the owners' arithmetic (some
// 100 instructions a record, times 2-3 for the fullest cell of a wave) and the
// LDS accesses of the sort are each a quarter to a half of the time, and the
// barriers keep a workgroup's own phases apart.  So a batch is small enough
// for two workgroups a CU (79 KB), which fill each other's gaps, and the next
// batch's records are read while this one is summed.  Against one workgroup of
// 1,024 threads a bin (two owners a cell for float records, LDS atomics for
// double ones), reverse sweep and sums together: 64^3, 131,071 particles x 320
// steps FP32C 2.24 -> 2.15 ms; 30^3, 40,001 x 100 FP64 626 -> 352 us; 64^3,
// 32,768 x 64 from within one cell 65.6 -> 0.27 ms (FP64), 342 -> 0.23 ms
// (FP32C), from 4 cells across 4.5 -> 0.36 and 14.1 -> 0.31 ms.
//
// The first nbins workgroups take a bin each.  A bin of more than `most`
// records is dealt to several: the extra workgroups find theirs from the bins'
// totals, and the parts of a bin add to G by atomics.
template <typename R>
struct BinSum {
    static constexpr int T = AdjBin::kCells;       // an owner per cell
    static constexpr int kChunk = 2048;            // segments scanned at a time
    static constexpr int RB = sizeof(R) == 4 ? 2048 : 1024;
    static constexpr int RPT = RB / T;
    static constexpr unsigned kLim = 32;
    static constexpr bool F32 = sizeof(R) == 4;
};

// a bin's records over all blocks
__global__ void __launch_bounds__(256) k_adj_bin_total(const unsigned* __restrict__ seg, int nblk,
                                                       unsigned* __restrict__ tot)
{
    unsigned n = 0;
    for (int i = threadIdx.x; i < nblk; i += 256) n += AdjPart::seg_count(seg[(size_t)blockIdx.x * nblk + i]);
    using Sum = hipcub::BlockReduce<unsigned, 256>;
    __shared__ typename Sum::TempStorage tmp;
    n = Sum(tmp).Sum(n);
    if (threadIdx.x == 0) tot[blockIdx.x] = n;
}

template <typename R>
__global__ void __launch_bounds__(BinSum<R>::T) __attribute__((amdgpu_waves_per_eu(4))) k_adj_bins_seg(
    const unsigned* __restrict__ keys, const AdjRec<R>* __restrict__ vals, const unsigned* __restrict__ seg,
    const unsigned* __restrict__ tot, int nblk, unsigned nbins, unsigned most, unsigned ncell, double* __restrict__ G)
{
    using C = BinSum<R>;
    constexpr int T = C::T, P = AdjPart::part<R>(), kChunk = C::kChunk, RB = C::RB, RPT = C::RPT;
    constexpr int IPT = kChunk / T, BPT = AdjPart::kMaxBins / T;
    using Scan = hipcub::BlockScan<unsigned, T>;
    __shared__ typename Scan::TempStorage scan_tmp;
    __shared__ unsigned pre[kChunk];
    __shared__ unsigned beg[kChunk];
    __shared__ unsigned cnt[T];
    __shared__ unsigned off[T];
    __shared__ __align__(8) R sb[6 * RB];          // staged records: Bbar 0-2, weights 3-5
    __shared__ int sbe[C::F32 ? RB : 1];           // and their exponents
    __shared__ unsigned full[RB / C::kLim];        // a batch's full cells: cell and count
    __shared__ unsigned nfull;
    __shared__ double part[2][24];                 // a full cell's sums, in turn
    const int tid = threadIdx.x;
    // this workgroup's bin, and which of its parts
    unsigned bin = blockIdx.x, mypart = 0u;
    if (bin >= nbins) {
        unsigned v[BPT], n[BPT], all;
#pragma unroll
        for (int q = 0; q < BPT; ++q) {
            const unsigned k = (unsigned)(tid * BPT + q);
            n[q] = k < nbins && tot[k] ? (tot[k] - 1u) / most : 0u;
            v[q] = n[q];
        }
        Scan(scan_tmp).ExclusiveSum(v, v, all);
        const unsigned x = bin - nbins;
        if (x >= all) return;
#pragma unroll
        for (int q = 0; q < BPT; ++q)
            if (v[q] <= x && x < v[q] + n[q]) {
                off[0] = (unsigned)(tid * BPT + q);
                off[1] = x - v[q] + 1u;
            }
        __syncthreads();
        bin = off[0];
        mypart = off[1];
    }
    const unsigned records = tot[bin], parts = records ? (records - 1u) / most + 1u : 0u;
    if (!parts) return;
    // its records [r0, r1) of the bin's
    const unsigned r0 = (unsigned)((unsigned long long)records * mypart / parts),
                   r1 = (unsigned)((unsigned long long)records * (mypart + 1u) / parts);
    const unsigned first = bin << AdjBin::kShift;
    double acc[24];
#pragma unroll
    for (int j = 0; j < 24; ++j) acc[j] = 0.0;
    cnt[tid] = 0u;
    if (tid < 48) part[tid / 24][tid % 24] = 0.0;
    if (tid == 0) nfull = 0u;
    const size_t row = (size_t)bin * (size_t)nblk;
    unsigned before = 0u;                     // records of the chunks before this one
    for (int c0 = 0; c0 < nblk && before < r1; c0 += kChunk) {
        const int nb = nblk - c0 < kChunk ? nblk - c0 : kChunk;
        unsigned e[IPT], v[IPT];
#pragma unroll
        for (int q = 0; q < IPT; ++q) {
            const int i = tid * IPT + q;
            e[q] = i < nb ? seg[row + c0 + i] : 0u;
            v[q] = AdjPart::seg_count(e[q]);
        }
        unsigned total;
        __syncthreads();                      // the previous chunk is done with pre / beg
        Scan(scan_tmp).ExclusiveSum(v, v, total);
#pragma unroll
        for (int q = 0; q < IPT; ++q) {
            const int i = tid * IPT + q;
            pre[i] = v[q];
            beg[i] = AdjPart::seg_start(e[q]);
        }
        __syncthreads();
        const unsigned f0 = r0 > before ? r0 - before : 0u, f1 = r1 - before < total ? r1 - before : total;
        before += total;
        unsigned loc[RPT];                    // a batch's records on their way, loc = T: none
        AdjRec<R> rv[RPT];
        auto load = [&](unsigned base) {
#pragma unroll
            for (int q = 0; q < RPT; ++q) {
                const unsigned f = base + (unsigned)(tid + q * T);
                loc[q] = T;
                if (f < f1) {
                    const long long r = seg_record<P>(pre, beg, nb, c0, f);
                    loc[q] = keys[r] - first;
                    rv[q] = vals[r];
                }
            }
        };
        load(f0);
        for (unsigned base = f0; base < f1; base += RB) {
            unsigned rank[RPT];
#pragma unroll
            for (int q = 0; q < RPT; ++q) rank[q] = loc[q] < (unsigned)T ? atomicAdd(&cnt[loc[q]], 1u) : 0u;
            __syncthreads();
            const unsigned n = cnt[tid];
            unsigned o;
            Scan(scan_tmp).ExclusiveSum(n, o);
            off[tid] = o;
            if (n > C::kLim) full[atomicAdd(&nfull, 1u)] = (unsigned)tid | (n << 16);
            __syncthreads();                  // off is written and cnt read
            cnt[tid] = 0u;
#pragma unroll
            for (int q = 0; q < RPT; ++q) {
                if (loc[q] < (unsigned)T) {
                    const unsigned d = off[loc[q]] + rank[q];
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        sb[c * RB + d] = rv[q].bb[c];
                        sb[(3 + c) * RB + d] = rv[q].w[c];
                    }
                    if constexpr (C::F32) sbe[d] = rv[q].e;
                }
            }
            __syncthreads();
            load(base + RB);
            const unsigned nf = nfull;
            // the owners sum their cell's records: corner q = (qx, qy, qz) in bits 0..2
            const unsigned end = n > C::kLim ? o : o + n;
            for (unsigned i = o; i < end; ++i) {
                const R b[3] = {sb[i], sb[RB + i], sb[2 * RB + i]};
                const R w0 = sb[3 * RB + i], w1 = sb[4 * RB + i], w2 = sb[5 * RB + i];
                const double sc = C::F32 ? ldexp(1.0, sbe[C::F32 ? i : 0]) : 1.0;
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const R W = ((q & 1) ? w0 : (R)1 - w0) * (((q >> 1) & 1) ? w1 : (R)1 - w1) *
                                ((q >> 2) ? w2 : (R)1 - w2);
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        if constexpr (C::F32) acc[3 * q + c] = fma((double)(W * b[c]), sc, acc[3 * q + c]);
                        else acc[3 * q + c] = fma(W, b[c], acc[3 * q + c]);
                    }
                }
            }
            // the full cells, by all: lane j of 32 the sum j = 3 q + c
            for (unsigned k = 0; k < nf; ++k) {
                const unsigned cell = full[k] & 0xffffu, i0 = off[cell], i1 = i0 + (full[k] >> 16);
                const int j = tid & 31, q = j / 3, c = j % 3;
                if (j < 24) {
                    double sum = 0.0;
                    for (unsigned i = i0 + (unsigned)(tid >> 5); i < i1; i += T / 32) {
                        const R w0 = sb[3 * RB + i], w1 = sb[4 * RB + i], w2 = sb[5 * RB + i];
                        const R W = ((q & 1) ? w0 : (R)1 - w0) * (((q >> 1) & 1) ? w1 : (R)1 - w1) *
                                    ((q >> 2) ? w2 : (R)1 - w2);
                        if constexpr (C::F32) sum = fma((double)(W * sb[c * RB + i]), ldexp(1.0, sbe[i]), sum);
                        else sum = fma(W, sb[c * RB + i], sum);
                    }
                    unsafeAtomicAdd(&part[k & 1][j], sum);
                }
                __syncthreads();
                if (tid == (int)cell) {       // read and cleared before the next but one adds to it
#pragma unroll
                    for (int m = 0; m < 24; ++m) {
                        acc[m] += part[k & 1][m];
                        part[k & 1][m] = 0.0;
                    }
                }
            }
            __syncthreads();                  // sb, full and nfull are read
            if (tid == 0) nfull = 0u;
        }
    }
    // the sums go out in the order of G, half of a cell's at a time: a lane's
    // own 24 are 192 B apart from its neighbour's, a line each
    double* const out = reinterpret_cast<double*>(sb);
    static_assert(sizeof(sb) >= 12 * T * sizeof(double), "half of the sums fit");
    const unsigned mine = ncell - first < (unsigned)T ? ncell - first : (unsigned)T;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 12; ++j) out[tid * 12 + j] = acc[12 * h + j];
        __syncthreads();
        for (unsigned k = tid; k < mine * 12; k += T) {
            if (out[k] == 0.0) continue;
            double* const g = G + (size_t)(first + k / 12) * 24 + 12 * h + k % 12;
            if (parts == 1u) *g += out[k];
            else unsafeAtomicAdd(g, out[k]);
        }
    }
}

}  // namespace

// Launches k_adj_bins_seg.  A bin is split where it holds more than 1.5 times
// what 512 workgroups, two a CU, would have each of all the records, and while
// a part keeps some 4,096 records to set against its 12,288 atomics.
template <typename R>
hipError_t adj_bins_seg(const unsigned* keys, const AdjRec<R>* vals, const unsigned* seg, unsigned* tot, int nblk,
                        unsigned nbins, unsigned ncell, double* G, hipStream_t stream)
{
    const long long records = (long long)nblk * AdjPart::part<R>();       // or fewer
    const long long most = std::max(4096LL, records * 3 / 1024);
    hipLaunchKernelGGL(k_adj_bin_total, dim3(nbins), dim3(256), 0, stream, seg, nblk, tot);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_adj_bins_seg<R>), dim3(nbins + (unsigned)(records / most)), dim3(BinSum<R>::T), 0, stream,
                       keys, vals, seg, tot, nblk, nbins, (unsigned)most, ncell, G);
    return hipGetLastError();
}

template hipError_t adj_bins_seg<float>(const unsigned*, const AdjRec<float>*, const unsigned*, unsigned*, int,
                                        unsigned, unsigned, double*, hipStream_t);
template hipError_t adj_bins_seg<double>(const unsigned*, const AdjRec<double>*, const unsigned*, unsigned*, int,
                                         unsigned, unsigned, double*, hipStream_t);

template hipError_t adj_sort_records<float>(void*, size_t&, const unsigned*, unsigned*,
                                            const AdjRec<float>*, AdjRec<float>*, long long, int,
                                            int, hipStream_t);
template hipError_t adj_sort_records<double>(void*, size_t&, const unsigned*, unsigned*,
                                             const AdjRec<double>*, AdjRec<double>*, long long,
                                             int, int, hipStream_t);

}  // namespace tpamd
