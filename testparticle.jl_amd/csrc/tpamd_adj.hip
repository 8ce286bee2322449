// tpamd_adj.hip -- the checkpointed adjoint of the fixed-step Boris solve
// (kernels and host driver; see tpamd_adjoint.h).
#include "tpamd_pusher.h"
#include "tpamd_adjoint.h"

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <vector>

namespace {

// ---------------------------------------------------------------------------
// Adjoint (see tpamd_adjoint.h).  The forward pass reuses the specialised
// Boris policies, so its trajectory is bit-identical to a solve of the same
// problem; FP64 checkpoints are taken every K steps.
// ---------------------------------------------------------------------------
// FP32C: float storage (the host checks it); FP64: storage T.  CELLS: the
// gathers read the grid's cell-replicated copy (one line per gather).
template <bool F32, bool PER, typename T = double, bool CELLS = false>
using AdjState = typename std::conditional<F32, S32G<kEUniform, 0, PER, CELLS>,
                                           S64G<kEUniform, 0, PER, T, CELLS>>::type;

template <bool F32, bool PER, typename T, bool CELLS>
__device__ __forceinline__ void adj_ckpt_store(const AdjParams& a, long long N, int seg, long long i,
                                               const AdjState<F32, PER, T, CELLS>& s)
{
    double* c = a.ckpt + (size_t)seg * 9 * N + i;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if constexpr (F32) {
            c[(size_t)d * N] = (double)s.pos.hi[d] + (double)s.pos.lo[d];
            c[(size_t)(3 + d) * N] = (double)s.pos.wrap[d];
        } else {
            c[(size_t)d * N] = s.pos.x[d];
            c[(size_t)(3 + d) * N] = 0.0;
        }
        c[(size_t)(6 + d) * N] = (double)s.v[d];
    }
}

template <bool F32, bool PER, typename T, bool CELLS>
__device__ __forceinline__ void adj_ckpt_load(const AdjParams& a, long long N, int seg, long long i,
                                              AdjState<F32, PER, T, CELLS>& s)
{
    const double* c = a.ckpt + (size_t)seg * 9 * N + i;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const double r = c[(size_t)d * N];
        if constexpr (F32) {
            s.pos.hi[d] = (float)r;
            s.pos.lo[d] = (float)(r - (double)s.pos.hi[d]);
            s.pos.wrap[d] = (int)c[(size_t)(3 + d) * N];
        } else {
            s.pos.x[d] = r;
        }
        s.v[d] = (typename AdjState<F32, PER, T, CELLS>::R)c[(size_t)(6 + d) * N];
    }
}

// cell coordinates of the current position, as the forward gather computes them
template <bool F32, bool PER, typename T, bool CELLS>
__device__ __forceinline__ void adj_cellcoord(const KParams& p, const AdjState<F32, PER, T, CELLS>& s,
                                              typename AdjState<F32, PER, T, CELLS>::R sc[3])
{
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if constexpr (F32) sc[d] = fmaf(s.pos.hi[d], p.B.inv_hf[d], s.pos.lo[d] * p.B.inv_hf[d]);
        else sc[d] = (s.pos.x[d] - p.B.origin[d]) * p.B.inv_h[d];
    }
}

// What the reverse step needs of a state, a row of the trajectory: the
// weights in its cell, its velocity and the cell.  The sign of a weight tells
// that a clamped grid is clamped along that axis (weights are never negative).
template <bool F32, bool PER, typename T, bool CELLS>
struct AdjCell {
    using S = AdjState<F32, PER, T, CELLS>;
    using R = typename S::R;
    R w[3], sc[3];
    unsigned key;
    __device__ __forceinline__ void locate(const KParams& p, const AdjParams& a, const S& s)
    {
        int i0[3], i1[3];
        adj_cellcoord<F32, PER, T, CELLS>(p, s, sc);
        key = kNoCell;
        w[0] = w[1] = w[2] = (R)0;
        if (adj_locate<PER, R>(p.B, sc, i0, i1, w))
            key = (unsigned)i0[0] + (unsigned)a.nc[0] * ((unsigned)i0[1] + (unsigned)a.nc[1] * (unsigned)i0[2]);
    }
    __device__ __forceinline__ void store(const KParams& p, const AdjParams& a, long long row, long long i,
                                          const S& s) const
    {
        const long long N = p.N;
        const auto b = gbl((R*)a.rows) + row * kAdjRow * N + i;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            R wd = w[d];
            if constexpr (!PER) {
                if (p.B.extrap == kExtrapClamp && !(sc[d] >= (R)0 && sc[d] <= (R)(p.B.n[d] - 1))) wd = -wd;
            }
            b[d * N] = wd;
            b[(3 + d) * N] = s.v[d];
        }
        gbl(a.row_key)[row * N + i] = key;
    }
};

// One forward step's velocity update U(v, x, h) with its row written on the
// way.  The cell is loaded first and the row stored behind it: the memory
// counter completes in order, so a wait for loads issued after the stores
// would be a wait for the stores too.
template <bool F32, bool PER, typename T, bool CELLS>
__device__ __forceinline__ void adj_step_row(const KParams& p, const AdjParams& a, long long row, long long i,
                                             const AdjState<F32, PER, T, CELLS>& s, double h,
                                             typename AdjState<F32, PER, T, CELLS>::R out[3])
{
    using R = typename AdjState<F32, PER, T, CELLS>::R;
    AdjCell<F32, PER, T, CELLS> q;
    q.locate(p, a, s);
    T raw[24];
    R c[8][3], B[3];
    const R E[3] = {(R)0, (R)0, (R)0};
    if (q.key != kNoCell) adj_corners<T, PER, CELLS>(p.B, a.nc, q.key, raw);
    q.store(p, a, row, i, s);
#pragma unroll
    for (int k = 0; k < 24; ++k) c[k / 3][k % 3] = (R)raw[k];
    if (q.key != kNoCell) adj_value<R>(c, q.w, B);
    else B[0] = B[1] = B[2] = (R)__builtin_nan("");
    s.template Uf<0>(p, E, B, s.v, h, out);
}

// Float adjoint state: (xbar, ubar) = (xb, ub) * 2^ex.  Rescales the
// mantissas so that the largest component lies in [0.5, 1) (exact powers of
// two; a zero or non-finite state is left as it is, and a non-finite one
// reaches the outputs, whose scan reports it).
__device__ __forceinline__ void adj_renorm(float xb[3], float ub[3], int& ex)
{
    const float m = fmaxf(fmaxf(fmaxf(fabsf(xb[0]), fabsf(xb[1])), fmaxf(fabsf(xb[2]), fabsf(ub[0]))),
                          fmaxf(fabsf(ub[1]), fabsf(ub[2])));
    if (m > 0.0f && m <= 3.4028235e38f) {
        int k;
        (void)frexpf(m, &k);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            xb[c] = ldexpf(xb[c], -k);
            ub[c] = ldexpf(ub[c], -k);
        }
        ex += k;
    }
}

// A row on its way to the reverse step: the state and the corner values of
// its cell, loaded together (the row's key, known ahead, addresses the cell)
template <bool F32, typename T>
struct AdjFetch {
    using R = typename std::conditional<F32, float, double>::type;
    R row[kAdjRow];
    T c[24];
};

// one reverse step at the state of a fetched row: (xbar, ubar) <- VJP of the
// step that started there, with rotation factor h and position step dt (0 on
// the row of the initial half-step, which moves no position).  The step's
// dL/dB contribution is returned (Bbar, weights, exponent).
template <bool F32, bool PER, typename T, bool CELLS>
__device__ __forceinline__ AdjRec<typename AdjState<F32, PER, T, CELLS>::R>
adj_step_back(const KParams& p, const AdjFetch<F32, T>& q, double h, double dt, bool with_dt,
              typename AdjState<F32, PER, T, CELLS>::R xb[3], typename AdjState<F32, PER, T, CELLS>::R ub[3], int& ex)
{
    using R = typename AdjState<F32, PER, T, CELLS>::R;
    R w[3], c[8][3], B[3], u[3];
    bool flat[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        flat[d] = false;
        w[d] = q.row[d];
        if constexpr (!PER) {
            flat[d] = copysign((R)1, w[d]) < (R)0;
            w[d] = fabs(w[d]);
        }
        u[d] = q.row[3 + d];
    }
#pragma unroll
    for (int k = 0; k < 24; ++k) c[k / 3][k % 3] = (R)q.c[k];
    adj_value<R>(c, w, B);
    const R hh = (R)h;
    R t[3], g[3], tb[3], un[3], Bb[3], xg[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        t[k] = hh * B[k];
        g[k] = with_dt ? ub[k] + (R)dt * xb[k] : ub[k];
    }
    boris_vjp<R>(u, t, g, un, tb);
#pragma unroll
    for (int k = 0; k < 3; ++k) Bb[k] = hh * tb[k];
    adj_xgrad<R>(p.B, c, w, Bb, xg);
    if constexpr (!PER) {
        // outside the node box a clamped field does not change along that axis
#pragma unroll
        for (int k = 0; k < 3; ++k)
            if (flat[k]) xg[k] = (R)0;
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        xb[k] += xg[k];
        ub[k] = un[k];
    }
    AdjRec<R> v;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        v.bb[k] = Bb[k];
        v.w[k] = w[k];
    }
    if constexpr (F32) {
        v.e = ex;                  // Bbar carries the state's scale at this step
        adj_renorm(xb, ub, ex);
    }
    return v;
}

// The forward pass.  ROWS: the whole trajectory, row 0 the initial state and
// row n + 1 the state before step n; otherwise a checkpoint every K steps.
template <bool F32, bool PER, typename T, bool CELLS, bool ROWS>
__global__ void __launch_bounds__(256) k_adj_forward(const KParams p, const AdjParams a)
{
    using S = AdjState<F32, PER, T, CELLS>;
    using R = typename S::R;
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    double lsum = 0.0;
    if (i < p.N) {
        S s;
        s.load(p, i);
        const double dt = p.dt;
        s.set_dt(dt);
        R vt[3];
        if constexpr (ROWS) adj_step_row<F32, PER, T, CELLS>(p, a, 0, i, s, -0.5 * dt, vt);   // boris.jl:514
        else s.template U<0>(p, s.v, -0.5 * dt, p.t0, vt);
#pragma unroll
        for (int c = 0; c < 3; ++c) s.v[c] = vt[c];
        double t = fma(-0.5, dt, p.t0);
        for (long long n = 0; n < p.nt; ++n) {
            t += dt;
            if constexpr (ROWS) {
                adj_step_row<F32, PER, T, CELLS>(p, a, n + 1, i, s, dt, vt);
            } else {
                if (n % a.K == 0) adj_ckpt_store<F32, PER, T, CELLS>(a, p.N, (int)(n / a.K), i, s);
                s.template U<0>(p, s.v, dt, t, vt);
            }
#pragma unroll
            for (int c = 0; c < 3; ++c) s.v[c] = vt[c];
            typename S::Pos xn;
            do_step(p, s, s.v, dt, xn);
            s.pos = xn;
        }
        double x[3];
        s.abs_pos(p, s.pos, x);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            a.xfinal[3 * i + c] = x[c];
            const double d = x[c] - a.targets[3 * i + c];
            lsum += d * d;
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) lsum += __shfl_xor(lsum, off, 64);
    if ((threadIdx.x & 63) == 0) unsafeAtomicAdd(a.loss, lsum / (double)p.N);
}

// the rows of segment `seg` from its checkpoint (segment 0: the initial state
// first), for solves whose trajectory is not kept whole
template <bool F32, bool PER, typename T, bool CELLS>
__global__ void __launch_bounds__(256) k_adj_rows(const KParams p, const AdjParams a, int seg)
{
    using S = AdjState<F32, PER, T, CELLS>;
    using R = typename S::R;
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= p.N) return;
    const long long n0 = (long long)seg * a.K;
    const int len = (int)((p.nt - n0) < a.K ? (p.nt - n0) : a.K);
    const double dt = p.dt;
    S s;
    long long row = 0;
    if (seg == 0) {
        AdjCell<F32, PER, T, CELLS> q;
        s.load(p, i);
        q.locate(p, a, s);
        q.store(p, a, row++, i, s);
    }
    adj_ckpt_load<F32, PER, T, CELLS>(a, p.N, seg, i, s);
    s.set_dt(dt);
    R vt[3];
    for (int j = 0; j < len; ++j) {
        adj_step_row<F32, PER, T, CELLS>(p, a, row++, i, s, dt, vt);
#pragma unroll
        for (int c = 0; c < 3; ++c) s.v[c] = vt[c];
        typename S::Pos xn;
        do_step(p, s, s.v, dt, xn);
        s.pos = xn;
    }
}

// dynamic LDS of k_adj_reverse<..., SORT = true>: the records, their keys,
// every row's place, the bin counters (one past the last) and the scan's wave sums
template <typename R>
constexpr size_t adj_lds_bytes(unsigned nbins)
{
    const size_t P = AdjPart::part<R>(), T = AdjPart::kThreads;
    return P * sizeof(AdjRec<R>) + P * sizeof(unsigned) + P * sizeof(unsigned short) +
           (((size_t)nbins + T) / T * T + T / 64) * sizeof(unsigned);
}

// Reverse sweep over rows [row0, row0 + nrow) of the row buffer, last row
// first, one thread per particle.  `top`: the adjoint state starts from the
// loss, else from the state the launch above left; `start`: the first row is
// the initial half-step's, and the sweep ends in the gradient.
//
// What bounds it: one thread is a chain of steps, but only the VJP's ~250
// instructions depend on the step before; rows and cells do not.  So D rows
// are in flight per thread, each as one group of loads (the row and, by its
// key, the cell), which hides the gather without occupancy: with SORT the
// records staged in LDS leave one block of 4 waves a CU.  What is left is
// memory: a row, a line of cells and a record, 184 B a step in FP32C, run at
// 5.3 TB/s (131,071 particles x 320 steps, 64^3 float cells: 1.46 ms; with
// the trajectory recomputed and the records sorted by a kernel of their own
// it was 2.9 ms).  512 threads a block, or half the records a block and two
// blocks a CU, measured within 5 %.
//
// SORT: per pass of S rows the block ranks the rows' cells by bin (LDS
// counters and a scan), writes every record to its place in LDS and the pass's
// records out contiguously: block b of the partition is this block's pass.
// Otherwise record `row * N + i` goes to its own slot (a zero one where there
// is none).
template <bool F32, bool PER, typename T, bool CELLS, bool SORT, int D>
__global__ void __launch_bounds__(AdjPart::kThreads) k_adj_reverse(const KParams p, const AdjParams a, long long row0,
                                                                   int nrow, int top, int start)
{
    using R = typename AdjState<F32, PER, T, CELLS>::R;
    constexpr int TH = AdjPart::kThreads, P = AdjPart::part<R>(), S = P / TH, NC = kAdjRow;
    constexpr unsigned kNone = 0xffffu;
    static_assert(S % D == 0, "the ring divides a pass");
    extern __shared__ __align__(16) char lds[];
    AdjRec<R>* sval = (AdjRec<R>*)lds;
    unsigned* skey = (unsigned*)(sval + P);
    unsigned short* slot = (unsigned short*)(skey + P);
    unsigned* cnt = (unsigned*)(slot + P);
    const int tid = threadIdx.x;
    const int nb4 = ((int)a.nbins + TH) / TH * TH;           // counters, padded: a multiple of TH
    unsigned* wsum = cnt + nb4;
    const long long N = p.N;
    const long long i = (long long)blockIdx.x * TH + tid;
    const bool mine = i < N;
    const double dt = p.dt;
    const double h = (p.q2m * 0.5) * dt, h0 = (p.q2m * 0.5) * (-0.5 * dt);
    R* st = (R*)a.state;
    R xb[3], ub[3];
    int ex = 0;                                                // float state: scale 2^ex
    if (!mine) {
#pragma unroll
        for (int c = 0; c < 3; ++c) xb[c] = ub[c] = (R)0;
    } else if (top) {
        double x0[3], m = 0.0;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            x0[c] = 2.0 / (double)N * (a.xfinal[3 * i + c] - a.targets[3 * i + c]);
            m = fmax(m, fabs(x0[c]));
        }
        if constexpr (F32) {
            if (m > 0.0 && m <= 1.0e300) (void)frexp(m, &ex);
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            xb[c] = (R)(F32 ? ldexp(x0[c], -ex) : x0[c]);
            ub[c] = (R)0;
        }
    } else {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            xb[c] = st[(size_t)c * N + i];
            ub[c] = st[(size_t)(3 + c) * N + i];
        }
        if constexpr (F32) ex = a.state_exp[i];
    }
    const int passes = (nrow + S - 1) / S;
    for (int pass = 0; pass < passes; ++pass) {
        const int last = nrow - 1 - pass * S;                 // this pass: rows last, last - 1, ...
        const int m = last + 1 < S ? last + 1 : S;
        const auto keys = gbl((const unsigned*)a.row_key) + (row0 + last) * N + i;
        unsigned total = 0;
        if constexpr (SORT) {
            for (int k = tid; k < nb4; k += TH) cnt[k] = 0u;
            __syncthreads();
            unsigned key[S], rank[S];
#pragma unroll
            for (int s = 0; s < S; ++s) key[s] = mine && s < m ? keys[-(long long)s * N] : kNoCell;
#pragma unroll
            for (int s = 0; s < S; ++s)
                rank[s] = key[s] != kNoCell ? atomicAdd(&cnt[key[s] >> AdjBin::kShift], 1u) : 0u;
            __syncthreads();
            // exclusive scan of the counters, nb4 / TH neighbours a thread
            const int per = nb4 / TH;
            unsigned sum = 0;
            for (int k = 0; k < per; ++k) sum += cnt[tid * per + k];
            unsigned inc = sum;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const unsigned v = __shfl_up(inc, off, 64);
                if ((tid & 63) >= off) inc += v;
            }
            if ((tid & 63) == 63) wsum[tid >> 6] = inc;
            __syncthreads();
            unsigned base = inc - sum;
#pragma unroll
            for (int w = 0; w < TH / 64; ++w) {
                if (w < (tid >> 6)) base += wsum[w];
                total += wsum[w];
            }
            for (int k = 0; k < per; ++k) {
                const unsigned v = cnt[tid * per + k];
                cnt[tid * per + k] = base;
                base += v;
            }
            __syncthreads();
#pragma unroll
            for (int s = 0; s < S; ++s) {
                unsigned d = kNone;
                if (key[s] != kNoCell) {
                    d = cnt[key[s] >> AdjBin::kShift] + rank[s];
                    skey[d] = key[s];
                }
                slot[s * TH + tid] = (unsigned short)d;
            }
            // the table: cnt[nbins] holds the total (the padding's counters are empty)
            const size_t blk = (size_t)blockIdx.x * passes + pass, nblk = (size_t)gridDim.x * passes;
            for (unsigned k = tid; k < a.nbins; k += TH)
                gbl(a.seg)[k * nblk + blk] = AdjPart::seg(cnt[k], cnt[k + 1] - cnt[k]);
            __syncthreads();
        }
        // a row's key again, from its place (SORT) or from the rows
        auto key_of = [&](int s) -> unsigned {
            if (!mine || s >= m) return kNoCell;
            if constexpr (SORT) {
                const unsigned d = slot[s * TH + tid];
                return d == kNone ? kNoCell : skey[d];
            } else {
                return keys[-(long long)s * N];
            }
        };
        auto fetch = [&](int s, AdjFetch<F32, T>& q) -> unsigned {
            const unsigned key = key_of(s);
            if (key != kNoCell) {
                const auto b = gbl((const R*)a.rows) + (row0 + last - s) * NC * N + i;
#pragma unroll
                for (int c = 0; c < NC; ++c) q.row[c] = b[c * N];
                adj_corners<T, PER, CELLS>(p.B, a.nc, key, q.c);
            }
            return key;
        };
        AdjFetch<F32, T> ring[D];
        unsigned rkey[D];
#pragma unroll
        for (int s = 0; s < D; ++s) rkey[s] = fetch(s, ring[s]);
        for (int s0 = 0; s0 < m; s0 += D) {
#pragma unroll
            for (int k = 0; k < D; ++k) {
                const int s = s0 + k;
                const unsigned key = rkey[k];
                const bool half = start && last - s == 0;     // the initial half-step's row
                if (key != kNoCell) {
                    const AdjRec<R> v = adj_step_back<F32, PER, T, CELLS>(p, ring[k], half ? h0 : h, half ? 0.0 : dt,
                                                                          !half, xb, ub, ex);
                    if constexpr (SORT) {
                        sval[slot[s * TH + tid]] = v;
                    } else {
                        gbl(a.rec_key)[(long long)(last - s) * N + i] = key;
                        ((AdjRec<R>*)a.rec_val)[(long long)(last - s) * N + i] = v;
                    }
                } else if (!SORT && mine && s < m) {
                    // a record that adds nothing, keyed to a cell that spreads such
                    // records over the bins
                    const long long r = (long long)(last - s) * N + i;
                    AdjRec<R> v{};
                    gbl(a.rec_key)[r] = (unsigned)(r % (long long)a.ncell);
                    ((AdjRec<R>*)a.rec_val)[r] = v;
                }
                rkey[k] = fetch(s + D, ring[k]);
            }
        }
        if constexpr (SORT) {
            __syncthreads();
            const size_t out = ((size_t)blockIdx.x * passes + pass) * P;
            typedef unsigned U4 __attribute__((ext_vector_type(4)));
            // P records are a multiple of 16 B, so a last partial vector stays inside
            const unsigned nv = (total * (unsigned)sizeof(AdjRec<R>) + 15u) / 16u, nk = (total + 3u) / 4u;
            const auto ov = gbl((U4*)((AdjRec<R>*)a.rec_val + out));
            const auto ok = gbl((U4*)(a.rec_key + out));
            for (unsigned k = tid; k < nv; k += TH) ov[k] = ((const U4*)sval)[k];
            for (unsigned k = tid; k < nk; k += TH) ok[k] = ((const U4*)skey)[k];
            __syncthreads();                                  // before the next pass writes LDS
        }
    }
    if (!mine) return;
    if (start) {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            a.grad_xv0[6 * i + c] = ldexp((double)xb[c], ex);
            a.grad_xv0[6 * i + 3 + c] = ldexp((double)ub[c], ex);
        }
    } else {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            st[(size_t)c * N + i] = xb[c];
            st[(size_t)(3 + c) * N + i] = ub[c];
        }
        if constexpr (F32) a.state_exp[i] = ex;
    }
}

__global__ void k_zero_f64(double* p, long long n)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0;
}

// counts the entries of a[0..n) that are not finite into *count
__global__ void __launch_bounds__(256) k_count_nonfinite(const double* __restrict__ a, long long n,
                                                         unsigned long long* count)
{
    unsigned long long c = 0;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        c += isfinite(a[i]) ? 0ull : 1ull;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off, 64);
    if ((threadIdx.x & 63) == 0 && c) atomicAdd(count, c);
}

template <bool F32, bool PER, typename T, bool CELLS>
int adjoint_run(tpamd_ctx* ctx, KParams p, const tpamd_field* B, const double* xv0, int64_t N,
                const double* targets, int K, int64_t nt, double* loss, double* dL_dB,
                double* dL_dxv0, tpamd_stats* stats, bool bycomp, bool ckpt)
{
    using R = typename AdjState<F32, PER, T, CELLS>::R;
    constexpr int TH = AdjPart::kThreads, P = AdjPart::part<R>(), S = P / TH, NC = kAdjRow;
    constexpr int D = F32 ? 4 : 2;
    const int nseg = (int)((nt + K - 1) / K);
    const size_t rs = sizeof(R);
    const int nx = B->d.n[0], ny = B->d.n[1], nz = B->d.n[2];
    const size_t nnodes = (size_t)nx * ny * nz;
    int nc[3];
    for (int k = 0; k < 3; ++k) nc[k] = PER ? B->d.n[k] : B->d.n[k] - 1;
    const unsigned ncell = (unsigned)nc[0] * (unsigned)nc[1] * (unsigned)nc[2];   // < 2^30
    const unsigned nbins = (ncell + AdjBin::kCells - 1) / AdjBin::kCells;
    // the reverse kernel groups the records while its bin counters fit in LDS
    const bool sort = nbins <= AdjPart::kMaxBins;
    const int64_t nrows = nt + 1;
    const long long nblocks = (N + TH - 1) / TH;
    HIP_TRY(ctx, hipSetDevice(ctx->device));
    // bytes of r rows, and of the records of a launch over r rows
    auto al = [](size_t x) { return (x + 255) & ~(size_t)255; };
    auto row_bytes = [&](int64_t r) { return al(rs * NC * (size_t)r * N) + al(sizeof(unsigned) * (size_t)r * N); };
    const size_t b_xv = al(sizeof(double) * 6 * N), b_tg = al(sizeof(double) * 3 * N), b_st = al(rs * 6 * (size_t)N),
                 b_se = al(sizeof(int) * (size_t)N), b_G = al(sizeof(double) * 24 * (size_t)ncell),
                 b_out = al(sizeof(double) * 3 * nnodes), b_gx = al(sizeof(double) * 6 * N), b_ls = al(sizeof(double)),
                 b_xf = al(sizeof(double) * 3 * N), b_nf = al(sizeof(unsigned long long));
    const size_t fixed = b_xv + b_tg + b_st + b_se + b_G + b_out + b_gx + b_ls + b_xf + b_nf;
    // The whole trajectory where the workspace takes at most 1/16 of the free
    // memory (or 4 GiB, or no more than with checkpoints), which the context
    // keeps for the next call; then a launch walks as many rows as make about
    // 2^24 records (some 0.5 GB in float), a multiple of a pass.  Otherwise
    // segments of K steps.  The trajectory saves the segments' second gathers:
    // FP32C 262,144 x 2,048 steps (15 GB) 40 ms against 48, FP64 131,072 x 1,000
    // (7 GB) 17 and 22.  But memory that each call allocates and frees is wiped in
    // between, at some 30 ms a GB once the device has been through its free
    // memory: not kept, the same FP64 call took 218 ms, 1 M x 2,048 FP32C (60 GB)
    // 1,620 against 200.
    size_t mem_free = 0, mem_total = 0;
    HIP_TRY(ctx, hipMemGetInfo(&mem_free, &mem_total));
    mem_free += ctx->d_buf_bytes;                            // ours to use again
    auto rec_slots = [&](int64_t r) {
        return sort ? (size_t)nblocks * (size_t)((r + S - 1) / S) * P : (size_t)r * (size_t)N;
    };
    auto rec_bytes = [&](int64_t r) {
        return (sort ? 1 : 2) * (al(sizeof(unsigned) * rec_slots(r)) + al(sizeof(AdjRec<R>) * rec_slots(r))) +
               al(sort ? sizeof(unsigned) * (size_t)nbins * ((size_t)nblocks * (size_t)((r + S - 1) / S) + 1) : 1);
    };
    const int64_t fit = (1LL << 24) / std::max<long long>(nblocks * TH, 1);
    int64_t rows_launch = std::min<int64_t>(nrows, std::max<int64_t>(sort ? S : 1, fit / S * S));
    const int64_t rows_seg = std::min<int64_t>((int64_t)K + 1, nrows);
    const size_t need_whole = fixed + row_bytes(nrows) + rec_bytes(rows_launch),
                 need_ckpt = fixed + al(sizeof(double) * 9 * (size_t)nseg * N) + row_bytes(rows_seg) + rec_bytes(rows_seg);
    const bool whole = !ckpt && (need_whole <= std::min(std::max((size_t)4 << 30, mem_free / 16), mem_free / 2) || need_whole <= need_ckpt);
    if (!whole) rows_launch = rows_seg;
    const size_t slots = rec_slots(rows_launch);
    int cellbits = 0;
    while ((1u << cellbits) < ncell) ++cellbits;
    size_t temp_bytes = 0;
    if (!sort)
        HIP_TRY(ctx, adj_sort_records<R>(nullptr, temp_bytes, nullptr, nullptr, nullptr, nullptr, (long long)slots,
                                         AdjBin::kShift, cellbits, ctx->stream));
    const size_t b_ck = whole ? 0 : al(sizeof(double) * 9 * (size_t)nseg * N),
                 b_rw = al(rs * NC * (size_t)(whole ? nrows : rows_launch) * N),
                 b_rk = al(sizeof(unsigned) * (size_t)(whole ? nrows : rows_launch) * N),
                 b_key = al(sizeof(unsigned) * slots), b_val = al(sizeof(AdjRec<R>) * slots),
                 seg_words = (size_t)nbins * (slots / P),         // and the bins' totals behind them
                 b_seg = al(sort ? sizeof(unsigned) * (seg_words + nbins) : 1), b_tmp = al(std::max<size_t>(temp_bytes, 1));
    const size_t total = fixed + b_ck + b_rw + b_rk + (sort ? 1 : 2) * (b_key + b_val) + b_seg + b_tmp;
    // the context's buffer, kept from call to call up to ctx->keep_bytes: an
    // allocation of this size is tens of microseconds, its release some
    // hundreds, and now and then either stalls for tens of milliseconds
    char* buf = nullptr;
    HIP_TRY(ctx, ctx_buffer(ctx, total, (void**)&buf));
    char* q = buf;
    auto take = [&](size_t n) { char* r = q; q += n; return (void*)r; };
    double* d_xv = (double*)take(b_xv);
    double* d_tg = (double*)take(b_tg);
    AdjParams a;
    a.state = take(b_st);
    a.state_exp = (int*)take(b_se);
    double* G = (double*)take(b_G);
    double* d_out = (double*)take(b_out);
    a.grad_xv0 = (double*)take(b_gx);
    a.loss = (double*)take(b_ls);
    unsigned long long* d_nf = (unsigned long long*)take(b_nf);   // d_out .. d_nf: read back in one span
    a.xfinal = (double*)take(b_xf);
    a.ckpt = whole ? nullptr : (double*)take(b_ck);
    a.rows = take(b_rw);
    a.row_key = (unsigned*)take(b_rk);
    a.rec_key = (unsigned*)take(b_key);
    a.rec_val = take(b_val);
    unsigned* keys1 = sort ? nullptr : (unsigned*)take(b_key);
    AdjRec<R>* vals1 = sort ? nullptr : (AdjRec<R>*)take(b_val);
    a.seg = (unsigned*)take(b_seg);
    void* d_tmp = take(b_tmp);
    a.targets = d_tg;
    a.K = K;
    a.nseg = nseg;
    a.ncell = ncell;
    a.nbins = nbins;
    for (int k = 0; k < 3; ++k) a.nc[k] = nc[k];
    p.xv0 = d_xv;
    hipStream_t st = ctx->stream;
    const dim3 block(256), grid((unsigned)((N + 255) / 256)), rgrid((unsigned)nblocks);
    const long long ng = 24 * (long long)ncell;
    const size_t lds = sort ? adj_lds_bytes<R>(nbins) : 0;
    float ms_f = 0.f, ms_r = 0.f;
    const HostPart in[2] = {{const_cast<double*>(xv0), 0, sizeof(double) * 6 * N},
                            {const_cast<double*>(targets), b_xv, sizeof(double) * 3 * N}};
    hipError_t e = stage_in(ctx, buf, b_xv + sizeof(double) * 3 * N, in, 2, st);
    if (e == hipSuccess && sort)
        e = hipFuncSetAttribute((const void*)k_adj_reverse<F32, PER, T, CELLS, true, D>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_zero_f64, dim3((unsigned)((ng + 255) / 256)), dim3(256), 0, st, G, ng);
        hipLaunchKernelGGL(k_zero_f64, dim3(1), dim3(64), 0, st, a.loss, 1LL);
        hipLaunchKernelGGL(k_zero_f64, dim3(1), dim3(64), 0, st, (double*)d_nf, 1LL);
        e = hipEventRecord(ctx->ev0, st);
    }
    if (e == hipSuccess) {
        if (whole) hipLaunchKernelGGL((k_adj_forward<F32, PER, T, CELLS, true>), grid, block, 0, st, p, a);
        else hipLaunchKernelGGL((k_adj_forward<F32, PER, T, CELLS, false>), grid, block, 0, st, p, a);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipEventRecord(ctx->ev1, st);
    // one launch over rows [row0, row0 + n): the reverse steps, then the bin sums
    auto sweep = [&](int64_t row0, int n, int top, int start) {
        if (sort) hipLaunchKernelGGL((k_adj_reverse<F32, PER, T, CELLS, true, D>), rgrid, dim3(TH), lds, st, p, a, (long long)row0, n, top, start);
        else hipLaunchKernelGGL((k_adj_reverse<F32, PER, T, CELLS, false, D>), rgrid, dim3(TH), 0, st, p, a, (long long)row0, n, top, start);
        hipError_t r = hipGetLastError();
        if (r != hipSuccess) return r;
        if (sort)
            return adj_bins_seg<R>(a.rec_key, (const AdjRec<R>*)a.rec_val, a.seg, a.seg + seg_words, (int)(nblocks * ((n + S - 1) / S)), nbins, ncell, G, st);
        const long long M = (long long)n * N;
        r = adj_sort_records<R>(d_tmp, temp_bytes, a.rec_key, keys1, (const AdjRec<R>*)a.rec_val, vals1, M, AdjBin::kShift, cellbits, st);
        if (r != hipSuccess) return r;
        hipLaunchKernelGGL((k_adj_bins<R>), dim3(nbins), dim3(AdjBin::kThreads), 0, st, keys1, vals1, M, ncell, G);
        return hipGetLastError();
    };
    if (whole) {
        for (int64_t end = nrows; end > 0 && e == hipSuccess;) {
            const int64_t row0 = std::max<int64_t>(0, end - rows_launch);
            e = sweep(row0, (int)(end - row0), end == nrows, row0 == 0);
            end = row0;
        }
    } else {
        for (int seg = nseg - 1; seg >= 0 && e == hipSuccess; --seg) {
            const int64_t len = std::min<int64_t>(K, nt - (int64_t)seg * K);
            hipLaunchKernelGGL((k_adj_rows<F32, PER, T, CELLS>), grid, block, 0, st, p, a, seg);
            e = hipGetLastError();
            if (e == hipSuccess) e = sweep(0, (int)(len + (seg == 0)), seg == nseg - 1, seg == 0);
        }
    }
    if (e == hipSuccess) {
        const dim3 ngrid((unsigned)((nx + 7) / 8), (unsigned)((ny + 7) / 8), (unsigned)((nz + 7) / 8));
        if (bycomp)
            hipLaunchKernelGGL(k_adj_nodes<true>, ngrid, dim3(512), 0, st, G, nx, ny, nz, nc[0], nc[1], nc[2], PER ? 1 : 0, d_out);
        else
            hipLaunchKernelGGL(k_adj_nodes<false>, ngrid, dim3(512), 0, st, G, nx, ny, nz, nc[0], nc[1], nc[2], PER ? 1 : 0, d_out);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipEventRecord(ctx->ev2, st);
    // the outputs are scanned for entries that are not finite (the loss, the
    // node gradient, the initial-state gradient)
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_count_nonfinite, dim3(1), dim3(64), 0, st, a.loss, 1LL, d_nf);
        hipLaunchKernelGGL(k_count_nonfinite, dim3((unsigned)std::min<size_t>((3 * nnodes + 255) / 256, 4096)),
                           dim3(256), 0, st, d_out, (long long)(3 * nnodes), d_nf);
        hipLaunchKernelGGL(k_count_nonfinite, dim3((unsigned)std::min<long long>((6 * N + 255) / 256, 4096)),
                           dim3(256), 0, st, a.grad_xv0, (long long)(6 * N), d_nf);
        e = hipGetLastError();
    }
    unsigned long long nonfinite = 0;
    const HostPart out[4] = {{dL_dB, 0, sizeof(double) * 3 * nnodes},
                             {dL_dxv0, b_out, sizeof(double) * 6 * N},
                             {loss, b_out + b_gx, sizeof(double)},
                             {&nonfinite, b_out + b_gx + b_ls, sizeof nonfinite}};
    if (e == hipSuccess) e = stage_out(ctx, (char*)d_out, b_out + b_gx + b_ls + sizeof nonfinite, out, 4, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    else (void)hipStreamSynchronize(st);
    if (e == hipSuccess) e = hipEventElapsedTime(&ms_f, ctx->ev0, ctx->ev1);
    if (e == hipSuccess) e = hipEventElapsedTime(&ms_r, ctx->ev1, ctx->ev2);
    ctx_trim(ctx);
    if (e != hipSuccess) return fail(ctx, TPAMD_ERR_DEVICE, "adjoint failed: %s", hipGetErrorString(e));
    if (stats) {
        stats->kernel_ms = ms_f;
        stats->aux_ms = ms_r;
        stats->particle_steps = nt * N;
        stats->nt = nt;
        stats->nout = 1;
        stats->max_len = 1;
        stats->total_ms = ms_f + ms_r;
    }
    if (nonfinite)
        return fail(ctx, TPAMD_ERR_NONFINITE,
                    "%llu entries of the loss and its gradients are not finite (the forward "
                    "trajectory left the field, or a gradient exceeds the double range)",
                    nonfinite);
    return TPAMD_OK;
}

}  // namespace

namespace tpamd {

int adjoint_launch(tpamd_ctx* ctx, const KParams& p, const tpamd_field* B, const double* xv0,
                   int64_t N, const double* targets, int K, int64_t nt, double* loss,
                   double* dL_dB, double* dL_dxv0, tpamd_stats* stats, bool f32, bool bf32,
                   bool per, bool cells, bool bycomp, bool ckpt)
{
#define TPAMD_ADJ(F32_, PER_, T_, CELLS_) \
    return adjoint_run<F32_, PER_, T_, CELLS_>(ctx, p, B, xv0, N, targets, K, nt, loss, dL_dB, dL_dxv0, stats, bycomp, ckpt)
    if (f32) {
        if (cells) {
            if (per) TPAMD_ADJ(true, true, float, true);
            TPAMD_ADJ(true, false, float, true);
        }
        if (per) TPAMD_ADJ(true, true, float, false);
        TPAMD_ADJ(true, false, float, false);
    }
    if (bf32) {
        if (per) TPAMD_ADJ(false, true, float, false);
        TPAMD_ADJ(false, false, float, false);
    }
    if (cells) {
        if (per) TPAMD_ADJ(false, true, double, true);
        TPAMD_ADJ(false, false, double, true);
    }
    if (per) TPAMD_ADJ(false, true, double, false);
    TPAMD_ADJ(false, false, double, false);
#undef TPAMD_ADJ
}

}  // namespace tpamd
