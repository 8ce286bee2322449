// tpamd_gridpair.h -- fixed-step Boris whose every step gathers from two
// grids: E and B gridded on one geometry (a simulation's output), or B a
// sequence of snapshots blended in time, from cell-replicated copies or, in
// solves too small to build them, from the node arrays.
//
// What bounds it: like the single-grid kernels, the rate of random 128-B
// lines (two for a double cell, so four a step; 8 to 16 from nodes), and in
// small solves the latency of a step's loads.  The generic kernel located the
// position for each grid and asked for the second grid's lines only when the
// first one's were back.  Here the position is located once and both gathers
// are asked for together.  The arithmetic is the generic policies', so are the
// results.  Measured, FP64 with cells: E and B on 97 x 80 x 113 nodes, 200,001
// particles x 300 steps: 7.28 -> 2.95 ms (1.55e10 particle-steps/s; 4.7 lines a
// step asked of the L2 and 2.7 missed, 5.2 TB/s); five snapshots of 64 x 61 x
// 96 nodes, 150,001 x 200: 5.68 -> 2.78 ms (3.5 missed, 4.9 TB/s).
#pragma once

#include "tpamd_pusher.h"

namespace {

enum { kPairEB = 0, kPairTime = 1 };

// the pair of arrays a step reads and how they combine: for kPairEB the first
// is E's and the second B's; for kPairTime snapshots k-1 and k, w their
// weight in time (the bracket is searched again only when t leaves it)
template <int MODE, bool CELLS>
struct GridPair {
    const void* c0;
    const void* c1;
    double w, tlo, thi;
    bool blend;
    __device__ __forceinline__ void init(const KParams& p)
    {
        if constexpr (MODE == kPairEB) {
            c0 = CELLS ? p.E.cells : p.E.data;
            c1 = CELLS ? p.B.cells : p.B.data;
        } else {
            tlo = 1.0;
            thi = 0.0;
        }
    }
    __device__ __forceinline__ void at(const KParams& p, double t)
    {
        if constexpr (MODE == kPairTime) {
            if (!(t >= tlo && t < thi)) {
                double unused;
                const int k = time_bracket(p.B, t, unused);
                blend = k > 0 && k < p.B.nsnap;
                const int k0 = k == 0 ? 0 : k - 1, k1 = k >= p.B.nsnap ? p.B.nsnap - 1 : k;
                c0 = CELLS ? snapshot_cells(p.B, k0) : snapshot(p.B, k0);
                c1 = CELLS ? snapshot_cells(p.B, k1) : snapshot(p.B, k1);
                tlo = k > 0 ? p.B.times[k - 1] : -__builtin_inf();
                thi = k < p.B.nsnap ? p.B.times[k] : __builtin_inf();
            }
            w = blend ? (t - tlo) / (thi - tlo) : 0.0;        // time_bracket's
        }
    }
};

template <int MODE, bool UXB, bool PER, typename T, bool CELLS>
struct S64P : S64 {
    static constexpr int kNS = 0;
    GridPair<MODE, CELLS> g;
    __device__ __forceinline__ void load(const KParams& p, long long i)
    {
        S64::load(p, i);
        g.init(p);
    }
    __device__ __forceinline__ void eval(const KParams& p, double t, double E[3], double B[3])
    {
        int i0[3], i1[3];
        double w[3];
        bool in = true;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const double s = (pos.x[d] - p.B.origin[d]) * p.B.inv_h[d];
            i0[d] = i1[d] = 0;
            w[d] = 0.0;
            in = locate_f64<PER>(p.B, d, s, i0[d], i1[d], w[d]) & in;
        }
        g.at(p, t);
        double f0[3], f1[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) f0[c] = f1[c] = __builtin_nan("");
        if (in) {
            if constexpr (CELLS) {
                const unsigned off = cell_offset(p.B, i0);
                T a[24], b[24];
                cell_load<T>(g.c0, off, a);
                cell_load<T>(g.c1, off, b);
                cell_blend<T, double>(a, w, f0);
                cell_blend<T, double>(b, w, f1);
            } else {
                // row by row: both gathers at once would ask for more lines
                // than the first-level cache holds between a line's pieces
                unsigned ox[2], oy[2], oz[2];
                offsets(p.B, i0, i1, sizeof(T), ox, oy, oz);
                trilinear<T, double>(g.c0, ox, oy, oz, w, f0);
                trilinear<T, double>(g.c1, ox, oy, oz, w, f1);
            }
        }
        if constexpr (MODE == kPairEB) {
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                E[c] = f0[c];
                B[c] = f1[c];
            }
        } else {
#pragma unroll
            for (int c = 0; c < 3; ++c) B[c] = g.blend ? (1.0 - g.w) * f0[c] + g.w * f1[c] : f0[c];
        }
        if constexpr (MODE == kPairTime) {
            if constexpr (UXB) cross3(B, p.E.v, E);
            else { E[0] = p.E.v[0]; E[1] = p.E.v[1]; E[2] = p.E.v[2]; }
        }
    }
    template <int ALG>
    __device__ __forceinline__ void U(const KParams& p, const double vin[3], double h, double t, double out[3])
    {
        double E[3], B[3];
        eval(p, t, E, B);
        Uf<ALG>(p, E, B, vin, h, out);
    }
};

template <int MODE, bool UXB, bool PER, bool CELLS>
struct S32P : S32C {
    static constexpr int kNS = 0;
    GridPair<MODE, CELLS> g;
    __device__ __forceinline__ void load(const KParams& p, long long i)
    {
        S32C::load(p, i);
        g.init(p);
    }
    __device__ __forceinline__ void eval(const KParams& p, double t, float E[3], float B[3])
    {
        int i0[3], i1[3];
        float w[3];
        bool in = true;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const float s = fmaf(pos.hi[d], p.B.inv_hf[d], pos.lo[d] * p.B.inv_hf[d]);
            i0[d] = i1[d] = 0;
            w[d] = 0.0f;
            in = locate_f32<PER>(p.B, d, s, i0[d], i1[d], w[d]) & in;
        }
        g.at(p, t);
        float f0[3], f1[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) f0[c] = f1[c] = __builtin_nanf("");
        if (in) {
            if constexpr (CELLS) {
                const unsigned off = cell_offset(p.B, i0);
                float a[24], b[24];
                cell_load<float>(g.c0, off, a);
                cell_load<float>(g.c1, off, b);
                cell_blend<float, float>(a, w, f0);
                cell_blend<float, float>(b, w, f1);
            } else {
                // row by row: both gathers at once would ask for more lines
                // than the first-level cache holds between a line's pieces
                unsigned ox[2], oy[2], oz[2];
                offsets(p.B, i0, i1, sizeof(float), ox, oy, oz);
                trilinear<float, float>(g.c0, ox, oy, oz, w, f0);
                trilinear<float, float>(g.c1, ox, oy, oz, w, f1);
            }
        }
        if constexpr (MODE == kPairEB) {
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                E[c] = f0[c];
                B[c] = f1[c];
            }
        } else {
            const float wf = (float)g.w;
#pragma unroll
            for (int c = 0; c < 3; ++c) B[c] = g.blend ? fmaf(wf, f1[c], (1.0f - wf) * f0[c]) : f0[c];
        }
        if constexpr (MODE == kPairTime) {
            if constexpr (UXB) {
                const float u[3] = {(float)p.E.v[0], (float)p.E.v[1], (float)p.E.v[2]};
                cross3f(B, u, E);
            } else {
#pragma unroll
                for (int c = 0; c < 3; ++c) E[c] = (float)p.E.v[c];
            }
        }
    }
    template <int ALG>
    __device__ __forceinline__ void U(const KParams& p, const float vin[3], double h, double t, float out[3])
    {
        float E[3], B[3];
        eval(p, t, E, B);
        Uf<ALG>(p, E, B, vin, h, out);
    }
};

template <class S>
void launch_pair(const LaunchReq& r)
{
    hipLaunchKernelGGL((k_fixed<S, 0>), r.g, r.b, 0, r.st, *r.p);
}

}  // namespace
