// tpamd_quad.h -- fixed-step Boris in fields that are the same everywhere,
// with no boundary, one particle per quad of lanes: lane c of the quad holds
// component c of x and v, and lane 3 the time (it is stepped as a position
// moving at velocity 1 without rotation, which is t + dt exactly).
//
// What bounds it: a solve of few particles is one wave's chain of dependent
// instructions (a wave issues one every ~7 cycles, whatever its parallelism),
// so the instructions a lane issues per step are the time.  Split by
// component, the other components come from the quad's other lanes by DPP
// quad permutations.  Formed in place, the two cross products of a step need
// each vector's two other components: four permutations (8 moves in FP64).
// A lane that holds component a of u can form component a + 2 of u x t from
// one permutation, u_a t_{a+1} - u_{a+1} t_a, and so on: in the rotating
// form below v moves by one component a step and is back after three, and a
// step takes three permutations.  The position stays in its lane: the
// component of v that it needs is among the next step's permutations.  In
// FP64 with E = 0 that is 17 vector instructions instead of 27: 1,024
// particles x 6,400 steps with every tenth state saved take 376 us instead of
// 526 (1.7e10 particle-steps/s).
//
// Every component is formed by the operations of boris_f64 / boris_f32 and
// their cross products in their order, so the results are those of
// run_fixed_impl bit for bit.  Control flow depends on the solve's
// parameters only, so the four lanes of a quad always execute together.
#pragma once

#include "tpamd_pusher.h"

namespace {

namespace quad {

// every lane of a quad_perm reads a lane of its own quad, so no lane keeps
// an old value and none is needed
template <int CTRL>
__device__ __forceinline__ float perm(float x)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), CTRL, 0xF, 0xF, true));
}
template <int CTRL>
__device__ __forceinline__ double perm(double x)
{
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_mov_dpp((int)(unsigned)b, CTRL, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(unsigned)(b >> 32), CTRL, 0xF, 0xF, true);
    return __longlong_as_double(((long long)(unsigned)hi << 32) | (unsigned)lo);
}
// the values of lanes c+1 and c+2 (mod 3) on lanes 0-2, lane 3 its own:
// quad_perm [1,2,0,3] and [2,0,1,3]; last(): lane 3's value on all four
template <class R>
__device__ __forceinline__ R next1(R x) { return perm<0xC9>(x); }
template <class R>
__device__ __forceinline__ R next2(R x) { return perm<0xD2>(x); }
__device__ __forceinline__ double last(double x) { return perm<0xFF>(x); }
template <class R>
__device__ __forceinline__ R pick(const R a[3], int c) { return c == 0 ? a[0] : (c == 1 ? a[1] : a[2]); }

// component of a cross product a x b as cross3 / cross3f form it:
// a1 b2 - a2 b1
__device__ __forceinline__ double crossc(double a1, double b2, double a2, double b1) { return a1 * b2 - a2 * b1; }
__device__ __forceinline__ float crossc(float a1, float b2, float a2, float b1) { return fmaf(a1, b2, -(a2 * b1)); }

// The update with rotation factor h in uniform fields: t, s of the three
// components starting from the lane's own, and the electric half-kicks as
// boris_f64 (v + h E) and boris_f32 (fma(h, E, v)) apply them.  EZ: E is
// zero.  The first kick is then left out and the last one, an addition of
// h E = +-0, kept: the kicks can only turn -0 into +0, the sign of a zero
// reaches nothing but signs of zeros on the way, and the last kick leaves
// the same one.
template <class R, bool EZ>
struct Spin {
    R t[3], s[3], e[3];
    R h;
    __device__ __forceinline__ void init(const R E[3], const R B[3], double hd, int lc)
    {
        R bt[3], bs[3], be[3];
        if constexpr (sizeof(R) == 8) {
            BorisConst64 k;
            k.init(E, B, hd);
#pragma unroll
            for (int j = 0; j < 3; ++j) { bt[j] = k.t[j]; bs[j] = k.s[j]; be[j] = k.hE[j]; }
            h = hd;
        } else {
            BorisConst32 k;
            k.init(E, B, (float)hd);
#pragma unroll
            for (int j = 0; j < 3; ++j) { bt[j] = k.t[j]; bs[j] = k.s[j]; be[j] = EZ ? k.h * E[j] : E[j]; }
            h = k.h;
        }
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const int c = lc + j >= 3 ? lc + j - 3 : lc + j;
            t[j] = lc == 3 ? R(0) : pick(bt, c);
            s[j] = lc == 3 ? R(0) : pick(bs, c);
            e[j] = lc == 3 ? R(0) : pick(be, c);
        }
    }
    __device__ __forceinline__ R kick(R v, int j) const
    {
        if constexpr (sizeof(R) == 8 || EZ) return v + e[j];
        else return fmaf(h, e[j], v);
    }
    // the update in place: component c in, component c out.  With EZ the
    // permutations of v are those of v without the kick, which a second
    // update of the same v shares.
    __device__ __forceinline__ R apply(R v) const
    {
        const R vm = EZ ? v : kick(v, 0);
        const R vp = vm + crossc(next1(vm), t[2], next2(vm), t[1]);
        return kick(vm + crossc(next1(vp), s[2], next2(vp), s[1]), 0);
    }
    // the update in the rotating form: component a = c + PH in, a + 1 out;
    // vc is the lane's own component c of the incoming v (PH 0: v itself)
    template <int PH>
    __device__ __forceinline__ R turn(R v, R& vc) const
    {
        constexpr int A1 = (PH + 1) % 3, A2 = (PH + 2) % 3;
        const R vm = EZ ? v : kick(v, PH);
        const R p1 = next1(vm), p2 = next2(vm);               // components a + 1, a + 2
        if constexpr (PH == 0) vc = v;
        else if constexpr (PH == 1) vc = EZ ? p2 : next2(v);
        else vc = EZ ? p1 : next1(v);
        const R vp = p2 + crossc(vm, t[A1], p1, t[PH]);       // component a + 2
        return kick(p1 + crossc(vp, s[PH], next1(vp), s[A2]), A1);
    }
};

// the position of one component: x + v dt (S64T::step), or the compensated
// pair of S32CT::step_impl without a frame, with the time beside it
struct Move64 {
    double x, dt;
    __device__ __forceinline__ void init(const KParams&, double x0, double t, double d, int lc)
    {
        x = lc == 3 ? t : x0;
        dt = d;
    }
    __device__ __forceinline__ void clock() {}
    __device__ __forceinline__ void go(double v) { x = x + v * dt; }
    __device__ __forceinline__ double now() const { return last(x); }
    __device__ __forceinline__ double pos() const { return x; }
};
struct Move32 {
    float hi, lo, dt_hi, dt_lo;
    double t, dt;
    __device__ __forceinline__ void init(const KParams& p, double x0, double t_, double d, int lc)
    {
        const double r0 = x0 - p.frame_origin[lc == 3 ? 0 : lc];   // S32CT::load_from (no period)
        hi = (float)r0;
        lo = (float)(r0 - (double)hi);
        dt = d;
        dt_hi = (float)dt;                                         // S32CT::set_dt
        dt_lo = (float)(dt - (double)dt_hi);
        t = t_;
    }
    __device__ __forceinline__ void clock() { t += dt; }
    __device__ __forceinline__ void go(float v)
    {
        const float d = fmaf(v, dt_hi, v * dt_lo);
        two_sum(hi, d + lo, hi, lo);
    }
    __device__ __forceinline__ double now() const { return t; }
    __device__ __forceinline__ double pos() const { return 0.0 + ((double)hi + (double)lo); }
};

// the fields of S64T::fields / S32CT::fields for zero / uniform kinds
template <class R>
__device__ __forceinline__ void uniform_fields(const KParams& p, R E[3], R B[3])
{
#pragma unroll
    for (int k = 0; k < 3; ++k) B[k] = p.B.kind == kFieldUniform ? (R)p.B.v[k] : R(0);
    if (p.e_is_uxb) {
        const R u[3] = {(R)p.E.v[0], (R)p.E.v[1], (R)p.E.v[2]};
        if constexpr (sizeof(R) == 8) cross3(B, u, E);        // E = -u x B = B x u
        else cross3f(B, u, E);
    } else {
#pragma unroll
        for (int k = 0; k < 3; ++k) E[k] = p.E.kind == kFieldUniform ? (R)p.E.v[k] : R(0);
    }
}

// A lane's place in its particle's records: component c of x and v on lanes
// 0-2, the time on lane 3, one 8-B slot and its step per record each.
struct Out {
    decltype(gbl((double*)nullptr)) at;
    unsigned step;
    bool vec;
    __device__ __forceinline__ void init(const KParams& p, long long i, int lc)
    {
        vec = lc < 3;
        at = vec ? gbl(p.out_u) + i * p.cap * 6 + lc : gbl(p.out_t) + i * p.cap;
        step = vec ? 6u : 1u;
    }
    __device__ __forceinline__ void put(double x, double v, double t)
    {
        at[0] = vec ? x : t;
        if (vec) at[3] = v;
        at += step;
    }
};

// n steps, none of which saves (boris.jl:454-457): q triples and r single
// ones.  ALIGN: the triples' loop starts on a 64-B line, as a lone wave's time
// depends on where its 7-8 lines of instructions begin (1,000 particles x 3,000
// steps FP64, E zero: 0.119 ms, 0.125-0.128 where it fell by itself; E not zero
// 0.135, 0.139-0.146).  Not between saves, where the padding runs each time (7
// x 500 steps, every fifth saved: 48 us with, 46 without).
template <bool ALIGN, class R, class M, bool EZ>
__device__ __forceinline__ void steps(const Spin<R, EZ>& step, R& v, M& m, int q, int r)
{
    if constexpr (ALIGN) asm volatile(".p2align 6");
    for (; q > 0; --q) {
        R vc;
        m.clock();
        v = step.template turn<0>(v, vc);
        m.clock();
        v = step.template turn<1>(v, vc);
        m.go(vc);
        m.clock();
        v = step.template turn<2>(v, vc);
        m.go(vc);
        m.go(v);
    }
    for (; r > 0; --r) {
        m.clock();
        v = step.apply(v);
        m.go(v);
    }
}

// run_fixed_impl<S64T / S32CT<analytic>, Boris, plain records, HOIST> with
// bnd_flags == 0, for lane lc of particle i's quad
template <class R, class M, bool EZ>
__device__ __forceinline__ void run(const KParams& p, long long i, int lc, const R E[3], const R B[3])
{
    const auto xv = gbl(p.xv0) + 6 * i;
    const int c = lc == 3 ? 0 : lc;
    const double x0 = xv[c];
    R v = lc == 3 ? R(1) : (R)xv[3 + c];
    const double dt = p.dt_pp ? gbl(p.dt_pp)[i] : p.dt;
    const double t0 = p.t0;
    M m;
    m.init(p, x0, fma(-0.5, dt, t0), dt, lc);                 // boris.jl:451
    Out out;
    out.init(p, i, lc);
    long long iout = 0;
    double tlast = 0.0;
    if (p.save_start) {                                       // :507-511
        out.put(sizeof(R) == 8 ? x0 : m.pos(), (double)v, t0);
        tlast = t0;
        iout = 1;
    }
    Spin<R, EZ> step, half;
    half.init(E, B, (p.q2m * 0.5) * (-0.5 * dt), lc);         // :514
    v = half.apply(v);
    step.init(E, B, (p.q2m * 0.5) * dt, lc);
    half.init(E, B, (p.q2m * 0.5) * (0.5 * dt), lc);
    const long long nt = p.nt;
    // the steps before the first that saves, it = K + 1, are K; then K - 1
    // follow each (a loop of 3 2^30 at a time is as good as one)
    constexpr long long kMost = 3LL << 30;
    long long left = nt;                                      // steps still to do
    long long quiet = p.save_every && p.K < nt ? p.K : nt;    // of which none of these saves
    const long long between = p.K - 1 < nt ? p.K - 1 : nt;
    const int bq = (int)(between < kMost ? between / 3 : 0), br = (int)(between < kMost ? between % 3 : 0);
    for (; quiet > kMost; quiet -= kMost, left -= kMost) steps<true, R, M, EZ>(step, v, m, 1 << 30, 0);
    steps<true, R, M, EZ>(step, v, m, (int)(quiet / 3), (int)(quiet % 3));
    left -= quiet;
    while (left > 0) {
        const R vprev = v;                                    // a step that saves (:463-472)
        const double x = m.pos();
        m.clock();
        v = step.apply(v);
        m.go(v);
        iout += 1;
        if (iout <= p.nout) {
            tlast = fma(-0.5, dt, m.now());
            out.put(x, (double)half.apply(vprev), tlast);
        }
        left -= 1;
        if (left >= between && between < kMost) {
            steps<false, R, M, EZ>(step, v, m, bq, br);
            left -= between;
        } else {
            quiet = left < between ? left : between;
            left -= quiet;
            for (; quiet > kMost; quiet -= kMost) steps<false, R, M, EZ>(step, v, m, 1 << 30, 0);
            steps<false, R, M, EZ>(step, v, m, (int)(quiet / 3), (int)(quiet % 3));
        }
    }
    // no particle leaves: every one makes nt steps
    const bool should = p.save_end || (p.save_every && nt > 0 && nt % p.K == 0);
    if (iout < p.nout && should) {                            // :522-543
        const double tf = p.dt_pp ? t0 + (double)nt * dt : p.t1;
        if (iout == 0 || tlast < tf) {
            const double dtf = tf - fma((double)nt - 0.5, dt, t0);
            half.init(E, B, (p.q2m * 0.5) * dtf, lc);
            out.put(m.pos(), (double)half.apply(v), tf);
            iout += 1;
        }
    }
    if (lc == 0) {                                            // :545-551
        gbl(p.out_len)[i] = (int)iout;
        gbl(p.retcode)[i] = (iout < p.nout) ? kRetTerminated : kRetSuccess;
    }
}

}  // namespace quad

// Four threads per particle: threadIdx 4 i + c.  No particle leaves, so one
// thread adds the steps of all: a sum per wave, 31,250 of them for 500,000
// particles, queues at 12 ns each on one address, 0.39 ms however short the
// solve, and waves that wait for it hold back the next ones.  Particles x 300
// steps FP64, with a sum per wave and without: 250,000 0.23 and 0.16 ms, 2 M
// 1.77 and 1.08 ms; FP32C 2 M 1.72 and 1.00 ms.
template <class R, class M>
__global__ void __launch_bounds__(256) k_fixed_quad(const KParams p)
{
    const long long g = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long i = g >> 2;
    R E[3], B[3];
    quad::uniform_fields<R>(p, E, B);
    // E zero with one sign in all components (of which no kick, or every
    // one, turns -0 into +0; the same in every thread)
    bool ez = true;
#pragma unroll
    for (int k = 0; k < 3; ++k) ez = ez && E[k] == R(0) && (copysign(R(1), E[k]) == copysign(R(1), E[0]));
    if (i < p.N) {
        const int lc = (int)(g & 3);
        if (ez) quad::run<R, M, true>(p, i, lc, E, B);
        else quad::run<R, M, false>(p, i, lc, E, B);
    }
    if (g == 0) atomicAdd(p.steps, (unsigned long long)p.N * (unsigned long long)p.nt);
}

}  // namespace
