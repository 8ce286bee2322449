// tpamd_dipole.h -- fixed-step Boris in a dipole B with E zero (trapped
// particles in a planetary field), FP64 and FP32C, one thread per particle.
//
// What bounds it: VALU issue (no memory traffic between records), so the
// instructions of a step are its time.  The step below does the arithmetic
// of the generic kernel (dipole_f64 / dipole_f32, boris_f64 / boris_f32, the
// position step and the boundary test), bit for bit, without what the
// generic forms spend on cases a belt particle never meets:
//   * sqrt and the divisions run the compiler's own IEEE sequences without
//     their scaling steps, which are identities inside the ranges that
//     `step` tests; the three divisions of s = 2t / (1 + t.t) share their
//     denominator's half, and the factor 2 (a power of two) joins the last
//     addition, v + 2 (v' x t / (1 + t.t)), as an exact fma;
//   * E = 0: the first half kick is left out and the last, an addition of
//     h E = +-0, kept: the kicks can only turn -0 into +0, the sign of a zero
//     reaches nothing but signs of zeros on the way, and the last kick leaves
//     the same one;
//   * |x|^2 is formed once per position, for the sphere test and the next
//     step's field, and one pair of compares decides both the sphere test
//     and the arithmetic range;
//   * the time is carried only where records ask for it.
// A lane that fails a range test takes the generic arithmetic for that step.
// Measured: FP64, 262,144 particles x 2,000 steps, 126 -> 100 VALU instructions
// a step, 2754 -> 1640-1700 us (3.1e11 particle-steps/s); FP32C, 1,000,003 x 1,500,
// 122 -> 94, 3347 -> 3172 us (4.7e11; the moves and compares that went issue
// beside float arithmetic, whose 84 operations are what its time is).
#pragma once

#include "tpamd_pusher.h"

namespace {

// the generic arithmetic with the fields fixed when the kernel is compiled
template <class Base>
struct DipoleOnly : Base {
    using R = typename Base::R;
    __device__ __forceinline__ void eval(const KParams& p, double, R E[3], R B[3]) const
    {
        E[0] = E[1] = E[2] = R(0);
        if constexpr (sizeof(R) == 8) dipole_f64(p.B, this->pos.x, B);
        else dipole_f32<Base::kFK>(p, p.B, this->pos, B);
    }
    template <int ALG>
    __device__ __forceinline__ void U(const KParams& p, const R vin[3], double h, double t, R out[3]) const
    {
        R E[3], B[3];
        eval(p, t, E, B);
        this->template Uf<ALG>(p, E, B, vin, h, out);
    }
};

// sqrt as the compiler forms it, without the scaling of tiny arguments
__device__ __forceinline__ double sqrt_norm(double a)
{
    const double y = __builtin_amdgcn_rsq(a);
    double g = a * y;
    double h = y * 0.5;
    const double e = fma(-h, g, 0.5);
    g = fma(g, e, g);
    const double d = fma(-g, g, a);
    h = fma(h, e, h);
    g = fma(d, h, g);
    const double d2 = fma(-g, g, a);
    return fma(d2, h, g);
}

template <class S>
struct DipoleStep;

// FP64.  Ranges of the fast arithmetic: |k| = |b0 R^3| in [2^-300, 2^300]
// and |x|^2 in (2^-160, 2^160), so r^5 in [2^-400, 2^400]: no operand,
// quotient or residual of sqrt and k / r^5 leaves the normal range, and
// v_div_scale would scale neither.  |t| <= 2 |h k| / r^3 < 2^60 by the lower
// bound on |x|^2, and t_c^2 >= 2^-600 is tested per step, so the quotients
// t_c / den, den in [1, 2^122], and their products with velocities that
// start at zero or above 2^-200 stay normal.
// On the equator (z = 0) and on the dipole's axis two components of t are
// zeros, at every step of a particle that moves there, and the arithmetic
// holds as well (a zero's quotient is that zero).  Those lanes fail the range
// test and are let through by their position: the test itself, with the zeros
// in it, would cost every lane three instructions a step.  262,144 protons on
// the equator x 1,000 steps take 1.05 ms (1.00 elsewhere); sent to the generic
// step they took 2.39.
template <>
struct DipoleStep<S64A> {
    static constexpr int kWaves = 6;   // waves per SIMD: 3 % over 4; what spills is the rare path's
    double lo, hi, k, h, kick;
    double r2;           // |x|^2; NaN outside the ranges, which sends the step to the generic arithmetic
    bool tz;             // |t_z| >= |h k| / r^3 is within its range wherever |x|^2 is
    __device__ __forceinline__ void init(const KParams& p, const S64A& s, double dt)
    {
        k = p.B.b0 * ((p.B.radius * p.B.radius) * p.B.radius);
        h = (p.q2m * 0.5) * dt;
        kick = h * 0.0;
        lo = __builtin_inf();
        hi = 0x1p160;
        const double hk = fabs(h * k);
        tz = hk >= 0x1p-56;
        bool fine = fabs(k) >= 0x1p-300 && fabs(k) <= 0x1p300 && hk > 0.0 && hk < 0x1p400;
#pragma unroll
        for (int c = 0; c < 3; ++c) fine = fine && (s.v[c] == 0.0 || fabs(s.v[c]) >= 0x1p-200);
        if (fine) {
            int e;
            (void)frexp(hk, &e);
            const int n = 2 * (e - 59);                        // |x|^3 >= |h k| 2^-59
            const int le = n >= 0 ? (n + 2) / 3 : n / 3;
            lo = ldexp(1.0, le > -160 ? le : -160);
        }
        if ((p.bnd_flags & kBndSphereIn) && p.rin2_hi > lo) lo = p.rin2_hi;
        if ((p.bnd_flags & kBndSphereOut) && p.rout2_lo < hi) hi = p.rout2_lo;
        if (!at(p, s.pos)) r2 = __builtin_nan("");
    }
    // |x|^2 of a position and whether it is inside both ranges
    __device__ __forceinline__ bool at(const KParams&, const S64A::Pos& q)
    {
        r2 = dot3(q.x, q.x);
        return (r2 > lo) & (r2 < hi);
    }
    // a step from the equator or the axis to velocity v, NaN if |x|^2 was out of range
    __device__ __forceinline__ bool flat(const S64A::Pos& q, const double v[3]) const
    {
        return tz & (v[0] == v[0]) & ((q.x[2] == 0.0) | ((q.x[0] == 0.0) & (q.x[1] == 0.0)));
    }
    // the update from s; false where its arithmetic left the ranges above
    __device__ __forceinline__ bool fast(const S64A& s, double out[3]) const
    {
        const double* x = s.pos.x;
        const double* v = s.v;
        const double r = sqrt_norm(r2);
        const double r5 = (r2 * r2) * r;
        SharedDiv q5;
        q5.init(r5);
        const double fac = q5.div(k);
        const double B[3] = {fac * ((-3.0 * x[0]) * x[2]), fac * ((-3.0 * x[1]) * x[2]),
                             fac * (r2 - (3.0 * x[2]) * x[2])};
        double t[3], tt[3], s2[3], vmt[3], vp[3], vps[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) t[c] = h * B[c];
#pragma unroll
        for (int c = 0; c < 3; ++c) tt[c] = t[c] * t[c];
        // the high words of the squares order as the squares do
        const unsigned least = min(min((unsigned)__double2hiint(tt[0]), (unsigned)__double2hiint(tt[1])),
                                   (unsigned)__double2hiint(tt[2]));
        const double den = 1.0 + ((tt[0] + tt[1]) + tt[2]);
        SharedDiv qd;
        qd.init(den);
#pragma unroll
        for (int c = 0; c < 3; ++c) s2[c] = qd.div(t[c]);       // s / 2
        cross3(v, t, vmt);
#pragma unroll
        for (int c = 0; c < 3; ++c) vp[c] = v[c] + vmt[c];
        cross3(vp, s2, vps);
#pragma unroll
        for (int c = 0; c < 3; ++c) out[c] = fma(2.0, vps[c], v[c]) + kick;
        // 2^-600 up to the largest finite number: not inf, not NaN
        return least - (423u << 20) < 0x7ff00000u - (423u << 20);
    }
};

// FP32C.  The position as float, hi + lo, and its |x|^2 serve the sphere
// test's float decision (outside()) and the next step's field.
template <>
struct DipoleStep<S32CA> {
    static constexpr int kWaves = 6;   // waves per SIMD: 3 % over 4; what spills is the rare path's
    float lo, hi, h, kick, rad, b0, xf[3];
    float r2;            // |x|^2; NaN outside (lo, hi)
    __device__ __forceinline__ void init(const KParams& p, const S32CA& s, double dt)
    {
        h = (float)((p.q2m * 0.5) * dt);
        kick = h * 0.0f;
        rad = (float)p.B.radius;
        b0 = (float)p.B.b0;
        lo = 0x1p-126f;                                         // rsq of a normal number
        hi = __builtin_inff();
        if ((p.bnd_flags & kBndSphereIn) && !(p.f32.rin2_skip <= lo)) lo = p.f32.rin2_skip;
        if ((p.bnd_flags & kBndSphereOut) && !(p.f32.rout2_skip >= hi)) hi = p.f32.rout2_skip;
        if (!at(p, s.pos)) r2 = __builtin_nanf("");
    }
    __device__ __forceinline__ bool at(const KParams& p, const Pos32& q)
    {
        pos_f32<kFkAnalytic>(p, q, xf);
        r2 = dot3f(xf, xf);
        return (r2 > lo) & (r2 < hi);
    }
    __device__ __forceinline__ bool flat(const Pos32&, const float*) const { return false; }
    // the update from s; false where 1 + t.t is past 2^60, or r2 is NaN
    __device__ __forceinline__ bool fast(const S32CA& s, float out[3]) const
    {
        const float* v = s.v;
        const float ir = __builtin_amdgcn_rsqf(r2);             // rsqrtf of a normal number
        const float q = rad * ir;
        const float fac = b0 * (q * q * q) * (ir * ir);         // dipole_f32
        const float B[3] = {fac * (-3.0f * xf[0] * xf[2]), fac * (-3.0f * xf[1] * xf[2]),
                            fac * fmaf(-3.0f * xf[2], xf[2], r2)};
        float t[3], s2[3], vmt[3], vp[3], vps[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) t[c] = h * B[c];
        const float den = 1.0f + dot3f(t, t);
        // 2 / den, den in [1, 2^60]: the IEEE division's sequence
        float rc = __builtin_amdgcn_rcpf(den);
        rc = fmaf(fmaf(-den, rc, 1.0f), rc, rc);
        float m = 2.0f * rc;
        m = fmaf(fmaf(-den, m, 2.0f), rc, m);
        const float rr = fmaf(fmaf(-den, m, 2.0f), rc, m);
#pragma unroll
        for (int c = 0; c < 3; ++c) s2[c] = t[c] * rr;
        cross3f(v, t, vmt);
#pragma unroll
        for (int c = 0; c < 3; ++c) vp[c] = v[c] + vmt[c];
        cross3f(vp, s2, vps);
#pragma unroll
        for (int c = 0; c < 3; ++c) out[c] = (v[c] + vps[c]) + kick;
        return den < 0x1p60f;
    }
};

// run_fixed_impl for these fields (plain records, Boris).  The step counter
// and the save schedule are those of the solve, not of a particle, so the
// loops stay uniform over the wave (their counters in scalar registers) and
// run until no lane's particle is left.  A particle that leaves is closed
// inside its last step, from the state before it; its lane then steps on
// without effect, so that every step overwrites the state in place (kept
// back for the lanes that leave, the state cost 40 register moves a step).
template <class S>
struct DipoleRun {
    using R = typename S::R;
    DipoleOnly<S> s;
    DipoleStep<S> f;
    double dt, t, tlast;
    long long i, steps;
    bool here;                   // this lane's particle is still inside

    // the closing record and the particle's outcome (boris.jl:522-551), after
    // final_step steps and n records
    __device__ __forceinline__ void finish(const KParams& p, long long final_step, long long n)
    {
        const bool should = p.save_end || (p.save_every && final_step > 0 && final_step % p.K == 0);
        if (n < p.nout && should) {
            const double t1 = p.dt_pp ? p.t0 + (double)p.nt * dt : p.t1;
            const double tf = (final_step == p.nt) ? t1 : fma((double)final_step, dt, p.t0);
            if (n == 0 || tlast < tf) {
                const double dtf = tf - fma((double)final_step - 0.5, dt, p.t0);
                R vf[3];
                s.template U<0>(p, s.v, dtf, tf, vf);
                record<false>(p, s, i, n, vf, tf);
                n += 1;
            }
        }
        gbl(p.out_len)[i] = (int)n;
        gbl(p.retcode)[i] = (n < p.nout) ? kRetTerminated : kRetSuccess;
        steps = final_step;
        here = false;
    }
    // one step (boris.jl:454-461) to (vn, xn)
    __device__ __forceinline__ void advance(const KParams& p, long long it, long long n, R vn[3],
                                            typename S::Pos& xn)
    {
        const bool good = f.fast(s, vn);
        do_step(p, s, vn, dt, xn);
        bool in = f.at(p, xn);
        // inside the range neither sphere test fires (see outside())
        const bool spheres = !(p.bnd_flags & ~(kBndSphereIn | kBndSphereOut));
        if (here & !(good & in & spheres)) {
            bool done = false;
            if (!good) {
                if (f.flat(s.pos, vn)) {
                    done = in & spheres;
                } else {
                    s.template U<0>(p, s.v, dt, t, vn);
                    do_step(p, s, vn, dt, xn);
                    in = f.at(p, xn);
                }
            }
            if (!in) f.r2 = (R)__builtin_nan("");              // the next step is not `good`
            if (!done && outside(p, s, xn, vn)) finish(p, it - 1, n);
        }
    }
    __device__ __forceinline__ void commit(const R vn[3], const typename S::Pos& xn)
    {
        s.pos = xn;
#pragma unroll
        for (int c = 0; c < 3; ++c) s.v[c] = vn[c];
    }
    template <bool TIMED>
    __device__ __forceinline__ void go(const KParams& p, long long it, long long n)
    {
        R vn[3];
        typename S::Pos xn;
        if constexpr (TIMED) t += dt;
        advance(p, it, n, vn, xn);
        commit(vn, xn);
    }
    // the steps it .. stop, none of which saves, n records so far: two a
    // pass, so that the state's registers change roles instead of being copied
    template <bool TIMED>
    __device__ __forceinline__ void run(const KParams& p, long long& it, long long stop, long long n)
    {
        for (; it < stop; it += 2) {
            go<TIMED>(p, it, n);
            go<TIMED>(p, it + 1, n);
            if (!__any(here)) return;
        }
        if (it == stop) go<TIMED>(p, it++, n);
    }
};

// particle i on this lane; `mine` is false on the lanes past the last one
template <class S>
__device__ __forceinline__ long long run_dipole(const KParams& p, long long i, bool mine)
{
    using R = typename S::R;
    DipoleRun<S> r;
    r.i = mine ? i : 0;
    r.here = mine;
    r.steps = 0;
    r.s.load(p, r.i);
    r.dt = p.dt_pp ? gbl(p.dt_pp)[r.i] : p.dt;
    r.s.set_dt(r.dt);
    long long n = 0;                                          // records of every particle inside
    r.tlast = 0.0;
    if (p.save_start) {                                       // boris.jl:507-511
        if (mine) record<false>(p, r.s, r.i, 0, r.s.v, p.t0);
        r.tlast = p.t0;
        n = 1;
    }
    R vt[3];
    r.s.template U<0>(p, r.s.v, -0.5 * r.dt, p.t0, vt);       // :514
#pragma unroll
    for (int c = 0; c < 3; ++c) r.s.v[c] = vt[c];
    r.f.init(p, r.s, r.dt);
    r.t = fma(-0.5, r.dt, p.t0);                              // :451
    const long long nt = p.nt;
    long long it = 1;
    long long next_save = p.save_every ? p.K + 1 : nt + 2;
    while (it <= nt && __any(r.here)) {
        const long long stop = next_save - 1 < nt ? next_save - 1 : nt;
        if (p.save_every) r.template run<true>(p, it, stop, n);
        else r.template run<false>(p, it, stop, n);
        if (it > nt || !__any(r.here)) break;
        next_save += p.K;                                     // it == next_save
        R vn[3];
        typename S::Pos xn;
        r.t += r.dt;
        r.advance(p, it, n, vn, xn);
        if (r.here && n < p.nout) {                           // :463-472
            const double tc = fma(-0.5, r.dt, r.t);
            r.s.template U<0>(p, r.s.v, 0.5 * r.dt, tc, vt);
            record<false>(p, r.s, r.i, n, vt, tc);
            r.tlast = tc;
        }
        r.commit(vn, xn);
        ++n;
        ++it;
    }
    if (r.here) r.finish(p, nt, n);
    return r.steps;
}

template <class S>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(DipoleStep<S>::kWaves))) k_fixed_dipole(const KParams p)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    add_steps(p, run_dipole<S>(p, i, i < p.N));
}

}  // namespace
