// shared_div_check -- SharedDiv (tpamd_device.h) and sqrt_norm
// (tpamd_dipole.h), which the dipole kernel uses in place of the compiler's
// IEEE double division and square root, against those on random operands
// across the ranges where they are used, the ranges' edges drawn on purpose:
//   * any d in [2^-400, 2^400] and |x| in [2^-512, 2^300];
//   * the kernel's k / r^5, |k| in [2^-300, 2^300], |x|^2 in (2^-160, 2^160);
//   * the kernel's t / (1 + t.t), |t| in [2^-300, 2^60];
//   * sqrt(|x|^2), |x|^2 in (2^-160, 2^160).
// Prints the counts of pairs and roots and of results that differ in any bit;
// exits 1 if any does.
//
// Every thread draws its own operands (xorshift64) and writes its counts and
// first differing operands to its own slots; the loop count is fixed.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <vector>

#include "tpamd_dipole.h"

namespace {

__device__ __forceinline__ unsigned long long next(unsigned long long& s)
{
    s ^= s << 13;
    s ^= s >> 7;
    s ^= s << 17;
    return s;
}

// 2^lo <= |x| <= 2^hi, the exponent uniform; one draw in 32 each an edge, one
// in 16 a mantissa of few bits
__device__ __forceinline__ double draw(unsigned long long& s, int lo, int hi)
{
    const unsigned sel = (unsigned)(next(s) >> 32) & 31u;
    if (sel == 0) return ldexp(1.0, lo);
    if (sel == 1) return ldexp(1.0, hi);
    unsigned long long m = next(s) >> 12;
    if (sel < 4) m &= m << 7;
    if (sel == 4) m |= 0xffffffffff000ull;
    const int e = lo + (int)((next(s) >> 16) % (unsigned long long)(hi - lo));
    return ldexp(1.0 + (double)m * 0x1p-52, e);
}

struct Counts {
    unsigned long long pairs, roots;       // that differ
};

__device__ __forceinline__ bool differs(double a, double b)
{
    return __double_as_longlong(a) != __double_as_longlong(b);
}

__global__ void __launch_bounds__(256) k_check(int iters, Counts* __restrict__ bad, double* __restrict__ first)
{
    const unsigned tid = blockIdx.x * blockDim.x + threadIdx.x;
    unsigned long long s = 0x9E3779B97F4A7C15ull ^ ((unsigned long long)(tid + 1) * 0xBF58476D1CE4E5B9ull);
    for (int k = 0; k < 8; ++k) next(s);
    Counts n{0, 0};
    for (int it = 0; it < iters; ++it) {
        const double r2 = draw(s, -160, 160);
        const double r = sqrt_norm(r2);
        if (differs(r, sqrt(r2))) {
            if (n.pairs + n.roots == 0) {
                first[2 * tid] = r2;
                first[2 * tid + 1] = 0.0;
            }
            ++n.roots;
        }
        double x, d;
        switch (it % 3) {
        case 0:
            x = draw(s, -512, 300);
            d = draw(s, -400, 400);
            break;
        case 1:
            x = draw(s, -300, 300);
            d = (r2 * r2) * r;
            break;
        default: {
            x = draw(s, -300, 60);
            const double a = draw(s, -300, 60), b = draw(s, -300, 60);
            d = 1.0 + ((x * x + a * a) + b * b);
        }
        }
        if (next(s) >> 63) x = -x;
        tpamd::SharedDiv q;
        q.init(d);
        if (differs(q.div(x), x / d)) {
            if (n.pairs + n.roots == 0) {
                first[2 * tid] = x;
                first[2 * tid + 1] = d;
            }
            ++n.pairs;
        }
    }
    bad[tid] = n;
}

}  // namespace

int main(int argc, char** argv)
{
    const int iters = argc > 1 ? atoi(argv[1]) : 1024;
    if (iters < 1 || iters > 65536) {
        fprintf(stderr, "shared_div_check: iterations must be in [1, 65536]\n");
        return 2;
    }
    const int blocks = 2048, threads = 256;
    const size_t n = (size_t)blocks * threads;
    Counts* d_bad = nullptr;
    double* d_first = nullptr;
    if (hipMalloc((void**)&d_bad, n * sizeof(Counts)) != hipSuccess ||
        hipMalloc((void**)&d_first, 2 * n * sizeof(double)) != hipSuccess) {
        fprintf(stderr, "shared_div_check: allocation failed\n");
        return 2;
    }
    hipLaunchKernelGGL(k_check, dim3(blocks), dim3(threads), 0, 0, iters, d_bad, d_first);
    std::vector<Counts> bad(n);
    std::vector<double> first(2 * n);
    if (hipDeviceSynchronize() != hipSuccess ||
        hipMemcpy(bad.data(), d_bad, n * sizeof(Counts), hipMemcpyDeviceToHost) != hipSuccess ||
        hipMemcpy(first.data(), d_first, 2 * n * sizeof(double), hipMemcpyDeviceToHost) != hipSuccess) {
        fprintf(stderr, "shared_div_check: kernel or copy failed\n");
        return 2;
    }
    Counts total{0, 0};
    long at = -1;
    for (size_t i = 0; i < n; ++i) {
        total.pairs += bad[i].pairs;
        total.roots += bad[i].roots;
        if (bad[i].pairs + bad[i].roots && at < 0) at = (long)i;
    }
    printf("{\"pairs\": %.0f, \"differing\": %llu, \"roots\": %.0f, \"roots_differing\": %llu", (double)n * iters,
           total.pairs, (double)n * iters, total.roots);
    if (at >= 0) printf(", \"first\": [\"%a\", \"%a\"]", first[2 * at], first[2 * at + 1]);
    printf("}\n");
    hipFree(d_bad);
    hipFree(d_first);
    return total.pairs + total.roots ? 1 : 0;
}
