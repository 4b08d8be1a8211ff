// chirp_table.hip -- the transformed kernel of a chirp-z convolution, once per
// plan, in twice the working precision: FP64 for FP32 plans, pairs of doubles
// (unevaluated sums hi + lo, about 106 bits; Dekker 1971, Knuth 4.2.2) for
// FP64 plans, rounded once.
//
// The table multiplies every spectrum of the plan, the same in both
// directions, so its error is not averaged over the data and adds up over a
// round trip.  Transformed in the working precision it was the larger part of
// a chirp-z transform's error (round trips of 1904 in FP32: 3.8e-7, 2.9e-7 with
// the exact table; 3063 in FP64: 7.2e-16, 5.7e-16).
//
// Bound by nothing that matters: M sum(radices) products, one thread per
// output of a stage, so the code is the plain DFT sum of each stage.
#include "kernels.h"

namespace sfft {

namespace {

struct DD {
    double hi, lo;
};

__device__ __forceinline__ DD quick_sum(double a, double b) {  // |a| >= |b|
    const double s = a + b;
    return {s, b - (s - a)};
}
__device__ __forceinline__ DD two_sum(double a, double b) {
    const double s = a + b, t = s - a;
    return {s, (a - (s - t)) + (b - t)};
}
__device__ __forceinline__ DD add(DD a, DD b) {
    DD s = two_sum(a.hi, b.hi);
    const DD t = two_sum(a.lo, b.lo);
    s = quick_sum(s.hi, s.lo + t.hi);
    return quick_sum(s.hi, s.lo + t.lo);
}
__device__ __forceinline__ DD mul(DD a, DD b) {
    const double p = a.hi * b.hi;
    return quick_sum(p, fma(a.hi, b.hi, -p) + (a.hi * b.lo + a.lo * b.hi));
}
__device__ __forceinline__ DD div(DD a, double b) {
    const double q = a.hi / b;
    return quick_sum(q, (fma(-q, b, a.hi) + a.lo) / b);
}
__device__ __forceinline__ DD neg(DD a) { return {-a.hi, -a.lo}; }
__device__ __forceinline__ double add(double a, double b) { return a + b; }
__device__ __forceinline__ double mul(double a, double b) { return a * b; }
__device__ __forceinline__ double neg(double a) { return -a; }

// (v / d) rounded once
__device__ __forceinline__ float scaled(double v, double d) { return (float)(v / d); }
__device__ __forceinline__ double scaled(DD v, double d) {
    const DD q = div(v, d);
    return q.hi + q.lo;
}

template <typename T>
struct Acc;
template <>
struct Acc<float> {
    using A = double;
};
template <>
struct Acc<double> {
    using A = DD;
};

template <typename A>
struct CA {
    A x, y;
};

// e^{-2 pi i m / len}, m < len.
__device__ __forceinline__ void root(uint64_t m, uint64_t len, CA<double> &w) {
    double s, c;
    sincospi(-2.0 * (double)m / (double)len, &s, &c);
    w = {c, s};
}
// The same in pairs: the Taylor series of the first octant, to terms below
// 2^-106.
__device__ __forceinline__ void root(uint64_t m, uint64_t len, CA<DD> &w) {
    const uint64_t oct = 8 * m / len, rem = 8 * m - oct * len;
    const uint64_t f = oct & 1 ? len - rem : rem;  // pi / 4 f / len from an axis
    const DD quarter_pi = {0x1.921fb54442d18p-1, 0x1.1a62633145c07p-55};
    const DD x = mul(div(DD{(double)f, 0.0}, (double)len), quarter_pi);
    const DD x2 = neg(mul(x, x)), one = {1.0, 0.0};
    DD s = one, c = one;
    for (int k = 28; k >= 2; k -= 2) {
        s = add(one, div(mul(s, x2), (double)(k * (k + 1))));
        c = add(one, div(mul(c, x2), (double)(k * (k - 1))));
    }
    s = mul(s, x);
    // octants 1, 2, 5 and 6 swap sine and cosine
    const bool swap = ((oct + 1) & 2) != 0;
    DD re = swap ? s : c, im = swap ? c : s;
    if (oct >= 2 && oct < 6) re = neg(re);
    if (oct < 4) im = neg(im);
    w = {re, im};
}

// roots[m] = e^{-2 pi i m / M}, and the convolution kernel b: the conjugate
// chirp e^{i pi n^2 / N} at n and M - n, 0 between.
template <typename A>
__global__ void k_kernel(CA<A> *b, CA<A> *roots, uint64_t n_len, uint64_t m_len) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t m = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; m < m_len; m += stride) {
        CA<A> v;
        root(m, m_len, v);
        roots[m] = v;
        const uint64_t n = m < n_len ? m : m_len - m;
        if (n < n_len) {
            root(n * n % (2 * n_len), 2 * n_len, v);
            v.y = neg(v.y);
        } else {
            v = {};
        }
        b[m] = v;
    }
}

// One Stockham stage of radix R (span ns) over M values, a thread per output.
template <typename A>
__global__ void k_stage(const CA<A> *x, CA<A> *y, const CA<A> *roots, uint64_t m_len, int radix,
                        uint64_t ns) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    const uint64_t nb = m_len / radix, step = nb / ns;
    for (uint64_t o = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; o < m_len; o += stride) {
        // output t of butterfly j: o = (j / ns) ns R + j mod ns + t ns
        const uint64_t k = o % (ns * radix), j = o / (ns * radix) * ns + k % ns;
        CA<A> s = x[j];
        for (int q = 1; q < radix; ++q) {
            const CA<A> v = x[j + q * nb], w = roots[q * k * step % m_len];
            s.x = add(s.x, add(mul(v.x, w.x), neg(mul(v.y, w.y))));
            s.y = add(s.y, add(mul(v.x, w.y), mul(v.y, w.x)));
        }
        y[o] = s;
    }
}

// bhat[k1 N2 + k2] = x[k1 + N1 k2] / M, N2 = M / N1.
template <typename T, typename A>
__global__ void k_round(const CA<A> *x, C2<T> *bhat, uint64_t m_len, uint64_t n1) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    const uint64_t n2 = m_len / n1;
    for (uint64_t m = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; m < m_len; m += stride) {
        const CA<A> v = x[m / n2 + n1 * (m % n2)];
        bhat[m] = {scaled(v.x, (double)m_len), scaled(v.y, (double)m_len)};
    }
}

}  // namespace

template <typename T>
size_t bs_kernel_work(size_t m_len) {
    return 3 * m_len * sizeof(CA<typename Acc<T>::A>);
}

template <typename T>
hipError_t bs_gen_kernel(C2<T> *bhat, size_t n_len, size_t m_len, size_t n1, void *work,
                         hipStream_t stream) {
    using A = typename Acc<T>::A;
    CA<A> *x = (CA<A> *)work, *y = x + m_len, *roots = y + m_len;
    const dim3 grid((unsigned)((m_len + 255) / 256 < 8192 ? (m_len + 255) / 256 : 8192));
    hipLaunchKernelGGL((k_kernel<A>), grid, dim3(256), 0, stream, x, roots, (uint64_t)n_len,
                       (uint64_t)m_len);
    size_t ns = 1, left = m_len;
    for (int radix : {4, 2, 3, 5, 7, 11, 13}) {
        for (; left % radix == 0; left /= radix) {
            hipLaunchKernelGGL((k_stage<A>), grid, dim3(256), 0, stream, x, y, roots,
                               (uint64_t)m_len, radix, (uint64_t)ns);
            ns *= (size_t)radix;
            CA<A> *t = x;
            x = y;
            y = t;
        }
    }
    if (left != 1) return hipErrorInvalidValue;  // a prime factor above 13
    hipLaunchKernelGGL((k_round<T, A>), grid, dim3(256), 0, stream, x, bhat, (uint64_t)m_len,
                       (uint64_t)n1);
    return hipGetLastError();
}

template size_t bs_kernel_work<float>(size_t);
template size_t bs_kernel_work<double>(size_t);
template hipError_t bs_gen_kernel<float>(C2<float> *, size_t, size_t, size_t, void *, hipStream_t);
template hipError_t bs_gen_kernel<double>(C2<double> *, size_t, size_t, size_t, void *,
                                          hipStream_t);

}  // namespace sfft
