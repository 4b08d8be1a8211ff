// chirp.h -- chirp-z transforms of short lengths in one launch.
//
// A length N with a prime factor above 13 is a cyclic convolution of length
// M >= 2N - 1 (bluestein.hip has the identity and the tables).  Where M
// complex values fit one workgroup's LDS the whole convolution runs in one
// kernel:
//   load x, times the chirp, zeros up to M  -> registers
//   forward FFT of length M                 -> registers (exchanges in LDS)
//   times the transformed kernel
//   inverse FFT of length M                 -> registers
//   times the chirp, first N values         -> HBM
// so that HBM sees each input and output once.  The separate launches (pre,
// two FFTs, product, post) move about 30 N values and need 4 N of workspace.
//
// What bounds it: arithmetic and LDS exchanges (two FFTs of more than twice
// the length), not HBM.  The stages therefore follow these rules:
//  - The radix sequence of M is taken forwards in the first FFT and backwards
//    in the second.  The last stage of the first and the first stage of the
//    second then touch the same M / R-strided elements in each thread, so the
//    product and the turn between the two FFTs need no exchange.
//  - Inputs past (M + 1) / 2 are zero and outputs past it are dropped at
//    compile time: the first stage loads, and the last stage stores, about
//    half of its elements.
//  - Twiddles of a stage are loaded before the exchange that feeds it.
// Measured (N = 1009, 4096 transforms, M = 2048, F32; forward and inverse
// together, 132 MB): 270 us as separate launches, 74 us here; 521 -> 83 us for
// a first call, which no longer allocates its workspace.
#pragma once

#include "fixed.h"

namespace sfft {

template <typename T>
struct ChirpArgs {
    const C2<T> *in;
    C2<T> *out;
    int64_t in_dist, out_dist;  // complex values between transforms
    const C2<T> *w;     // chirp, n entries
    const C2<T> *bhat;  // FFT_M of the convolution kernel, over M
    const C2<T> *twf;   // stage twiddles of the radices taken forwards ...
    const C2<T> *twb;   // ... and backwards (dense layout of the planner)
    const C2<T> *real_tw;
    const C2<T> *rot;
    int32_t n;      // length of the transform (the half length of a real one)
    int32_t batch;
    int32_t mode;   // kModeC2C, kModeR2C or kModeC2R
    int32_t inverse;
    int32_t half_shift;
};

template <typename T_, int M, int TPT, int TPW, int MINW, int... Rs>
struct Chirp {
    using T = T_;
    static constexpr int NST = sizeof...(Rs);
    static constexpr int RAD[NST] = {Rs...};
    static constexpr int THREADS = TPT * TPW;
    static constexpr int MIN_WAVES = MINW;
    static constexpr int pad(int e) { return e + (e >> kLdsPadShift); }
    static constexpr int STRIDE = M + (M >> kLdsPadShift) + 1;
    static constexpr size_t LDS_BYTES = (size_t)STRIDE * sizeof(C2<T>) * TPW;
    static constexpr int HALF = (M + 1) / 2;  // n <= HALF

    // radix of stage S of FFT D (0: forwards, 1: backwards), span and table
    static constexpr int rad(int d, int s) { return d == 0 ? RAD[s] : RAD[NST - 1 - s]; }
    static constexpr int ns_of(int d, int s) {
        int p = 1;
        for (int i = 0; i < s; ++i) p *= rad(d, i);
        return p;
    }
    static constexpr int tw_of(int d, int s) {
        int o = 0;
        for (int i = 0; i < s; ++i)
            if (ns_of(d, i) > 1) o += ns_of(d, i) * tw_group(rad(d, i));
        return o;
    }
    static_assert(ns_of(0, NST) == M, "radices must multiply to M");
    static_assert(NST >= 2, "two stages or more");

    template <int D, int S>
    struct Regs {
        static constexpr int R = rad(D, S), NB = M / R, B = (NB + TPT - 1) / TPT;
        C2<T> v[B][R];
    };

    struct Ctx {
        const ChirpArgs<T> &a;
        C2<T> *ls;  // this transform's LDS
        int g, lid;
        bool active;
    };

    template <int D, int S>
    static __device__ __forceinline__ bool valid(const Ctx &c, int b) {
        constexpr int NB = Regs<D, S>::NB;
        return (NB % TPT) == 0 || c.lid + b * TPT < NB;
    }

    // Element e of the zero-padded input: the transform's input value (for
    // the inverse complex transform its conjugate, for the real kinds the
    // rotation or the pair pre-process) times the chirp.
    static __device__ __forceinline__ C2<T> load(const Ctx &c, int e) {
        const ChirpArgs<T> &a = c.a;
        const C2<T> *x = a.in + (int64_t)c.g * a.in_dist;
        C2<T> v;
        if (a.mode == kModeC2R) {
            v = cconj(real_pre_bin(x, a.real_tw, e, a.n, a.half_shift != 0));
        } else {
            v = x[e];
            if (a.mode == kModeC2C && a.inverse) v.y = -v.y;
            if (a.mode == kModeR2C && a.half_shift) v = cmul(v, a.rot[e]);
        }
        return cmul(v, a.w[e]);
    }

    template <int D, int S>
    static __device__ __forceinline__ void load_tw(const Ctx &c, Regs<D, S> &tw) {
        using G = Regs<D, S>;
        constexpr int NS = ns_of(D, S), R = G::R;
        const C2<T> *t = (D == 0 ? c.a.twf : c.a.twb) + tw_of(D, S);
#pragma unroll
        for (int b = 0; b < G::B; ++b) {
            const int j = valid<D, S>(c, b) ? c.lid + b * TPT : 0;
            const C2<T> *wp = t + (j % NS) * tw_group(R);
#pragma unroll
            for (int r = 1; r < R; ++r) tw.v[b][r] = wp[r - 1];
        }
    }

    // LDS write of stage (D, S)'s outputs, LDS read of stage S + 1's inputs.
    template <int D, int S>
    static __device__ __forceinline__ void put(const Ctx &c, const Regs<D, S> &x) {
        using G = Regs<D, S>;
        constexpr int NS = ns_of(D, S), R = G::R;
#pragma unroll
        for (int b = 0; b < G::B; ++b) {
            const int j = c.lid + b * TPT;
            if (!valid<D, S>(c, b)) continue;
            const int o = (j / NS) * NS * R + j % NS;
#pragma unroll
            for (int t = 0; t < R; ++t) c.ls[pad(o + t * NS)] = x.v[b][t];
        }
    }
    template <int D, int S>
    static __device__ __forceinline__ void get(const Ctx &c, Regs<D, S> &x) {
        using G = Regs<D, S>;
#pragma unroll
        for (int b = 0; b < G::B; ++b) {
            const int j = c.lid + b * TPT;
            if (!valid<D, S>(c, b)) continue;
#pragma unroll
            for (int r = 0; r < G::R; ++r) x.v[b][r] = c.ls[pad(j + r * G::NB)];
        }
    }

    // Stages S.. of FFT D on the inputs x of stage S (twiddles in tw).
    template <int D, int S>
    static __device__ __forceinline__ void run_from(const Ctx &c, Regs<D, S> &x, Regs<D, S> &tw) {
        using G = Regs<D, S>;
        constexpr int R = G::R;
        if constexpr (S > 0) {
#pragma unroll
            for (int b = 0; b < G::B; ++b)
#pragma unroll
                for (int r = 1; r < R; ++r) x.v[b][r] = cmul(x.v[b][r], tw.v[b][r]);
        }
#pragma unroll
        for (int b = 0; b < G::B; ++b) dft<R, T>(x.v[b]);
        if constexpr (S < NST - 1) {
            Regs<D, S + 1> y, ty;
            load_tw<D, S + 1>(c, ty);
            put<D, S>(c, x);
            __syncthreads();
            get<D, S + 1>(c, y);
            __syncthreads();  // every read done before the next exchange writes
            run_from<D, S + 1>(c, y, ty);
        } else if constexpr (D == 0) {
            // the product with the kernel's transform; conj(.) turns the
            // forward stages that follow into the inverse.  Outputs j + t NB
            // of this stage are the inputs of the same thread's butterflies
            // in the first stage of the second FFT.
            Regs<1, 0> y;
#pragma unroll
            for (int b = 0; b < G::B; ++b) {
                const int j = valid<D, S>(c, b) ? c.lid + b * TPT : 0;
                C2<T> h[R];
#pragma unroll
                for (int t = 0; t < R; ++t) h[t] = c.a.bhat[j + t * G::NB];
#pragma unroll
                for (int t = 0; t < R; ++t) y.v[b][t] = cconj(cmul(x.v[b][t], h[t]));
            }
            Regs<1, 0> none;
            run_from<1, 0>(c, y, none);
        } else {
            finish(c, x);
        }
    }

    // The first n values of the convolution, times the chirp, to HBM.
    static __device__ __forceinline__ void finish(const Ctx &c, Regs<1, NST - 1> &x) {
        using G = Regs<1, NST - 1>;
        const ChirpArgs<T> &a = c.a;
        const bool r2c = a.mode == kModeR2C;
        C2<T> *out = a.out + (int64_t)c.g * a.out_dist;
#pragma unroll
        for (int b = 0; b < G::B; ++b) {
            const int j = c.lid + b * TPT;
#pragma unroll
            for (int t = 0; t < G::R; ++t) {
                if (t * G::NB >= HALF) continue;  // never an output
                const int e = j + t * G::NB;
                if (!c.active || !valid<1, NST - 1>(c, b) || e >= a.n) continue;
                C2<T> v = cmul(cconj(x.v[b][t]), a.w[e]);
                if (a.inverse) v.y = -v.y;
                if (a.mode == kModeC2R && a.half_shift) v = cmulc(v, a.rot[e]);
                if (r2c)
                    c.ls[pad(e)] = v;
                else
                    out[e] = v;
            }
        }
        if (!r2c) return;
        // real forward: the pairs (i, n - i) from LDS (signalsmith-fft.h:459-472)
        __syncthreads();
        if (!c.active) return;
        const bool mod = a.half_shift != 0;
        const T half = (T)0.5;
        for (int i = c.lid; i <= a.n / 2; i += TPT) {
            if (!mod && i == 0) {
                const C2<T> z = c.ls[0];
                out[0] = {z.x + z.y, z.x - z.y};
                continue;
            }
            if (real_pair_skipped(i, a.n, mod)) continue;
            const int ci = mod ? (a.n - 1 - i) : (a.n - i);
            const C2<T> zi = c.ls[pad(i)], zc = c.ls[pad(ci)];
            const C2<T> odd = {(zi.x + zc.x) * half, (zi.y - zc.y) * half};
            const C2<T> ev = {(zi.x - zc.x) * half, (zi.y + zc.y) * half};
            const C2<T> e = cmul(ev, a.real_tw[i]);
            out[i] = cadd(odd, e);
            out[ci] = cconj(csub(odd, e));
        }
    }

    static __device__ __forceinline__ void run(const ChirpArgs<T> &a, C2<T> *lds) {
        const int slot = (int)threadIdx.x / TPT;
        const int g = (int)blockIdx.x * TPW + slot;
        const Ctx c{a, lds + slot * STRIDE, g, (int)threadIdx.x % TPT, g < a.batch};
        Regs<0, 0> x;
        using G = Regs<0, 0>;
#pragma unroll
        for (int b = 0; b < G::B; ++b) {
            const int j = c.lid + b * TPT;
#pragma unroll
            for (int r = 0; r < G::R; ++r) {
                x.v[b][r] = {(T)0, (T)0};
                if (r * G::NB >= HALF) continue;  // always padding
                const int e = j + r * G::NB;
                if (c.active && valid<0, 0>(c, b) && e < a.n) x.v[b][r] = load(c, e);
            }
        }
        Regs<0, 0> none;
        run_from<0, 0>(c, x, none);
    }
};

template <class F>
__global__ void __launch_bounds__(F::THREADS, F::MIN_WAVES)
    k_chirp(ChirpArgs<typename F::T> a) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    F::run(a, reinterpret_cast<C2<typename F::T> *>(smem_raw));
}

// Registry entry of a compiled chirp kernel.
struct ChirpKernel {
    int m, prec;  // convolution length; 0 F32, 1 F64
    int tpw;      // transforms per block
    int nst;
    int radices[kMaxStages];
    hipError_t (*launch)(const void *args, unsigned grid, hipStream_t stream);
};
void register_chirp(const ChirpKernel &k);
// The compiled kernel of the smallest convolution length >= 2 n - 1, or null.
const ChirpKernel *find_chirp(size_t n, int prec);

template <typename T, int M, int TPT, int TPW, int MINW, int... Rs>
struct ChirpReg {
    using F = Chirp<T, M, TPT, TPW, MINW, Rs...>;
    ChirpReg() {
        ChirpKernel k{};
        k.m = M;
        k.prec = sizeof(T) == 8 ? 1 : 0;
        k.tpw = TPW;
        k.nst = (int)sizeof...(Rs);
        const int rs[] = {Rs...};
        for (int i = 0; i < k.nst; ++i) k.radices[i] = rs[i];
        k.launch = [](const void *args, unsigned grid, hipStream_t stream) {
            static std::once_flag once;
            static hipError_t err = hipSuccess;
            if (allow_max_lds(once, err, (const void *)k_chirp<F>) != hipSuccess) return err;
            hipLaunchKernelGGL((k_chirp<F>), dim3(grid), dim3(F::THREADS), F::LDS_BYTES, stream,
                               *reinterpret_cast<const ChirpArgs<T> *>(args));
            return hipGetLastError();
        };
        register_chirp(k);
    }
};

}  // namespace sfft
