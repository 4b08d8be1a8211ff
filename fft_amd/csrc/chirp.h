// chirp.h -- chirp-z transforms in one launch (short lengths) or three.
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
// together, 132 MB): 270 us as separate launches, 66 us here; 521 -> 72 us for
// a first call, which no longer allocates its workspace.
//
// Longer lengths take M = N1 N2 and three launches over a workspace of M
// values per transform, element n = n1 N2 + n2 at its own place:
//   columns (k_chirp_in):  x times the chirp, zeros, FFT of length N1
//   rows    (k_chirp, ROWS): times W_M^{k1 n2}, FFT of length N2, times the
//           transformed kernel, conj, FFT of length N2, times W_M^{k1 n2}
//   columns (k_chirp_out): FFT of length N1, conj, times the chirp
// The four-step transform of the first FFT and that of the second meet in the
// middle: the second undoes the first's digit order, so neither is transposed
// and both row FFTs (with the product between them) are one launch.  The
// workspace is written and read twice (about 10 N values of HBM traffic in
// all) where the launch sequence with two-pass FFTs moved about 30 N.
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
    int32_t rows;  // rows of a convolution of three launches: transform g is
                   // row g mod rows, and w / bhat hold rows x M entries
};

template <typename T_, int M, int TPT, int TPW, int MINW, bool ROWS, int... Rs>
struct Chirp {
    using T = T_;
    static constexpr int NST = sizeof...(Rs);
    static constexpr int RAD[NST] = {Rs...};
    static constexpr int THREADS = TPT * TPW;
    static constexpr int MIN_WAVES = MINW;
    static constexpr int pad(int e) { return e + (e >> kLdsPadShift); }
    static constexpr int STRIDE = M + (M >> kLdsPadShift) + 1;
    static constexpr size_t LDS_BYTES = (size_t)STRIDE * sizeof(C2<T>) * TPW;
    static constexpr int HALF = ROWS ? M : (M + 1) / 2;  // n <= HALF

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
        const C2<T> *w, *bhat;
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
        if constexpr (ROWS) return cmul(x[e], c.w[e]);
        C2<T> v;
        if (a.mode == kModeC2R) {
            v = cconj(real_pre_bin(x, a.real_tw, e, a.n, a.half_shift != 0));
        } else {
            v = x[e];
            if (a.mode == kModeC2C && a.inverse) v.y = -v.y;
            if (a.mode == kModeR2C && a.half_shift) v = cmul(v, a.rot[e]);
        }
        return cmul(v, c.w[e]);
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
                for (int t = 0; t < R; ++t) h[t] = c.bhat[j + t * G::NB];
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
                if (!c.active || !valid<1, NST - 1>(c, b)) continue;
                if constexpr (ROWS) {
                    out[e] = cmul(x.v[b][t], c.w[e]);
                    continue;
                }
                if (e >= a.n) continue;
                C2<T> v = cmul(cconj(x.v[b][t]), c.w[e]);
                if (a.inverse) v.y = -v.y;
                if (a.mode == kModeC2R && a.half_shift) v = cmulc(v, a.rot[e]);
                if (r2c)
                    c.ls[pad(e)] = v;
                else
                    out[e] = v;
            }
        }
        if (ROWS || !r2c) return;
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
        const size_t row = ROWS ? (size_t)(g % a.rows) * M : 0;
        const Ctx c{a,  lds + slot * STRIDE, g, (int)threadIdx.x % TPT, g < a.batch, a.w + row,
                    a.bhat + row};
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
                if (c.active && valid<0, 0>(c, b) && (ROWS || e < a.n)) x.v[b][r] = load(c, e);
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

// The column passes of a convolution of three launches (IN: the first, else
// the last).  A block holds TPW adjacent columns (256-byte rows), lanes over
// columns in every stage: HBM rows and LDS (odd column pitch) are both read
// and written without conflicts, and the lanes of a column group share their
// twiddles.  Two stages (R0, R1), so one exchange.
template <typename T>
struct ChirpColArgs {
    const C2<T> *in;
    C2<T> *out;
    int64_t in_dist, out_dist;  // complex values between transforms
    const C2<T> *w;             // chirp, n entries
    const C2<T> *tw;            // twiddles of the second stage
    const C2<T> *real_tw;
    const C2<T> *rot;
    FastDiv tiles;  // column tiles per transform
    int32_t n, n2;  // transform length, columns
    int32_t mode, inverse, half_shift;
};

template <typename T_, int TPW, bool IN, int R0, int R1>
struct ChirpCol {
    using T = T_;
    static constexpr int N1 = R0 * R1;
    static constexpr int TPT = R0 > R1 ? R0 : R1;  // stage 0: R1 butterflies, stage 1: R0
    static constexpr int THREADS = TPT * TPW;
    static constexpr int MIN_WAVES = sizeof(T) == 8 ? 2 : 4;
    static constexpr int pad(int e) { return e + (e >> kLdsPadShift); }
    static constexpr int STRIDE = (N1 + (N1 >> kLdsPadShift)) | 1;
    static constexpr size_t LDS_BYTES = (size_t)STRIDE * sizeof(C2<T>) * TPW;

    static __device__ __forceinline__ void run(const ChirpColArgs<T> &a, C2<T> *lds) {
        const int col = (int)threadIdx.x % TPW, lid = (int)threadIdx.x / TPW;
        const uint32_t b = fdiv(blockIdx.x, a.tiles);
        const int c = (int)(blockIdx.x - b * a.tiles.d) * TPW + col;
        const C2<T> *x = a.in + (int64_t)b * a.in_dist;
        C2<T> *y = a.out + (int64_t)b * a.out_dist;
        C2<T> *ls = lds + col * STRIDE;
        const int n2 = a.n2;
        if (lid < R1) {
            C2<T> v[R0];
#pragma unroll
            for (int r = 0; r < R0; ++r) {
                const int e = (lid + r * R1) * n2 + c;
                v[r] = {(T)0, (T)0};
                if constexpr (IN) {
                    if (2 * r >= R0) continue;  // always padding: e >= M / 2 >= n
                    if (e < a.n) v[r] = load(a, x, e);
                } else {
                    v[r] = x[e];
                }
            }
            dft<R0, T>(v);
#pragma unroll
            for (int t = 0; t < R0; ++t) ls[pad(lid * R0 + t)] = v[t];
        }
        C2<T> w[R1];
        if (lid < R0) {
#pragma unroll
            for (int r = 1; r < R1; ++r) w[r] = a.tw[lid * tw_group(R1) + r - 1];
        }
        __syncthreads();
        if (lid >= R0) return;
        C2<T> v[R1];
        v[0] = ls[pad(lid)];
#pragma unroll
        for (int r = 1; r < R1; ++r) v[r] = cmul(ls[pad(lid + r * R0)], w[r]);
        dft<R1, T>(v);
#pragma unroll
        for (int t = 0; t < R1; ++t) {
            const int e = (lid + t * R0) * n2 + c;
            if constexpr (IN) {
                y[e] = v[t];
            } else {
                if (2 * t >= R1) continue;  // never an output
                if (e >= a.n) continue;
                C2<T> z = cmul(cconj(v[t]), a.w[e]);
                if (a.inverse) z.y = -z.y;
                if (a.mode == kModeC2R && a.half_shift) z = cmulc(z, a.rot[e]);
                y[e] = z;
            }
        }
    }

    static __device__ __forceinline__ C2<T> load(const ChirpColArgs<T> &a, const C2<T> *x, int e) {
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
};

template <class F>
__global__ void __launch_bounds__(F::THREADS, F::MIN_WAVES)
    k_chirp_col(ChirpColArgs<typename F::T> a) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    F::run(a, reinterpret_cast<C2<typename F::T> *>(smem_raw));
}

// Registry entry of a compiled chirp kernel.
enum : int { kChirpWhole = 0, kChirpRows = 1, kChirpCols = 2 };
struct ChirpKernel {
    int m, prec;  // convolution, row or column length; 0 F32, 1 F64
    int part;     // kChirpWhole, kChirpRows or kChirpCols
    int tpt, tpw;  // threads per transform, row or column; these per block
    int nst;
    int radices[kMaxStages];
    // out: the second column pass (kChirpCols)
    hipError_t (*launch)(const void *args, int out, unsigned grid, hipStream_t stream);
};
void register_chirp(const ChirpKernel &k);
// The compiled kernel of the smallest convolution length >= 2 n - 1, or null.
const ChirpKernel *find_chirp(size_t n, int prec);
// The column and row kernels of the smallest M = N1 N2 >= 2 n - 1 (the larger
// N1 where two have the same M); false if there is none.
bool find_chirp_split(size_t n, int prec, const ChirpKernel *&cols, const ChirpKernel *&rows);

template <class K, class Args>
hipError_t chirp_launch(const K *kernel, unsigned threads, size_t lds, const void *args,
                        unsigned grid, hipStream_t stream, std::once_flag &once,
                        hipError_t &err) {
    if (allow_max_lds(once, err, (const void *)kernel) != hipSuccess) return err;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(threads), lds, stream,
                       *reinterpret_cast<const Args *>(args));
    return hipGetLastError();
}

template <typename T, bool ROWS, int M, int TPT, int TPW, int MINW, int... Rs>
struct ChirpReg {
    using F = Chirp<T, M, TPT, TPW, MINW, ROWS, Rs...>;
    ChirpReg() {
        ChirpKernel k{};
        k.m = M;
        k.prec = sizeof(T) == 8 ? 1 : 0;
        k.part = ROWS ? kChirpRows : kChirpWhole;
        k.tpt = TPT;
        k.tpw = TPW;
        k.nst = (int)sizeof...(Rs);
        const int rs[] = {Rs...};
        for (int i = 0; i < k.nst; ++i) k.radices[i] = rs[i];
        k.launch = [](const void *args, int, unsigned grid, hipStream_t stream) {
            static std::once_flag once;
            static hipError_t err = hipSuccess;
            return chirp_launch<void(ChirpArgs<T>), ChirpArgs<T>>(
                k_chirp<F>, F::THREADS, F::LDS_BYTES, args, grid, stream, once, err);
        };
        register_chirp(k);
    }
};

template <typename T, int TPW, int R0, int R1>
struct ChirpColReg {
    using FI = ChirpCol<T, TPW, true, R0, R1>;
    using FO = ChirpCol<T, TPW, false, R0, R1>;
    ChirpColReg() {
        ChirpKernel k{};
        k.m = R0 * R1;
        k.prec = sizeof(T) == 8 ? 1 : 0;
        k.part = kChirpCols;
        k.tpt = FI::TPT;
        k.tpw = TPW;
        k.nst = 2;
        k.radices[0] = R0;
        k.radices[1] = R1;
        k.launch = [](const void *args, int out, unsigned grid, hipStream_t stream) {
            static std::once_flag once_in, once_out;
            static hipError_t err_in = hipSuccess, err_out = hipSuccess;
            return out ? chirp_launch<void(ChirpColArgs<T>), ChirpColArgs<T>>(
                             k_chirp_col<FO>, FO::THREADS, FO::LDS_BYTES, args, grid, stream,
                             once_out, err_out)
                       : chirp_launch<void(ChirpColArgs<T>), ChirpColArgs<T>>(
                             k_chirp_col<FI>, FI::THREADS, FI::LDS_BYTES, args, grid, stream,
                             once_in, err_in);
        };
        register_chirp(k);
    }
};

}  // namespace sfft
