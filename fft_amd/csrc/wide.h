// wide.h -- column passes whose tile does not fit LDS as complex values.
//
// A column tile should be at least 64 bytes wide: of a 4096-length FP32 column
// LDS holds four (32-byte rows), and neighbouring tiles then fetch the same
// HBM lines again.  Here a tile of eight columns (256 KB) stays in registers,
// and the exchange between two stages goes through LDS one component at a time
// (real parts, then imaginary parts), so that a plane of the tile is all LDS
// has to hold.  One block per CU, 512 threads of 64 values: no next tile can be
// held beside this one, and the loads of a tile are in flight with the stores
// of the tile before it instead.
//
// The arithmetic is that of the runtime-planned pass for the same radices, so
// the bits are the same.
#pragma once

#include "fixed.h"
#include "kernels.h"

namespace sfft {

constexpr int kFineEntries = 1 << kFineShift;

template <typename T_, int N, int TPT, int TPW, int MODE, class SCH, int... Rs>
struct Wide {
    using T = typename FixedElem<T_>::T;
    using ST = Storage<T, typename FixedElem<T_>::S>;
    using FX = Fixed<T_, N, TPT, TPW, MODE, SCH, Rs...>;  // addresses, table offsets
    static constexpr int MINW = SCH::MINW;
    static constexpr bool PREFETCH = true;  // (persistent)
    static constexpr int NST = sizeof...(Rs);
    static constexpr int RAD[NST] = {Rs...};
    static constexpr int THREADS = TPT * TPW;
    static constexpr int EL = N / TPT;  // values per thread
    static constexpr uint32_t DB = FX::DB;
    static constexpr int pad(int e) { return e + (e >> kLdsPadShift); }
    // plane pitch of a column: columns 8 banks apart, which with lanes of 8
    // columns x 8 consecutive (or 17-strided) elements meets every bank once
    static constexpr int STRIDE = (pad(N) + 63) / 64 * 64 + 8;
    static constexpr size_t PLANE_BYTES = (size_t)STRIDE * TPW * sizeof(T);
    // The fine table of a two-level four-step twiddle, where it fits beside
    // the planes: its index c e mod 2^shift scatters over the lanes, 64 cache
    // lines a load from L1 (4096 x 4096: 114 us with both levels in memory).
    static constexpr int FINE = MODE == kModeColRow && sizeof(T) == 4 ? kFineEntries : 0;
    static constexpr size_t LDS_BYTES = PLANE_BYTES + (size_t)FINE * sizeof(C2<T>);
    static constexpr int ns_of(int s) { return FX::ns_of(s); }
    static constexpr bool even() {
        for (int r : {Rs...})
            if ((N / r) % TPT) return false;
        return true;
    }
    static_assert(N % TPT == 0 && even(), "whole butterflies per thread in every stage");

    // lanes over columns, except where rows are stored
    template <int S>
    static __device__ __forceinline__ void map_of(int &slot, int &lid) {
        constexpr bool ROWS = MODE == kModeColRow && S == NST - 1;
        const int tid = (int)threadIdx.x;
        slot = ROWS ? tid / TPT : tid % TPW;
        lid = ROWS ? tid % TPT : tid / TPW;
    }

    // stage S's outputs to stage S + 1's inputs, one plane at a time.  Every
    // LDS address is the thread's base plus a constant: butterflies of a
    // thread are TPT apart, and TPT, NS R and N / R are multiples of the pad
    // period (or the run of a butterfly's outputs stays within one).
    template <int S>
    static __device__ __forceinline__ void exchange(T *lds, C2<T> (&v)[EL]) {
        constexpr int R = RAD[S], NS = ns_of(S), RN = RAD[S + 1], NBN = N / RN;
        constexpr int P = 1 << kLdsPadShift;
        static_assert(TPT % NS == 0, "a thread's butterflies share j mod NS");
        static_assert(NS % P == 0 || (NS == 1 && R <= P && P % R == 0), "separable write addresses");
        static_assert(NBN % P == 0 && TPT % P == 0, "separable read addresses");
        int slot, lid, slotn, lidn;
        map_of<S>(slot, lid);
        map_of<S + 1>(slotn, lidn);
        T *ls = lds + (slot * STRIDE + pad((lid / NS) * NS * R + lid % NS));
        const T *ln = lds + (slotn * STRIDE + pad(lidn));
        auto put = [&](auto part) {
            constexpr bool IM = decltype(part)::value;
#pragma unroll
            for (int b = 0; b < EL / R; ++b)
#pragma unroll
                for (int t = 0; t < R; ++t)
                    ls[pad(b * TPT * R) + pad(t * NS)] = IM ? v[b * R + t].y : v[b * R + t].x;
        };
        auto get = [&](auto part) {
            constexpr bool IM = decltype(part)::value;
#pragma unroll
            for (int b = 0; b < EL / RN; ++b)
#pragma unroll
                for (int r = 0; r < RN; ++r) {
                    const T q = ln[pad(b * TPT) + pad(r * NBN)];
                    if constexpr (IM)
                        v[b * RN + r].y = q;
                    else
                        v[b * RN + r].x = q;
                }
        };
        put(std::integral_constant<bool, false>{});
        __syncthreads();
        get(std::integral_constant<bool, false>{});
        __syncthreads();
        put(std::integral_constant<bool, true>{});
        __syncthreads();
        get(std::integral_constant<bool, true>{});
        __syncthreads();
    }

    template <int S>
    static __device__ __forceinline__ void stages_from(const FixedArgs<T> &a, T *lds,
                                                       C2<T> (&v)[EL]) {
        constexpr int R = RAD[S], NS = ns_of(S);
        int slot, lid;
        map_of<S>(slot, lid);
#pragma unroll
        for (int b = 0; b < EL / R; ++b) {
            C2<T> x[R];
            if constexpr (NS > 1) {
                const int k = (lid + b * TPT) % NS;
                const C2<T> *w = a.tw + (FX::tw_of(S) + k * tw_group(R));
                // (FP64: four twiddles at a time, for registers)
                constexpr int Q = sizeof(T) == 8 ? 4 : R;
                x[0] = v[b * R];
#pragma unroll
                for (int r0 = 0; r0 < R; r0 += Q) {
                    C2<T> q[Q];
#pragma unroll
                    for (int r = 0; r < Q; ++r)
                        if (r0 + r > 0 && r0 + r < R) q[r] = w[r0 + r - 1];
#pragma unroll
                    for (int r = 0; r < Q; ++r)
                        if (r0 + r > 0 && r0 + r < R) x[r0 + r] = cmul(v[b * R + r0 + r], q[r]);
                    if (Q < R) __builtin_amdgcn_sched_barrier(0);
                }
            } else {
#pragma unroll
                for (int r = 0; r < R; ++r) x[r] = v[b * R + r];
            }
            dft<R, T>(x);
#pragma unroll
            for (int r = 0; r < R; ++r) v[b * R + r] = x[r];
            // one butterfly's temporaries at a time: the tile fills the
            // registers
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (S + 1 < NST) {
            exchange<S>(lds, v);
            stages_from<S + 1>(a, lds, v);
        }
    }

    static __device__ __forceinline__ void load(const FixedArgs<T> &a, int g, int lid,
                                                C2<T> (&v)[EL]) {
        if (g >= a.total_slots) return;
        constexpr int R = RAD[0], NB = N / R;
        const char *src = reinterpret_cast<const char *>(a.in);
        uint32_t t, c;
        FX::column_of(a, g, t, c);
        const uint32_t es = (uint32_t)a.in_es * DB;
        const uint32_t lane =
            (t * (uint32_t)a.in_bs + c * (uint32_t)a.in_ss) * DB + (uint32_t)lid * es;
#pragma unroll
        for (int b = 0; b < EL / R; ++b)
#pragma unroll
            for (int r = 0; r < R; ++r) {
                v[b * R + r] = FX::ld(src + (lane + (uint32_t)(b * TPT + r * NB) * es));
                flip_im(v[b * R + r], a.flip_in);
            }
    }

    static __device__ __forceinline__ void store(const FixedArgs<T> &a, const C2<T> *fine, int g,
                                                 int lid, C2<T> (&v)[EL]) {
        if (g >= a.total_slots) return;
        constexpr int S = NST - 1, R = RAD[S], NS = ns_of(S);
        char *dst = reinterpret_cast<char *>(a.out);
        uint32_t t, c;
        FX::column_of(a, g, t, c);
        const uint32_t es = (uint32_t)a.out_es * DB;
        const uint32_t base = (t * (uint32_t)a.out_bs + c * (uint32_t)a.out_ss) * DB;
        const uint32_t mask = (1u << a.ptw_shift) - 1u;
#pragma unroll
        for (int b = 0; b < EL / R; ++b) {
            const uint32_t o = (uint32_t)(lid + b * TPT);  // NS R = N: j < NS
            // four-step factors W_N^{c e}, a butterfly's loads together (FP64:
            // four at a time)
            constexpr int Q = sizeof(T) == 8 ? 4 : R;
#pragma unroll
            for (int r0 = 0; r0 < R; r0 += Q) {
                C2<T> f[Q];
            if (a.post_tw && a.ptw_full) {
#pragma unroll
                for (int r = 0; r < Q; ++r)
                    f[r] = a.ptw_full[c * (uint32_t)N + (o + (uint32_t)((r0 + r) * NS))];
            } else if (a.post_tw) {
                C2<T> co[Q];
#pragma unroll
                for (int r = 0; r < Q; ++r) {
                    const uint32_t m = c * (o + (uint32_t)((r0 + r) * NS));
                    co[r] = a.ptw_coarse[m >> a.ptw_shift];
                    if (FINE && fine)
                        f[r] = fine[m & mask];
                    else
                        f[r] = a.ptw_fine[m & mask];
                }
#pragma unroll
                for (int r = 0; r < Q; ++r) f[r] = cmul(f[r], co[r]);
            }
#pragma unroll
            for (int r = 0; r < Q; ++r) {
                C2<T> y = v[b * R + r0 + r];
                flip_im(y, a.flip_out);
                if (a.post_tw) y = cmul(y, f[r]);
                FX::st(dst + (base + (o + (uint32_t)((r0 + r) * NS)) * es), y);
            }
            __builtin_amdgcn_sched_barrier(0);
            }
        }
    }

    static __device__ __forceinline__ void run(const FixedArgs<T> &a, char *lds_c) {
        T *lds = reinterpret_cast<T *>(lds_c);
        const int ngroups = (a.total_slots + TPW - 1) / TPW;
        int slot, lid, slot_out, lid_out;
        map_of<0>(slot, lid);
        map_of<NST - 1>(slot_out, lid_out);
        // (XCD-contiguous windows: tiles narrower than a line share it)
        const int G = (int)gridDim.x;
        C2<T> *fine = nullptr;
        if constexpr (FINE > 0) {
            if (a.post_tw && !a.ptw_full && (1 << a.ptw_shift) <= FINE) {
                fine = reinterpret_cast<C2<T> *>(lds_c + PLANE_BYTES);
                for (int i = (int)threadIdx.x; i < (1 << a.ptw_shift); i += THREADS)
                    fine[i] = a.ptw_fine[i];  // (read after the exchanges' barriers)
            }
        }
        for (int grp = (int)xcd_tile(blockIdx.x, (unsigned)G); grp < ngroups; grp += G) {
            C2<T> v[EL];
            load(a, grp * TPW + slot, lid, v);
            stages_from<0>(a, lds, v);
            store(a, fine, grp * TPW + slot_out, lid_out, v);
        }
    }
};

// Registers the column passes of a wide tile (registry kind 3).
template <typename T, int N, int TPT, int TPW, class SCH, int... Rs>
struct WideCol {
    template <int MODE>
    using F = Wide<T, N, TPT, TPW, MODE, SCH, Rs...>;
    WideCol() {
        FixedKernel k{};
        k.n = N;
        k.prec = FixedElem<T>::prec;
        k.real = 3;
        k.tpt = TPT;
        k.tpw = k.row_tpw = k.col_tpw = TPW;
        fixed_fill_radices<Rs...>(k);
        k.lds_bytes = F<kModeColRow>::LDS_BYTES;
        k.launch = [](const void *args, int mode, unsigned grid, hipStream_t s) {
            return mode == kModeColCol ? fixed_launch_one<F<kModeColCol>>(args, grid, s)
                                       : fixed_launch_one<F<kModeColRow>>(args, grid, s);
        };
        k.blocks_per_cu = [](int mode) {
            return mode == kModeColCol ? fixed_occupancy<F<kModeColCol>>()
                                       : fixed_occupancy<F<kModeColRow>>();
        };
        register_fixed(k);
    }
};

}  // namespace sfft
