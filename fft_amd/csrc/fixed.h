// fixed.h -- compile-time planned, persistent, software-pipelined transforms.
//
// For the lengths that carry most traffic the radix sequence, spans, thread
// layout and LDS offsets are template constants: index arithmetic folds into
// immediates and each kernel holds only its own stages.  The kernels compute
// exactly what the runtime-planned pass kernel computes for the same radices
// (same butterflies, same twiddle table, explicit FMAs), so a plan gives the
// same bits on either path.
//
// Two schedules:
//  - One group of slots per block.  Several blocks share a CU, and one's loads
//    overlap another's stages.  With nothing carried round a loop the kernels
//    need 54-90 registers in FP32 instead of 100-170 (the compiler hoists
//    every stage's addresses out of a persistent loop), so 16 to 32 waves stay
//    resident.
//  - Persistent + pipelined, where the tile leaves room for one block per CU
//    only: a block walks groups blockIdx.x, blockIdx.x + gridDim.x, ...; the
//    first stage of a group takes its elements from registers loaded during
//    the previous group, and right after that the next group's loads are
//    issued, so HBM reads overlap the remaining stages.
// The first measured faster at nearly every length whose tile is 80 KB or
// less (256 MB launches, first / second): complex FP32 median 1.08x of 106
// lengths, FP64 1.05x of 112 up to 4860, real 1.13x forward and 1.17x inverse
// of 98 (up to 2.0x), column passes 1.09x (first pass) and 1.19x (second) of
// 38; the second at nearly every length above it (0.80-0.96x).
// Blocks sized for the second schedule are too large for the first: two or
// three per CU, each waiting for its own loads.  Between 30 and 130 MB a launch
// that cost up to 25 % against the second, and lengths that lost 4 % or more
// hold half as many transforms per block (FP64 64 MB, persistent / one group /
// half: 400 24.4 / 30.5 / 26.3 us, 125 27.4 / 32.8 / 27.7, 75 29.5 / 32.1 / 24.4;
// 128 MB: 47.7 / 50.5 / 44.3, 50.1 / 58.0 / 47.3, 47.7 / 52.5 / 43.7), those of one
// transform per block other twiddle loads (Sched TW), or the second schedule
// back (kPersist: FP32 7680, FP64 3240, 3600, 3840, 4320).
#pragma once

#include "stockham.h"

namespace sfft {

constexpr bool ct_pow2(int x) { return x > 0 && (x & (x - 1)) == 0; }

template <typename T>
struct FixedArgs {
    const C2<T> *in;
    C2<T> *out;
    const C2<T> *tw;       // stage twiddles (dense layout of the runtime planner)
    const C2<T> *real_tw;  // twiddlesMinusI, N/4 + 1 entries of the real length
    const C2<T> *rot;      // half-shift rotations
    int32_t total_slots;
    uint32_t flip_in;      // sign-bit mask xor-ed into Im at the HBM load (inverse)
    uint32_t flip_out;     // ... and at the HBM store
    int32_t half_shift;
    // column passes of two-pass plans: slot g is column c = g mod spt of
    // transform b = g / spt; element e of it sits at b bs + c ss + e es
    // (element strides of the input and of the output)
    FastDiv spt;
    int32_t in_bs, in_ss, in_es;
    int32_t out_bs, out_ss, out_es;
    int32_t post_tw, ptw_shift;  // first pass: output element e times W_N^{c e}
    const C2<T> *ptw_fine, *ptw_coarse;
    const C2<T> *ptw_full;  // or null: W_N^{c e} at c N + e (N: this pass' length)
    FastDiv tiles;  // paired column modes: tiles per transform
    uint32_t near;  // column modes: the launch's data fits the L2 caches
};

// Paired column modes.  Bin m = c + S e of a two-pass real transform (column c
// of S = spt, element e of N) pairs with h - m (h - 1 - m for the half shift),
// h = S N: element N - 1 - e of the mirror column S - c (S - 1 - c).  Only
// column 0 (without the shift) pairs within itself at N - e, and the middle
// column at N - 1 - e.  A tile of TPW slots therefore holds TPW / 2 adjacent
// columns and, in the other half of its slots, their mirror columns, and the
// pair sums need nothing from outside the tile: the values are exchanged
// through LDS once (forward: after the last stage; inverse: before the first).
// Without this the forward transform ran a third pass over the output
// (k_real_post) and the inverse the runtime-planned pass with two gathered
// loads an element: 96000 x 512 forward 231 -> 204 us, inverse 246 -> 199;
// 131072 x 256 158 -> 122 and 152 -> 128.
__host__ __device__ inline uint32_t pair_columns(uint32_t s, bool shifted) {
    return (shifted ? (s - 1) / 2 : s / 2) + 1;  // columns that are not mirror images
}

// Sign flip of the imaginary part by a uniform xor mask (0 or the sign bit).
__device__ __forceinline__ void flip_im(C2<float> &x, uint32_t m) {
    x.y = __uint_as_float(__float_as_uint(x.y) ^ m);
}
__device__ __forceinline__ void flip_im(C2<double> &x, uint32_t m) {
    unsigned long long u = __double_as_longlong(x.y);
    u ^= (unsigned long long)m << 32;
    x.y = __longlong_as_double(u);
}

// Schedule knobs of a compiled plan:
//   PFS   stage that issues the next group's loads (>= 0: that stage,
//         -1 the last, -2 the one before)
//   MINW  minimum waves per SIMD the register allocation must allow (0: the
//         compiler's choice) -- more resident blocks per CU, fewer registers
//   PAIR  load twiddles two per 16-byte load (else one per load)
//   PF_FIRST  in the prefetch stage, issue the prefetch before (1) or after
//         (0) the next stage's twiddle loads
//   PADSH one LDS pad element per 2^PADSH elements (kLdsNoPad: none)
//   NT    non-temporal HBM accesses: bit 0 the loads of the input (a single
//         pass, or a first column pass), bit 1 the stores of the final
//         output (a single pass, or a second column pass), bit 2 also in the
//         inverse real kernel of a real pair (else only its forward one);
//         the intermediate of a two-pass plan always keeps the default policy.
//         (On the real 2048 pair of the bench step, non-temporal accesses in
//         the forward kernel made it 10 % faster and the inverse leg that
//         follows it 10 % slower, with no net gain; they are not used there.)
//   TW    1 or 0: one-group kernels load a stage's twiddles before the exchange
//         that feeds it, or after it (-1: as TW_EARLY below has it).
constexpr int kLdsNoPad = 30;
constexpr int kNoPrefetch = -100;  // PFS: never persistent
constexpr int kPersist = 100;      // PFS + kPersist: persistent at any tile size
constexpr unsigned kXcdWindow = 256;  // blocks numbered XCD-contiguously together
// Largest tile of which two blocks fit a CU.
constexpr size_t kSharedCuLds = 80 * 1024;
template <int PFS_, int MINW_, int PAIR_ = 1, int PF_FIRST_ = 0, int PADSH_ = kLdsPadShift,
          int NT_ = 0, int TW_ = -1>
struct Sched {
    static constexpr int PFS = PFS_;
    static constexpr int MINW = MINW_;
    static constexpr int PAIR = PAIR_;
    static constexpr int PF_FIRST = PF_FIRST_;
    static constexpr int PADSH = PADSH_;
    static constexpr int NT = NT_;
    static constexpr int TW = TW_;
    static constexpr bool ROT = false;
};
// Column passes that also rotate (half-bin shifted real transforms): the
// rotations are read as the data is, from a table of one transform.  Kernels of
// their own, because the branch alone cost the plain 1024 pass 20 % (2^20 x 16
// 125 -> 160 us).  Against the runtime-planned pass, both directions of 128 MB
// batches: 1.1-1.4x (218700 397 -> 286 us, FP64 100000 355 -> 255).
template <class S>
struct Rotated : S {
    static constexpr bool ROT = true;
};

// Element type of a compiled kernel: float / double (stored as is), or
// Stored<StoreF16 / StoreBF16> (16-bit pairs in HBM, float arithmetic).
template <class S>
struct Stored {};
template <typename E>
struct FixedElem {
    using T = E;
    using S = StoreNative;
    static constexpr int prec = sizeof(E) == 8 ? 1 : 0;
};
template <>
struct FixedElem<Stored<StoreF32>> {  // FP32 in HBM under FP64 arithmetic
    using T = double;
    using S = StoreF32;
    static constexpr int prec = 4;
};
template <class S_>
struct FixedElem<Stored<S_>> {
    using T = float;
    using S = S_;
    static constexpr int prec = std::is_same<S_, StoreF16>::value ? 2 : 3;
};

template <typename T_, int N, int TPT, int TPW, int MODE, class SCH, int... Rs>
struct Fixed {
    using T = typename FixedElem<T_>::T;
    using ST = Storage<T, typename FixedElem<T_>::S>;
    static constexpr bool PERSIST = SCH::PFS > kPersist / 2;  // (PFS may be negative)
    static constexpr int PFS = PERSIST ? SCH::PFS - kPersist : SCH::PFS;
    static constexpr int MINW = SCH::MINW;
    static constexpr int NST = sizeof...(Rs);
    static constexpr int RAD[NST] = {Rs...};
    static constexpr int THREADS = TPT * TPW;
    // Column modes: stage 0 (and the last stage of the second pass) map
    // adjacent lanes to adjacent slots (columns), so the strided HBM accesses
    // coalesce across columns; the other stages keep slot-major lanes.
    static constexpr bool PRE = MODE == kModeColRowPre, POST = MODE == kModeColColPost;
    static constexpr bool PAIR = PRE || POST;
    static constexpr bool COL = MODE == kModeColRow || MODE == kModeColCol || PAIR;
    static constexpr bool COL_OUT = MODE == kModeColCol;
    static constexpr int PADSH = SCH::PADSH;
    static constexpr int pad(int e) { return e + (e >> PADSH); }
    static constexpr int STRIDE = N + (N >> PADSH) + 1;
    static constexpr uint32_t EB = sizeof(C2<T>);  // bytes per element in LDS
    static constexpr uint32_t DB = ST::kBytes;      // and in HBM
    static constexpr bool NT_MODE = MODE != kModeC2R || (SCH::NT & 4);
    // (the mirror columns of neighbouring pair tiles share lines: no hint)
    static constexpr bool NT_LD =
        ST::native && (SCH::NT & 1) && NT_MODE && MODE != kModeColCol && !PAIR;
    static constexpr bool NT_ST =
        ST::native && (SCH::NT & 2) && NT_MODE && MODE != kModeColRow && !PAIR;
    using V2 = T __attribute__((ext_vector_type(2)));
    static __device__ __forceinline__ C2<T> ld(const char *p) {
        if constexpr (NT_LD) {
            const V2 v = __builtin_nontemporal_load(reinterpret_cast<const V2 *>(p));
            return {v.x, v.y};
        } else {
            return ST::load(p, 0);
        }
    }
    static __device__ __forceinline__ void st(char *p, C2<T> v) {
        if constexpr (NT_ST) {
            V2 w;
            w.x = v.x;
            w.y = v.y;
            __builtin_nontemporal_store(w, reinterpret_cast<V2 *>(p));
        } else {
            ST::store(p, 0, v);
        }
    }
    static constexpr size_t LDS_BYTES =
        (NST > 1 || MODE != kModeC2C) ? (size_t)STRIDE * EB * TPW : 0;
    // Persistent and pipelined only where one block fills a CU (see the top of
    // the file).
    static constexpr bool PREFETCH =
        SCH::PFS != kNoPrefetch && (PERSIST || LDS_BYTES > kSharedCuLds);
    // One group per block: a stage's twiddles are loaded before the exchange
    // that feeds it (FP32 column passes 1-3 % faster, FP64 ones 4-9 %, one 4096
    // transform 5.4 -> 5.1 us; FP64 single passes in blocks of the persistent
    // schedule's size, short of registers, would be up to 14 % slower, and those
    // in blocks of half that are 1-5 % faster: their Sched says so).
    static constexpr bool TW_EARLY =
        !PREFETCH && (SCH::TW >= 0 ? SCH::TW == 1 : sizeof(T) == 4 || COL);

    static constexpr int ns_of(int s) {
        int p = 1;
        for (int i = 0; i < s; ++i) p *= RAD[i];
        return p;
    }
    static constexpr int tw_of(int s) {
        int o = 0;
        for (int i = 0; i < s; ++i)
            if (ns_of(i) > 1) o += ns_of(i) * tw_group(RAD[i]);
        return o;
    }
    static constexpr int bfly_of(int s) { return (N / RAD[s] + TPT - 1) / TPT; }
    static constexpr int PF = bfly_of(0) * RAD[0];
    // The next group's first-stage loads are issued in stage PF_STAGE, after
    // the twiddle loads of that stage and of the next one: vector-memory
    // counters drain in issue order, so waiting for a twiddle never waits for
    // the (slower) HBM prefetch.  (The inverse paired mode issues them a stage
    // later: with the pairs' values they need too many registers in stage 0,
    // 180 -> 145 us at 100000 x 160; with a first radix of 25 that measured
    // the other way round, 211 -> 230 us at 46875 x 400.)
    static constexpr int PF_STAGE =
        !PREFETCH ? NST : PRE && RAD[0] <= 16 ? 1 : PFS >= 0 ? (PFS < NST ? PFS : NST - 1) : ((NST + PFS) > 0 ? (NST + PFS) : 0);
    static_assert(ns_of(NST) == N, "radices must multiply to N");
    static_assert(!COL || NST >= 2, "column kernels need two stages or more");

    // Column c of transform t in slot `slot` of the pass' slot g (g = first
    // slot of the group + slot); false if the slot holds none.
    static __device__ __forceinline__ bool column_of(const FixedArgs<T> &a, int g, uint32_t &t,
                                                     uint32_t &c) {
        if constexpr (PAIR) {
            const uint32_t q = (uint32_t)g / TPW, slot = (uint32_t)g % TPW;
            const uint32_t s = a.spt.d;
            const bool mod = a.half_shift != 0;
            t = fdiv(q, a.tiles);
            const uint32_t cp = (q - t * a.tiles.d) * (TPW / 2) + slot % (TPW / 2);
            c = cp;
            if (g >= a.total_slots || cp >= pair_columns(s, mod)) return false;
            if (slot < TPW / 2) return true;
            c = mod ? s - 1 - cp : s - cp;
            return c != cp && c < s;  // (a column that pairs within itself has no mirror)
        } else {
            t = fdiv((uint32_t)g, a.spt);
            c = (uint32_t)g - t * a.spt.d;
            return g < a.total_slots;
        }
    }

    // Partner of element e of the column c in slot `slot`: LDS index.
    static __device__ __forceinline__ int partner(const FixedArgs<T> &a, uint32_t c, int slot,
                                                  int e) {
        const uint32_t s = a.spt.d;
        const bool mod = a.half_shift != 0;
        const bool own = mod ? 2 * c + 1 == s : (c == 0 || 2 * c == s);
        const int ps = own ? slot : (slot + TPW / 2) % TPW;
        const int pe = (!mod && c == 0) ? (e == 0 ? 0 : N - e) : N - 1 - e;
        return ps * STRIDE + pad(pe);
    }
    // Pair index i of bin m (whose table entry both of its bins use): the
    // smaller of the two, but h / 2 for the shifted kind's middle pair.
    static __device__ __forceinline__ uint32_t pair_index(uint32_t m, uint32_t h, bool mod) {
        const uint32_t mm = mod ? h - 1 - m : h - m;
        const uint32_t i = m < mm ? m : mm;
        return (mod && (h & 1) == 0 && i == h / 2 - 1) ? h / 2 : i;
    }

    // thread -> (slot, element lane) of stage S; gbase = first slot of the group
    template <int S>
    static __device__ __forceinline__ void map_of(const FixedArgs<T> &a, int gbase, int &g,
                                                  int &slot, int &lid, bool &active) {
        constexpr bool CM = COL && (S == 0 || (S == NST - 1 && COL_OUT));
        const int tid = (int)threadIdx.x;
        slot = CM ? tid % TPW : tid / TPT;
        lid = CM ? tid / TPW : tid % TPT;
        g = gbase + slot;
        active = g < a.total_slots;
    }

    // twiddles of stage S for this thread's butterflies
    template <int S, bool = (S < NST)>
    struct TwBuf {
        C2<T> w[1][2];
    };
    template <int S>
    struct TwBuf<S, true> {
        C2<T> w[bfly_of(S)][RAD[S] > 1 ? RAD[S] : 2];
    };

    template <int S>
    static __device__ __forceinline__ void load_tw(const FixedArgs<T> &a, TwBuf<S> &tb,
                                                   bool active, int lid) {
        if constexpr (S < NST) {
            constexpr int R = RAD[S], NS = ns_of(S), NB = N / R, B = bfly_of(S);
            constexpr int TWG = tw_group(R);
            if constexpr (NS > 1) {
#pragma unroll
                for (int b = 0; b < B; ++b) {
                    const int j = lid + b * TPT;
                    if (active && ((NB % TPT) == 0 || j < NB)) {
                        const int k = j % NS;
                        const C2<T> *wp = a.tw + (tw_of(S) + k * TWG);
                        if constexpr (sizeof(T) == 4 && SCH::PAIR && (TWG % 2) == 0) {
                            // 16-byte aligned groups: two twiddles per load
                            const float4 *w4 = reinterpret_cast<const float4 *>(wp);
#pragma unroll
                            for (int p = 0; p < TWG / 2; ++p) {
                                const float4 q = w4[p];
                                if (2 * p + 1 < R) tb.w[b][2 * p + 1] = {q.x, q.y};
                                if (2 * p + 2 < R) tb.w[b][2 * p + 2] = {q.z, q.w};
                            }
                        } else {
#pragma unroll
                            for (int r = 1; r < R; ++r) tb.w[b][r] = wp[r - 1];
                        }
                    }
                }
            }
        }
    }

    // stage-0 element loads of slot g into pf (contiguous batch, or a column)
    static __device__ __forceinline__ void load0(const FixedArgs<T> &a, C2<T> (&pf)[PF], int g,
                                                 int lid) {
        constexpr int R = RAD[0], NB = N / R, B = bfly_of(0);
        if (g >= a.total_slots) return;
        const char *src = reinterpret_cast<const char *>(a.in);
        if constexpr (COL) {
            uint32_t t, c;
            if (!column_of(a, g, t, c) && PAIR) return;
            const uint32_t es = (uint32_t)a.in_es * DB;
            const uint32_t lane =
                (t * (uint32_t)a.in_bs + c * (uint32_t)a.in_ss) * DB + (uint32_t)lid * es;
#pragma unroll
            for (int b = 0; b < B; ++b) {
                if ((NB % TPT) == 0 || lid + b * TPT < NB) {
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        pf[b * R + r] = ld(src + (lane + (uint32_t)(b * TPT + r * NB) * es));
                }
            }
            return;
        }
        const uint32_t lane = ((uint32_t)g * (uint32_t)N + (uint32_t)lid) * DB;
#pragma unroll
        for (int b = 0; b < B; ++b) {
            if ((NB % TPT) == 0 || lid + b * TPT < NB) {
#pragma unroll
                for (int r = 0; r < R; ++r)
                    pf[b * R + r] = ld(src + (lane + (uint32_t)((b * TPT + r * NB) * DB)));
            }
        }
    }

    // Stage S.  TW_READY: its twiddles were loaded by the previous stage.
    // PF_HERE: also load stage S+1's twiddles into tn, then issue the next
    // group's first-stage loads into pf.
    template <int S, bool TW_READY, bool PF_HERE>
    static __device__ __forceinline__ void stage(const FixedArgs<T> &a, char *lds_c, int g_in,
                                                 bool active_in, int slot_in, int lid_in,
                                                 C2<T> (&pf)[PF], int g_next, TwBuf<S> &tb,
                                                 TwBuf<S + 1> &tn) {
        constexpr int R = RAD[S], NS = ns_of(S), NB = N / R, B = bfly_of(S);
        // column modes: g_in is the group's first slot and each stage maps
        // its own lanes (the next stage's twiddles and the prefetch use theirs)
        int g = g_in, slot = slot_in, lid = lid_in, lid_n = lid_in, lid_pf = lid_in;
        bool active = active_in, active_n = active_in;
        if constexpr (COL) {
            map_of<S>(a, g_in, g, slot, lid, active);
            int gx, sx;
            map_of<S + 1>(a, g_in, gx, sx, lid_n, active_n);
            bool ax;
            map_of<0>(a, g_in, gx, sx, lid_pf, ax);
        }
        constexpr bool FIRST = (S == 0), LAST = (S == NST - 1);
        constexpr bool SRC_PF = FIRST && MODE != kModeC2R && !PRE;
        constexpr bool DST_G = LAST && MODE != kModeR2C;
        constexpr bool SEP_R = ct_pow2(NB) || (NB % (1 << PADSH)) == 0;
        constexpr bool SEP_W = (NS % (1 << PADSH)) == 0 || (ct_pow2(NS) && ct_pow2(R));
        const uint32_t lsb = (uint32_t)(slot * STRIDE) * EB;

        auto jvalid = [&](int b) { return (NB % TPT) == 0 || lid + b * TPT < NB; };

        C2<T> v[B][R];
        if constexpr (SRC_PF) {
#pragma unroll
            for (int b = 0; b < B; ++b)
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    v[b][r] = pf[b * R + r];
                    flip_im(v[b][r], a.flip_in);
                }
        }
        // inverse real: the raw bins of the tile to LDS, their pairs'
        // pre-process there (its table loads go before the prefetch, as every
        // other table load)
        constexpr bool PRE_HERE = FIRST && PRE;
        PairWork<PRE_HERE> pair;
        if constexpr (PRE_HERE) {
            C2<T> *ls = reinterpret_cast<C2<T> *>(lds_c);
#pragma unroll
            for (int b = 0; b < B; ++b)
                if (jvalid(b)) {
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        ls[slot * STRIDE + pad(lid + b * TPT + r * NB)] = pf[b * R + r];
                }
            pair.init(a, g - slot);
        }
        if constexpr (!TW_READY) load_tw<S>(a, tb, active, lid);
        if constexpr (PF_HERE) {
            if constexpr (SCH::PF_FIRST) {
                if (PREFETCH && MODE != kModeC2R && g_next >= 0) load0(a, pf, g_next, lid_pf);
                load_tw<S + 1>(a, tn, active_n, lid_n);
            } else {
                load_tw<S + 1>(a, tn, active_n, lid_n);
                if (PREFETCH && MODE != kModeC2R && g_next >= 0) load0(a, pf, g_next, lid_pf);
            }
        }
        if constexpr (PRE_HERE) {
            __syncthreads();
            pair_pre(a, reinterpret_cast<C2<T> *>(lds_c), pair);
            __syncthreads();
        }
        if constexpr (SRC_PF) {
            if (MODE == kModeR2C && a.half_shift) {
#pragma unroll
                for (int b = 0; b < B; ++b) {
                    const int j = lid + b * TPT;
                    if (active && jvalid(b)) {
#pragma unroll
                        for (int r = 0; r < R; ++r) v[b][r] = cmul(v[b][r], a.rot[j + r * NB]);
                    }
                }
            }
            if constexpr (SCH::ROT && MODE == kModeColRow) {
                uint32_t t, c;
                column_of(a, g, t, c);
#pragma unroll
                for (int b = 0; b < B; ++b) {
                    const uint32_t j = (uint32_t)(lid + b * TPT);
                    if (active && jvalid(b)) {
#pragma unroll
                        for (int r = 0; r < R; ++r)
                            v[b][r] = cmul(v[b][r], a.rot[c + (j + (uint32_t)(r * NB)) *
                                                                  (uint32_t)a.in_es]);
                    }
                }
            }
        } else {
#pragma unroll
            for (int b = 0; b < B; ++b) {
                const int j = lid + b * TPT;
                if (active && jvalid(b)) {
                    if constexpr (SEP_R) {
                        const uint32_t la = lsb + (uint32_t)pad(j) * EB;
#pragma unroll
                        for (int r = 0; r < R; ++r)
                            v[b][r] = *reinterpret_cast<const C2<T> *>(
                                lds_c + (la + (uint32_t)(pad(r * NB) * EB)));
                    } else {
#pragma unroll
                        for (int r = 0; r < R; ++r)
                            v[b][r] = *reinterpret_cast<const C2<T> *>(
                                lds_c + (lsb + (uint32_t)pad(j + r * NB) * EB));
                    }
                }
            }
            __syncthreads();  // all reads done before any slot is overwritten
        }
#pragma unroll
        for (int b = 0; b < B; ++b) {
            if (active && jvalid(b)) {
                if constexpr (NS > 1) {
#pragma unroll
                    for (int r = 1; r < R; ++r) v[b][r] = cmul(v[b][r], tb.w[b][r]);
                }
                dft<R, T>(v[b]);
            }
        }
        if constexpr (TW_EARLY && !LAST) load_tw<S + 1>(a, tn, active_n, lid_n);
        if constexpr (DST_G && POST) {
            // the spectrum's tile to LDS, then its pairs to HBM
            // (signalsmith-fft.h:459-472)
            C2<T> *ls = reinterpret_cast<C2<T> *>(lds_c);
#pragma unroll
            for (int b = 0; b < B; ++b) {
                const int j = lid + b * TPT;
                if (jvalid(b)) {
#pragma unroll
                    for (int t2 = 0; t2 < R; ++t2)
                        ls[slot * STRIDE + pad((j / NS) * NS * R + j % NS + t2 * NS)] = v[b][t2];
                }
            }
            PairWork<true> pair_out;
            pair_out.init(a, g - slot);
            __syncthreads();
            pair_post(a, ls, pair_out);
            __syncthreads();  // the tile is read before the next one's exchange
        } else if constexpr (DST_G && COL) {
            char *dst = reinterpret_cast<char *>(a.out);
            uint32_t t, c;
            const bool held = column_of(a, g, t, c);
            if constexpr (PAIR) active = held;
            const uint32_t es = (uint32_t)a.out_es * DB;
            const uint32_t sbase = (t * (uint32_t)a.out_bs + c * (uint32_t)a.out_ss) * DB;
            const uint32_t mask = (1u << a.ptw_shift) - 1u;
#pragma unroll
            for (int b = 0; b < B; ++b)
#pragma unroll
                for (int t2 = 0; t2 < R; ++t2) flip_im(v[b][t2], a.flip_out);
            if constexpr (SCH::ROT && COL_OUT) {
#pragma unroll
                for (int b = 0; b < B; ++b) {
                    const int j = lid + b * TPT;
                    if (active && jvalid(b)) {
                        const int o = (j / NS) * NS * R + j % NS;
#pragma unroll
                        for (int t2 = 0; t2 < R; ++t2)
                            v[b][t2] = cmulc(v[b][t2], a.rot[c + (uint32_t)(o + t2 * NS) *
                                                                     (uint32_t)a.out_es]);
                    }
                }
            }
            if (a.post_tw && a.ptw_full) {
                // the four-step factors from the full table: the lanes of a
                // slot read consecutive entries (lanes without a butterfly
                // read entry 0; never stored)
                const uint32_t crow = active ? c * (uint32_t)N : 0u;
#pragma unroll
                for (int b = 0; b < B; ++b) {
                    const int j = (active && jvalid(b)) ? lid + b * TPT : 0;
                    const int o = (j / NS) * NS * R + j % NS;
#pragma unroll
                    for (int t2 = 0; t2 < R; ++t2)
                        v[b][t2] = cmul(v[b][t2], a.ptw_full[crow + (uint32_t)(o + t2 * NS)]);
                }
            } else if (a.post_tw) {
                // the four-step factors of every element, loaded together
                // (lanes without a butterfly read entry 0; never stored)
#pragma unroll
                for (int b = 0; b < B; ++b) {
                    const int j = (active && jvalid(b)) ? lid + b * TPT : 0;
                    const int o = (j / NS) * NS * R + j % NS;
#pragma unroll
                    for (int t2 = 0; t2 < R; ++t2) {
                        const uint32_t m = active ? c * (uint32_t)(o + t2 * NS) : 0u;
                        v[b][t2] = cmul(v[b][t2],
                                        cmul(a.ptw_fine[m & mask], a.ptw_coarse[m >> a.ptw_shift]));
                    }
                }
            }
#pragma unroll
            for (int b = 0; b < B; ++b) {
                const int j = lid + b * TPT;
                if (active && jvalid(b)) {
                    const int o = (j / NS) * NS * R + j % NS;
#pragma unroll
                    for (int t2 = 0; t2 < R; ++t2)
                        st(dst + (sbase + (uint32_t)(o + t2 * NS) * es), v[b][t2]);
                }
            }
        } else if constexpr (DST_G) {
            char *dst = reinterpret_cast<char *>(a.out);
            const uint32_t sbase = (uint32_t)g * (uint32_t)N;
#pragma unroll
            for (int b = 0; b < B; ++b) {
                const int j = lid + b * TPT;
                if (active && jvalid(b)) {
                    const int o = (j / NS) * NS * R + j % NS;
                    const uint32_t lo = (sbase + (uint32_t)o) * DB;
#pragma unroll
                    for (int t = 0; t < R; ++t) {
                        C2<T> y = v[b][t];
                        flip_im(y, a.flip_out);
                        if (MODE == kModeC2R && a.half_shift) y = cmulc(y, a.rot[o + t * NS]);
                        st(dst + (lo + (uint32_t)(t * NS * DB)), y);
                    }
                }
            }
        } else {
#pragma unroll
            for (int b = 0; b < B; ++b) {
                const int j = lid + b * TPT;
                if (active && jvalid(b)) {
                    const int o = (j / NS) * NS * R + j % NS;
                    if constexpr (SEP_W) {
                        const uint32_t la = lsb + (uint32_t)pad(o) * EB;
#pragma unroll
                        for (int t = 0; t < R; ++t)
                            *reinterpret_cast<C2<T> *>(
                                lds_c + (la + (uint32_t)(pad(t * NS) * EB))) = v[b][t];
                    } else {
#pragma unroll
                        for (int t = 0; t < R; ++t)
                            *reinterpret_cast<C2<T> *>(
                                lds_c + (lsb + (uint32_t)pad(o + t * NS) * EB)) = v[b][t];
                    }
                }
            }
            __syncthreads();
        }
    }

    // A thread's pairs of a paired tile: column c in its slot (of the first
    // TPW / 2), elements e0 + k STEP, and their table entries.
    template <bool USED>
    struct PairWork {};
    template <>
    struct PairWork<true> {
        static constexpr int H = TPW > 1 ? TPW / 2 : 1, STEP = THREADS / H,
                             IT = (N + STEP - 1) / STEP;
        int slot, e0;
        uint32_t t, c;
        bool held;
        C2<T> w[IT];
        __device__ __forceinline__ void init(const FixedArgs<T> &a, int gbase) {
            slot = (int)threadIdx.x % H;
            e0 = (int)threadIdx.x / H;
            held = column_of(a, gbase + slot, t, c) && e0 < STEP;
            const uint32_t s = a.spt.d, h = s * (uint32_t)N;
#pragma unroll
            for (int k = 0; k < IT; ++k) {
                const int e = e0 + k * STEP;
                w[k] = a.real_tw[held && e < N
                                     ? pair_index(c + s * (uint32_t)e, h, a.half_shift != 0)
                                     : 0u];
            }
        }
        // Calls f(k, z, o, m, mm, first): bins m (LDS place z) and mm (place
        // o) of each pair; first: m is the pair's bin i.
        template <typename F>
        __device__ __forceinline__ void each(const FixedArgs<T> &a, F &&f) const {
            if (!held) return;
            const uint32_t s = a.spt.d, h = s * (uint32_t)N;
            const bool mod = a.half_shift != 0;
            // within one column each pair is met from both sides
            const bool own = mod ? 2 * c + 1 == s : (c == 0 || 2 * c == s);
#pragma unroll
            for (int k = 0; k < IT; ++k) {
                const int e = e0 + k * STEP;
                if (e >= N) continue;
                const uint32_t m = c + s * (uint32_t)e;
                const uint32_t mm = mod ? h - 1 - m : h - m;
                if (own && m > mm && m != 0) continue;
                f(k, slot * STRIDE + pad(e), partner(a, c, slot, e), m, mm,
                  pair_index(m, h, mod) == m);
            }
        }
    };

    // Forward real post-process of a tile whose spectrum is in LDS: both bins
    // of each pair stored at base + bin (rows of TPW / 2 columns).
    static __device__ __forceinline__ void pair_post(const FixedArgs<T> &a, const C2<T> *ls,
                                                     const PairWork<true> &p) {
        const bool mod = a.half_shift != 0;
        char *dst = reinterpret_cast<char *>(a.out) + (size_t)(p.t * (uint32_t)a.out_bs) * DB;
        const T half = (T)0.5;
        p.each(a, [&](int k, int z, int o, uint32_t m, uint32_t mm, bool first) {
            const C2<T> zm = ls[z], zo = ls[o];
            if (!mod && m == 0) {
                st(dst, {zm.x + zm.y, zm.x - zm.y});
                return;
            }
            const uint32_t i = first ? m : mm, ci = first ? mm : m;
            const C2<T> zi = first ? zm : zo, zc = first ? zo : zm;
            const C2<T> odd = {(zi.x + zc.x) * half, (zi.y - zc.y) * half};
            const C2<T> ev = {(zi.x - zc.x) * half, (zi.y + zc.y) * half};
            const C2<T> ew = cmul(ev, p.w[k]);
            if (i != ci) st(dst + i * DB, cadd(odd, ew));
            st(dst + ci * DB, cconj(csub(odd, ew)));
        });
    }

    // Inverse real pre-process of a tile's raw bins in LDS, in place: conj(.)
    // of each pre-processed bin (signalsmith-fft.h:478-492).
    static __device__ __forceinline__ void pair_pre(const FixedArgs<T> &a, C2<T> *ls,
                                                    const PairWork<true> &p) {
        const bool mod = a.half_shift != 0;
        p.each(a, [&](int k, int z, int o, uint32_t m, uint32_t mm, bool first) {
            const C2<T> xm = ls[z], xo = ls[o];
            if (!mod && m == 0) {
                ls[z] = {xm.x + xm.y, -(xm.x - xm.y)};
                return;
            }
            const int li = first ? z : o, lc = first ? o : z;
            const C2<T> x = first ? xm : xo, x2 = first ? xo : xm;
            const C2<T> odd = {x.x + x2.x, x.y - x2.y};
            const C2<T> erot = {x.x - x2.x, x.y + x2.y};
            const C2<T> ev = cmulc(erot, p.w[k]);
            if (li != lc) ls[li] = cconj(cadd(odd, ev));
            ls[lc] = csub(odd, ev);  // conj(conj(odd - ev))
        });
    }

    template <int S, bool TW_READY>
    static __device__ __forceinline__ void stages_from(const FixedArgs<T> &a, char *lds_c, int g,
                                                       bool active, int slot, int lid,
                                                       C2<T> (&pf)[PF], int g_next,
                                                       TwBuf<S> &tb) {
        if constexpr (S < NST) {
            TwBuf<S + 1> tn;
            constexpr bool PF_HERE = (S == PF_STAGE);
            stage<S, TW_READY, PF_HERE>(a, lds_c, g, active, slot, lid, pf, g_next, tb, tn);
            stages_from<S + 1, PF_HERE || TW_EARLY>(a, lds_c, g, active, slot, lid, pf, g_next,
                                                     tn);
        }
    }

    // Real inverse pre-process (pairs i, h - i) from HBM into LDS, storing
    // conj(.) so the forward stages compute the inverse (signalsmith-fft.h:478-492).
    static __device__ __forceinline__ void real_pre(const FixedArgs<T> &a, char *lds_c, int g,
                                                    bool active, int slot, int lid) {
        constexpr int H = N;
        C2<T> *ls = reinterpret_cast<C2<T> *>(lds_c) + slot * STRIDE;
        const bool mod = a.half_shift != 0;
        if (active) {
            const C2<T> *x = a.in + (size_t)g * H;
            if (!mod && lid == 0) {
                const C2<T> v = x[0];
                ls[0] = {v.x + v.y, -(v.x - v.y)};
            }
            // kRealBatch pairs at a time, their loads issued before any use
            for (int i0 = (mod ? 0 : 1) + lid; i0 <= H / 2; i0 += kRealBatch * TPT) {
                C2<T> va[kRealBatch], vb[kRealBatch], tw[kRealBatch];
#pragma unroll
                for (int k = 0; k < kRealBatch; ++k) {
                    const int i = i0 + k * TPT;
                    if (i <= H / 2) {
                        const int ci = mod ? (H - 1 - i) : (H - i);
                        va[k] = x[i];
                        vb[k] = x[ci];
                        tw[k] = a.real_tw[i];
                    }
                }
#pragma unroll
                for (int k = 0; k < kRealBatch; ++k) {
                    const int i = i0 + k * TPT;
                    if (i > H / 2 || real_pair_skipped(i, H, mod)) continue;
                    const int ci = mod ? (H - 1 - i) : (H - i);
                    const C2<T> v = va[k], v2 = vb[k];
                    const C2<T> odd = {v.x + v2.x, v.y - v2.y};
                    const C2<T> erot = {v.x - v2.x, v.y + v2.y};
                    const C2<T> ev = cmulc(erot, tw[k]);
                    const C2<T> p = cadd(odd, ev);
                    const C2<T> m = csub(odd, ev);
                    ls[pad(i)] = cconj(p);
                    ls[pad(ci)] = m;
                }
            }
        }
        __syncthreads();
    }

    // Real forward post-process from the spectrum in LDS to HBM
    // (signalsmith-fft.h:459-472).
    static __device__ __forceinline__ void real_post(const FixedArgs<T> &a, char *lds_c, int g,
                                                     bool active, int slot, int lid) {
        constexpr int H = N;
        const C2<T> *ls = reinterpret_cast<const C2<T> *>(lds_c) + slot * STRIDE;
        const bool mod = a.half_shift != 0;
        if (active) {
            C2<T> *y = a.out + (size_t)g * H;
            if (!mod && lid == 0) {
                const C2<T> z = ls[0];
                y[0] = {z.x + z.y, z.x - z.y};
            }
            const T half = (T)0.5;
            // (one pair at a time: grouping the pairs' loads measured slower
            // here, 4.15 -> 3.91 TB/s at 2048, unlike the pre-process)
            for (int i = (mod ? 0 : 1) + lid; i <= H / 2; i += TPT) {
                if (real_pair_skipped(i, H, mod)) continue;
                const int ci = mod ? (H - 1 - i) : (H - i);
                const C2<T> zi = ls[pad(i)], zc = ls[pad(ci)];
                const C2<T> odd = {(zi.x + zc.x) * half, (zi.y - zc.y) * half};
                const C2<T> ev = {(zi.x - zc.x) * half, (zi.y + zc.y) * half};
                const C2<T> e = cmul(ev, a.real_tw[i]);
                y[i] = cadd(odd, e);
                y[ci] = cconj(csub(odd, e));
            }
        }
        __syncthreads();
    }

    static __device__ __forceinline__ void run(const FixedArgs<T> &a, char *lds_c) {
        const int tid = (int)threadIdx.x;
        const int slot = tid / TPT, lid = tid % TPT;
        // stage-0 lanes (the prefetch): column-major in the column modes
        const int slot0 = COL ? tid % TPW : slot, lid0 = COL ? tid / TPW : lid;
        const int ngroups = (a.total_slots + TPW - 1) / TPW;
        C2<T> pf[PF];
        if constexpr (COL) {
            // Column tiles share HBM lines with their neighbours when a tile
            // is narrower than 128 bytes, or when the rows of a strided side
            // do not start on 128-byte lines (a row pitch that is no multiple
            // of 128 bytes): then each window of gridDim.x groups is numbered
            // so that every XCD (blocks go round-robin over them) runs a
            // contiguous run of groups, whose shared lines meet in one L2.
            const int G = (int)gridDim.x;
            constexpr bool NARROW = TPW * (int)DB < 128;
            const auto odd_pitch = [](int32_t es) {
                return es != 1 && (((uint32_t)es * DB) & 127u) != 0;
            };
            const bool share =
                PAIR || NARROW || a.near || odd_pitch(a.in_es) || odd_pitch(a.out_es);
            // (One tile per block: windows of kXcdWindow blocks.  Ranges over
            // the whole launch would set the XCDs 1/8 of the batch apart, at
            // equal places of equal rows, which for power-of-two strides are
            // the same memory channels.  Where the data fits the L2s they are
            // right: a transform then stays on one XCD from pass to pass.)
            const bool whole = PREFETCH || a.near;
            const unsigned win = whole ? 0u : blockIdx.x / kXcdWindow * kXcdWindow;
            const unsigned wb = blockIdx.x - win;
            const unsigned wn = whole || (unsigned)G - win < kXcdWindow ? (unsigned)G - win
                                                                        : kXcdWindow;
            const int off = (int)(win + (share ? xcd_tile(wb, wn) : wb));
            int grp = off;
            if constexpr (!PREFETCH) {  // one tile per block
                load0(a, pf, grp * TPW + slot0, lid0);
                TwBuf<0> t0;
                stages_from<0, false>(a, lds_c, grp * TPW, grp * TPW < a.total_slots, slot, lid,
                                      pf, -1, t0);
                return;
            }
            if (grp < ngroups) load0(a, pf, grp * TPW + slot0, lid0);
            for (int w = 0; w < ngroups; w += G, grp += G) {
                if (grp >= ngroups) break;  // the last window's spare blocks
                const int gn = grp + G;
                const int g_next = gn < ngroups ? gn * TPW + slot0 : -1;
                TwBuf<0> t0;
                stages_from<0, false>(a, lds_c, grp * TPW, grp * TPW < a.total_slots, slot, lid,
                                      pf, g_next, t0);
            }
            return;
        }
        if constexpr (!PREFETCH) {  // one group of transforms per block
            const int g = (int)blockIdx.x * TPW + slot;
            const bool active = g < a.total_slots;
            if (MODE != kModeC2R) load0(a, pf, g, lid);
            if constexpr (MODE == kModeC2R) real_pre(a, lds_c, g, active, slot, lid);
            TwBuf<0> t0;
            stages_from<0, false>(a, lds_c, g, active, slot, lid, pf, -1, t0);
            if constexpr (MODE == kModeR2C) real_post(a, lds_c, g, active, slot, lid);
            return;
        }
        int grp = (int)blockIdx.x;
        if (MODE != kModeC2R && grp < ngroups) load0(a, pf, grp * TPW + slot0, lid0);
        for (; grp < ngroups; grp += (int)gridDim.x) {
            // column modes pass the group's first slot; the stages map lanes
            const int g = grp * TPW + (COL ? 0 : slot);
            const bool active = g < a.total_slots;
            const int gn = grp + (int)gridDim.x;
            const int g_next = gn < ngroups ? gn * TPW + slot0 : -1;
            if constexpr (MODE == kModeC2R) real_pre(a, lds_c, g, active, slot, lid);
            TwBuf<0> t0;
            stages_from<0, false>(a, lds_c, g, active, slot, lid, pf, g_next, t0);
            if constexpr (MODE == kModeR2C) real_post(a, lds_c, g, active, slot, lid);
        }
    }
};

template <class F>
__global__ void __launch_bounds__(F::THREADS, F::MINW > 0 ? F::MINW : 1)
    k_fixed(FixedArgs<typename F::T> a) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    F::run(a, reinterpret_cast<char *>(smem_raw));
}

// Registry entry of a compiled fixed kernel.
struct FixedKernel {
    int n;          // complex length of the core transform
    int variant;    // schedule variant (0 = default)
    int prec;       // 0 F32, 1 F64
    int real;       // 0: C2C kernel; 1: real pair (R2C forward + C2R inverse);
                    // 2: column passes of two-pass plans (kModeColRow, kModeColCol)
                    // 3: the same in wider tiles, for launches that fill the device
                    // 4: kModeColRow in narrower tiles, for launches of few
    bool paired;    // 2: with the paired modes of real transforms
    int tpt, tpw;
    int row_tpw, col_tpw;  // 2 to 4: columns per block in kModeColRow, kModeColCol
    int cus_per_tile;  // 4: for launches of less than a (wide) tile per so many CUs
    int nst;
    int radices[kMaxStages];
    size_t lds_bytes;
    // launch(args, mode, grid, stream): mode kModeC2C / kModeR2C / kModeC2R
    hipError_t (*launch)(const void *args, int mode, unsigned grid, hipStream_t stream);
    int (*blocks_per_cu)(int mode);
};

void register_fixed(const FixedKernel &k);
// variant < 0: the default (variant 0); returns nullptr if none
const FixedKernel *find_fixed(int n, int prec, int real, int variant = -1);
int fixed_variant_count(int n, int prec, int real);

template <class F>
hipError_t fixed_launch_one(const void *args, unsigned grid, hipStream_t stream) {
    static std::once_flag lds_once;
    static hipError_t lds_err = hipSuccess;
    if (allow_max_lds(lds_once, lds_err, (const void *)k_fixed<F>) != hipSuccess) return lds_err;
    hipLaunchKernelGGL((k_fixed<F>), dim3(grid), dim3(F::THREADS), F::LDS_BYTES, stream,
                       *reinterpret_cast<const FixedArgs<typename F::T> *>(args));
    return hipGetLastError();
}

// Blocks per CU to launch at most: the resident ones of a persistent kernel,
// any number of the others.
template <class F>
int fixed_occupancy() {
    if (!F::PREFETCH) return 1 << 22;
    int blocks = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, (const void *)k_fixed<F>,
                                                     F::THREADS, F::LDS_BYTES) != hipSuccess) {
        (void)hipGetLastError();
        return 1;
    }
    return blocks > 0 ? blocks : 1;
}

template <int... Rs>
inline void fixed_fill_radices(FixedKernel &k) {
    k.nst = (int)sizeof...(Rs);
    const int rs[] = {Rs...};
    for (int i = 0; i < k.nst; ++i) k.radices[i] = rs[i];
}

// Registers the complex kernel of one compile-time plan (namespace scope
// object in a .hip file).
template <typename T, int N, int TPT, int TPW, class SCH, int VARIANT, int... Rs>
struct FixedC2C {
    using F = Fixed<T, N, TPT, TPW, kModeC2C, SCH, Rs...>;
    FixedC2C() {
        FixedKernel k{};
        k.n = N;
        k.variant = VARIANT;
        k.prec = FixedElem<T>::prec;
        k.real = 0;
        k.tpt = TPT;
        k.tpw = TPW;
        fixed_fill_radices<Rs...>(k);
        k.lds_bytes = F::LDS_BYTES;
        k.launch = [](const void *args, int, unsigned grid, hipStream_t s) {
            return fixed_launch_one<F>(args, grid, s);
        };
        k.blocks_per_cu = [](int) { return fixed_occupancy<F>(); };
        register_fixed(k);
    }
};

// Registers the real forward / inverse pair of one compile-time plan of the
// half-length complex core N (real length 2N), SF and SI the schedules of the two.
template <typename T, int N, int TPT, int TPW, class SF, class SI, int VARIANT, int... Rs>
struct FixedRealOf {
    using FR = Fixed<T, N, TPT, TPW, kModeR2C, SF, Rs...>;
    using FI = Fixed<T, N, TPT, TPW, kModeC2R, SI, Rs...>;
    FixedRealOf() {
        FixedKernel k{};
        k.n = N;
        k.variant = VARIANT;
        k.prec = FixedElem<T>::prec;
        k.real = 1;
        k.tpt = TPT;
        k.tpw = TPW;
        fixed_fill_radices<Rs...>(k);
        k.lds_bytes = FR::LDS_BYTES;
        k.launch = [](const void *args, int mode, unsigned grid, hipStream_t s) {
            return mode == kModeC2R ? fixed_launch_one<FI>(args, grid, s)
                                    : fixed_launch_one<FR>(args, grid, s);
        };
        k.blocks_per_cu = [](int mode) {
            return mode == kModeC2R ? fixed_occupancy<FI>() : fixed_occupancy<FR>();
        };
        register_fixed(k);
    }
};

template <typename T, int N, int TPT, int TPW, class SCH, int VARIANT, int... Rs>
using FixedReal = FixedRealOf<T, N, TPT, TPW, SCH, SCH, VARIANT, Rs...>;

// Registers the column passes of one compile-time plan of column length N
// (registry kind 2): the first pass of a two-pass plan (kModeColRow, WR columns
// per block), the second (kModeColCol, WC), and with REAL their paired forms
// for real transforms (kModeColRowPre, kModeColColPost, TPW) and the rotating
// ones (kModeColRowRot, kModeColColRot: the plain passes' tiles).  KIND 3: a
// wider tile of the same radices.
template <typename T, int N, int TPT, int TPW, int WR, int WC, class SCH, int VARIANT, bool REAL,
          int KIND, int... Rs>
struct FixedColOf {
    template <int MODE>
    using F = Fixed<T, N, TPT, MODE == kModeColRow ? WR : MODE == kModeColCol ? WC : TPW, MODE,
                    SCH, Rs...>;
    template <int MODE>
    using FRot = Fixed<T, N, TPT, MODE == kModeColRow ? WR : WC, MODE, Rotated<SCH>, Rs...>;
    FixedColOf() {
        FixedKernel k{};
        k.n = N;
        k.variant = VARIANT;
        k.prec = FixedElem<T>::prec;
        k.real = KIND;
        k.paired = REAL;
        k.tpt = TPT;
        k.tpw = TPW;
        k.row_tpw = WR;
        k.col_tpw = WC;
        fixed_fill_radices<Rs...>(k);
        k.lds_bytes = F<kModeColRow>::LDS_BYTES;
        k.launch = [](const void *args, int mode, unsigned grid, hipStream_t s) {
            if constexpr (REAL) {
                if (mode == kModeColRowPre)
                    return fixed_launch_one<F<kModeColRowPre>>(args, grid, s);
                if (mode == kModeColColPost)
                    return fixed_launch_one<F<kModeColColPost>>(args, grid, s);
                if (mode == kModeColRowRot)
                    return fixed_launch_one<FRot<kModeColRow>>(args, grid, s);
                if (mode == kModeColColRot)
                    return fixed_launch_one<FRot<kModeColCol>>(args, grid, s);
            }
            return mode == kModeColCol ? fixed_launch_one<F<kModeColCol>>(args, grid, s)
                                       : fixed_launch_one<F<kModeColRow>>(args, grid, s);
        };
        k.blocks_per_cu = [](int mode) {
            if constexpr (REAL) {
                if (mode == kModeColRowPre) return fixed_occupancy<F<kModeColRowPre>>();
                if (mode == kModeColColPost) return fixed_occupancy<F<kModeColColPost>>();
                if (mode == kModeColRowRot) return fixed_occupancy<FRot<kModeColRow>>();
                if (mode == kModeColColRot) return fixed_occupancy<FRot<kModeColCol>>();
            }
            return mode == kModeColCol ? fixed_occupancy<F<kModeColCol>>()
                                       : fixed_occupancy<F<kModeColRow>>();
        };
        register_fixed(k);
    }
};
template <typename T, int N, int TPT, int TPW, int WR, int WC, class SCH, int... Rs>
using FixedCol =
    FixedColOf<T, N, TPT, TPW, WR, WC, SCH, 0, std::is_arithmetic<T>::value, 2, Rs...>;
// Registers the plain first pass in a narrower tile (registry kind 4), for
// launches of less than a tile of the ordinary width per CUS compute units.
template <typename T, int N, int TPT, int TPW, int CUS, class SCH, int... Rs>
struct FixedRowNarrow {
    using F = Fixed<T, N, TPT, TPW, kModeColRow, SCH, Rs...>;
    FixedRowNarrow() {
        FixedKernel k{};
        k.n = N;
        k.prec = FixedElem<T>::prec;
        k.real = 4;
        k.tpt = TPT;
        k.tpw = k.row_tpw = TPW;
        k.cus_per_tile = CUS;
        fixed_fill_radices<Rs...>(k);
        k.lds_bytes = F::LDS_BYTES;
        k.launch = [](const void *args, int, unsigned grid, hipStream_t s) {
            return fixed_launch_one<F>(args, grid, s);
        };
        k.blocks_per_cu = [](int) { return fixed_occupancy<F>(); };
        register_fixed(k);
    }
};
template <typename T, int N, int TPT, int TPW, class SCH, int... Rs>
using FixedColWide = FixedColOf<T, N, TPT, TPW, TPW, TPW, SCH, 0, false, 3, Rs...>;

}  // namespace sfft
