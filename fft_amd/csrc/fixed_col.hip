// fixed_col.hip -- compile-time column passes of two-pass plans, complex
// FP32, FP64 and F32X.  FixedCol<type, column length N, threads per column,
// columns per block in the paired modes, in the first pass, in the second,
// Sched<...>, radices...>; a two-pass plan whose column length has one uses it
// for that pass (same radices as the runtime-planned pass, so the same bits).
// Tile widths by measurement (256 MB per launch, 256 columns): wide rows pay in
// the first pass, whose input comes from HBM (128: 64 columns 103 us, 32 112, 16
// 123), more blocks in the second, which reads what the last-level cache still
// holds (512: 8 columns 81 us, 16 89; 2048: 4 columns 104, 8 122).
// Such a wide first pass leaves CUs idle where a launch has few tiles.  Below a
// tile per CU 128 and 144 take half the width, and 625 below a tile per two
// (FixedRowNarrow<..., columns, CUs per tile, ...>; both directions, wide / narrow:
// 20736 x 21 24.9 / 20.0 us, x 102 45.0 / 40.9, 90000 x 26 51.8 / 38.3, 16000 x 64
// 32.3 / 29.3, x 131 48.0 / 46.5; 625: 78125 x 14 37.8 / 33.2, but x 26 44.0 /
// 59.3).  81 gains and loses 4 % and keeps the wide one.
// FP32 and FP64 first passes read their input non-temporally (Sched NT 1;
// 2^19 x 64 and 2^18 x 128 +13-15 %, 1024 and 2048 +3-6 %); non-temporal output
// stores of the second pass slowed the lengths whose output is read back (the
// real post-process) and some others (up to 8 %).
#include "fixed.h"

namespace sfft {
namespace {
const FixedCol<float, 128, 8, 32, 64, 32, Sched<0, 0, 0, 0, kLdsPadShift, 1>, 16, 8> col128;
const FixedRowNarrow<float, 128, 8, 32, 1, Sched<0, 0, 0, 0, kLdsPadShift, 1>, 16, 8> row128;
const FixedCol<float, 256, 16, 32, 32, 32, Sched<0, 0, 0, 0, kLdsPadShift, 1>, 16, 16> col256;
const FixedCol<float, 512, 32, 16, 16, 8, Sched<0, 0, 0, 0, kLdsPadShift, 1>, 16, 16, 2> col512;
const FixedCol<float, 1024, 64, 8, 8, 8, Sched<0, 0, 0, 0, kLdsPadShift, 1>, 16, 16, 4> col1024;
const FixedCol<float, 2048, 128, 8, 8, 4, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift, 1>, 16, 16, 8>
    col2048;
// FP64 (16-byte values; 256 MB per launch with 256 columns, first / second
// pass, runtime-planned pass -> here): 128 103/87 -> 93/80 us, 256 107/87 ->
// 97/82, 512 121/95 -> 113/89, 1024 158/133 -> 135/111, 2048 198/155 -> 163/138.
// 172 registers, two waves per SIMD: a third (168 registers) spilled, 111 -> 128
// us in the second pass of 1024.
const FixedCol<double, 128, 8, 16, 16, 16, Sched<0, 0, 0, 0, kLdsPadShift, 1>, 16, 8> col128d;
const FixedCol<double, 256, 16, 16, 16, 16, Sched<0, 0, 0, 0, kLdsPadShift, 1>, 16, 16> col256d;
const FixedCol<double, 512, 32, 8, 8, 8, Sched<0, 0, 0, 0, kLdsPadShift, 1>, 16, 16, 2> col512d;
const FixedCol<double, 1024, 64, 4, 4, 4, Sched<0, 0, 0, 0, kLdsPadShift, 1>, 16, 16, 4> col1024d;
const FixedCol<double, 2048, 128, 4, 4, 4, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift, 1>, 16, 16, 8>
    col2048d;
// FP32 storage under FP64 arithmetic: the same shapes
using X = Stored<StoreF32>;
const FixedCol<X, 128, 8, 16, 16, 16, Sched<0, 0, 0, 0>, 16, 8> col128x;
const FixedCol<X, 256, 16, 16, 16, 16, Sched<0, 0, 0, 0>, 16, 16> col256x;
const FixedCol<X, 512, 32, 8, 8, 8, Sched<0, 0, 0, 0>, 16, 16, 2> col512x;
const FixedCol<X, 1024, 64, 4, 4, 4, Sched<0, 0, 0, 0>, 16, 16, 4> col1024x;
const FixedCol<X, 2048, 128, 4, 4, 4, Sched<kNoPrefetch, 0, 0, 0>, 16, 16, 8> col2048x;
}  // namespace
}  // namespace sfft
