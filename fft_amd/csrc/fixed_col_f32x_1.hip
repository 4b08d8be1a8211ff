// fixed_col_f32x_1.hip -- compile-time column passes of two-pass plans
// of FP32 storage under FP64 arithmetic, part 2 of 2 of the mixed-radix lengths
// of fixed_col_mixed.hip and fixed_col_large.hip: FP64 shapes.  Bound by HBM and
// LDS; batches of 128 MB, both passes against runtime-planned ones: 1.1-2.1x
// (26244 374 -> 176 us, 186624 338 -> 188, 972000 347 -> 204).
#include "fixed.h"

namespace sfft {
namespace {
using X = Stored<StoreF32>;
const FixedCol<X, 125, 9, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 5, 5, 5> x125;
const FixedCol<X, 144, 12, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 12, 12> x144;
const FixedCol<X, 160, 16, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 10> x160;
const FixedCol<X, 180, 15, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 12> x180;
const FixedCol<X, 200, 14, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 8, 5, 5> x200;
const FixedCol<X, 225, 15, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 15> x225;
const FixedCol<X, 243, 27, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 9, 9, 3> x243;
const FixedCol<X, 270, 23, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 6, 3> x270;
const FixedCol<X, 300, 20, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 5, 4> x300;
const FixedCol<X, 324, 36, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 9, 6, 6> x324;
const FixedCol<X, 375, 25, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 5, 5> x375;
const FixedCol<X, 400, 27, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 5, 5> x400;
const FixedCol<X, 432, 36, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 12, 6, 6> x432;
const FixedCol<X, 480, 32, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 15, 2> x480;
const FixedCol<X, 500, 50, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 10, 10, 5> x500;
const FixedCol<X, 576, 48, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 6, 6> x576;
const FixedCol<X, 625, 42, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 5, 5, 5, 5> x625;
const FixedCol<X, 648, 72, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 12, 9, 6> x648;
const FixedCol<X, 720, 48, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 15, 3> x720;
const FixedCol<X, 750, 75, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 10, 5> x750;
const FixedCol<X, 800, 80, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 10, 10, 8> x800;
const FixedCol<X, 864, 72, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 12, 12, 6> x864;
const FixedCol<X, 960, 64, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 15, 4> x960;
const FixedCol<X, 1000, 100, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 10, 10, 10> x1000;
}  // namespace
}  // namespace sfft
