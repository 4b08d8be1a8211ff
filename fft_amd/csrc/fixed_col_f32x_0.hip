// fixed_col_f32x_0.hip -- compile-time column passes of two-pass plans
// of FP32 storage under FP64 arithmetic, part 1 of 2 of the mixed-radix lengths
// of fixed_col_mixed.hip and fixed_col_large.hip: FP64 shapes.  Bound by HBM and
// LDS; batches of 128 MB, both passes against runtime-planned ones: 1.1-2.1x
// (26244 374 -> 176 us, 186624 338 -> 188, 972000 347 -> 204).
#include "fixed.h"

namespace sfft {
namespace {
using X = Stored<StoreF32>;
const FixedCol<X, 81, 9, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 9, 9> x81;
const FixedCol<X, 135, 15, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 9> x135;
const FixedCol<X, 150, 15, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 10> x150;
const FixedCol<X, 162, 18, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 9, 9, 2> x162;
const FixedCol<X, 192, 16, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 12> x192;
const FixedCol<X, 216, 18, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 6, 6, 6> x216;
const FixedCol<X, 240, 16, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 15> x240;
const FixedCol<X, 250, 25, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 10, 5, 5> x250;
const FixedCol<X, 288, 24, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 12, 12, 2> x288;
const FixedCol<X, 320, 22, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 5, 4> x320;
const FixedCol<X, 360, 24, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 8, 3> x360;
const FixedCol<X, 384, 26, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 8, 3> x384;
const FixedCol<X, 405, 45, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 9, 9, 5> x405;
const FixedCol<X, 450, 30, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 15, 2> x450;
const FixedCol<X, 486, 54, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 9, 9, 6> x486;
const FixedCol<X, 540, 45, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 6, 6> x540;
const FixedCol<X, 600, 40, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 8, 5> x600;
const FixedCol<X, 640, 43, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 8, 5> x640;
const FixedCol<X, 675, 45, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 15, 3> x675;
const FixedCol<X, 729, 81, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 9, 9, 9> x729;
const FixedCol<X, 768, 52, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 16, 3> x768;
const FixedCol<X, 810, 90, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 10, 9, 9> x810;
const FixedCol<X, 900, 60, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 15, 4> x900;
const FixedCol<X, 972, 108, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 12, 9, 9> x972;
}  // namespace
}  // namespace sfft
