// fixed_col_f64_1.hip -- compile-time column passes of two-pass plans, FP64
// (and the paired passes of real ones): part 2 of 3 of the mixed-radix column
// lengths of fixed_col_mixed.hip, with the radices and threads the runtime
// planner's cost model chooses in FP64 and the widest tile of up to 16 columns
// (256-byte rows) of which two blocks fit a CU.
#include "fixed.h"

namespace sfft {
namespace {
const FixedCol<double, 225, 15, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 15> d225;
const FixedCol<double, 240, 16, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 15> d240;
const FixedCol<double, 243, 27, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 9, 9, 3> d243;
const FixedCol<double, 250, 25, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 10, 5, 5> d250;
const FixedCol<double, 270, 23, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 6, 3> d270;
const FixedCol<double, 288, 24, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 12, 12, 2> d288;
const FixedCol<double, 300, 20, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 5, 4> d300;
const FixedCol<double, 320, 22, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 5, 4> d320;
const FixedCol<double, 324, 36, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 9, 6, 6> d324;
const FixedCol<double, 360, 24, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 8, 3> d360;
const FixedCol<double, 375, 25, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 5, 5> d375;
}  // namespace
}  // namespace sfft
