// fixed_col_f64_0.hip -- compile-time column passes of two-pass plans, FP64
// (and the paired passes of real ones): part 1 of 3 of the mixed-radix column
// lengths of fixed_col_mixed.hip, with the radices and threads the runtime
// planner's cost model chooses in FP64 and the widest tile of up to 16 columns
// (256-byte rows) of which two blocks fit a CU.
#include "fixed.h"

namespace sfft {
namespace {
const FixedCol<double, 81, 9, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 9, 9> d81;
const FixedCol<double, 125, 9, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 5, 5, 5> d125;
const FixedCol<double, 135, 15, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 9> d135;
const FixedCol<double, 144, 12, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 12, 12> d144;
const FixedCol<double, 150, 15, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 10> d150;
const FixedCol<double, 160, 16, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 10> d160;
const FixedCol<double, 162, 18, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 9, 9, 2> d162;
const FixedCol<double, 180, 15, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 12> d180;
const FixedCol<double, 192, 16, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 12> d192;
const FixedCol<double, 200, 14, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 8, 5, 5> d200;
const FixedCol<double, 216, 18, 16, 16, 16, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 6, 6, 6> d216;
}  // namespace
}  // namespace sfft
