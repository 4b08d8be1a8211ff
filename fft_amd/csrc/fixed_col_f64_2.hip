// fixed_col_f64_2.hip -- compile-time column passes of two-pass plans, FP64
// (and the paired passes of real ones): part 3 of 3 of the mixed-radix column
// lengths of fixed_col_mixed.hip, with the radices and threads the runtime
// planner's cost model chooses in FP64 and the widest tile of up to 16 columns
// (256-byte rows) of which two blocks fit a CU.
#include "fixed.h"

namespace sfft {
namespace {
const FixedCol<double, 384, 26, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 8, 3> d384;
const FixedCol<double, 400, 27, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 5, 5> d400;
const FixedCol<double, 405, 45, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 9, 9, 5> d405;
const FixedCol<double, 432, 36, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 12, 6, 6> d432;
const FixedCol<double, 450, 30, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 15, 2> d450;
const FixedCol<double, 480, 32, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 15, 2> d480;
const FixedCol<double, 486, 54, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 9, 9, 6> d486;
const FixedCol<double, 500, 50, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 10, 10, 5> d500;
const FixedCol<double, 540, 45, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 6, 6> d540;
const FixedCol<double, 625, 42, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 5, 5, 5, 5> d625;
const FixedCol<double, 729, 81, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 9, 9, 9> d729;
}  // namespace
}  // namespace sfft
