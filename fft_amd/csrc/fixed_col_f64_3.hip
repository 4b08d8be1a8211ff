// fixed_col_f64_3.hip -- compile-time column passes of two-pass plans, FP64:
// column lengths 576 to 1000 (part 1 of 2), which with those of
// fixed_col_mixed.hip give nearly every fast length up to 2^20 a split of two
// compiled passes.  Radices and threads of the runtime planner's cost model at
// 16 elements a thread, the widest tile of which two blocks fit a CU.
#include "fixed.h"

namespace sfft {
namespace {
const FixedCol<double, 576, 48, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 6, 6> c576;
const FixedCol<double, 600, 40, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 8, 5> c600;
const FixedCol<double, 640, 43, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 8, 5> c640;
const FixedCol<double, 648, 72, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 12, 9, 6> c648;
const FixedCol<double, 675, 45, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 15, 3> c675;
const FixedCol<double, 720, 48, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 15, 3> c720;
const FixedCol<double, 750, 75, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 10, 5> c750;
const FixedCol<double, 768, 52, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 16, 3> c768;
}  // namespace
}  // namespace sfft
