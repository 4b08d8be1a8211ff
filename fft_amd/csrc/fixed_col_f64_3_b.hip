// fixed_col_f64_3_b.hip -- compile-time column passes of two-pass plans, FP64:
// column lengths 576 to 1000 (part 2 of 2), which with those of
// fixed_col_mixed.hip give nearly every fast length up to 2^20 a split of two
// compiled passes.  Radices and threads of the runtime planner's cost model at
// 16 elements a thread, the widest tile of which two blocks fit a CU.
#include "fixed.h"

namespace sfft {
namespace {
const FixedCol<double, 800, 80, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 10, 10, 8> c800;
const FixedCol<double, 810, 90, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 10, 9, 9> c810;
const FixedCol<double, 864, 72, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 12, 12, 6> c864;
const FixedCol<double, 900, 60, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 15, 4> c900;
const FixedCol<double, 960, 64, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 15, 4> c960;
const FixedCol<double, 972, 108, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 12, 9, 9> c972;
const FixedCol<double, 1000, 100, 4, 4, 4, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 10, 10, 10> c1000;
}  // namespace
}  // namespace sfft
