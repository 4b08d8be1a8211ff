// fixed_col_large_b.hip -- compile-time column passes of two-pass plans, FP32:
// column lengths 576 to 1000 (part 2 of 2), which with those of
// fixed_col_mixed.hip give nearly every fast length up to 2^20 a split of two
// compiled passes.  Radices and threads of the runtime planner's cost model at
// 16 elements a thread, the widest tile of which two blocks fit a CU.
#include "fixed.h"

namespace sfft {
namespace {
const FixedCol<float, 800, 50, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 25, 16, 2> c800;
const FixedCol<float, 810, 90, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 10, 9, 9> c810;
const FixedCol<float, 864, 72, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 12, 12, 6> c864;
const FixedCol<float, 900, 60, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 15, 15, 4> c900;
const FixedCol<float, 960, 64, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 16, 15, 4> c960;
const FixedCol<float, 972, 108, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 12, 9, 9> c972;
const FixedCol<float, 1000, 100, 8, 8, 8, Sched<0, 0, 0, 0, kLdsNoPad, 1>, 10, 10, 10> c1000;
}  // namespace
}  // namespace sfft
