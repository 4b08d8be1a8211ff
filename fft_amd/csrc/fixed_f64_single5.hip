// fixed_f64_single5.hip -- compile-time plans, complex FP64, single
// pass: part 2 of 2 of the fast lengths that the other files leave.
// Radices are those the runtime planner's cost model chooses at 16 elements a
// thread, so that bits and every other use of the plan stay as they were;
// about 256 threads a block; one group per block (the persistent form of these
// kernels had lost).  Bound by HBM.  Listed where faster over both directions
// with neither 3 % slower, batches of 128 MB:
// 1.17-1.8x over the runtime-planned pass, median 1.23x.
#include "fixed.h"

namespace sfft {
namespace {
const FixedC2C<double, 120, 8, 32, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 8> c120;
const FixedC2C<double, 240, 16, 16, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15> c240;
const FixedC2C<double, 4500, 300, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 5, 4> c4500;
const FixedC2C<double, 5625, 375, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 5, 5> c5625;
const FixedC2C<double, 6250, 417, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 5, 5, 5, 5, 5, 2> c6250;
const FixedC2C<double, 6750, 450, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 15, 2> c6750;
const FixedC2C<double, 7500, 500, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 5, 5, 5, 4> c7500;
}  // namespace
}  // namespace sfft
