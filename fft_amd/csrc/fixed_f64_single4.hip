// fixed_f64_single4.hip -- compile-time plans, complex FP64, single
// pass: part 1 of 2 of the fast lengths that the other files leave.
// Radices are those the runtime planner's cost model chooses at 16 elements a
// thread, so that bits and every other use of the plan stay as they were;
// about 256 threads a block; one group per block (the persistent form of these
// kernels had lost).  Bound by HBM.  Listed where faster over both directions
// with neither 3 % slower, batches of 128 MB:
// 1.17-1.8x over the runtime-planned pass, median 1.23x.
#include "fixed.h"

namespace sfft {
namespace {
const FixedC2C<double, 64, 4, 64, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 4> c64;
const FixedC2C<double, 128, 8, 32, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 8> c128;
const FixedC2C<double, 4050, 338, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 6, 3> c4050;
const FixedC2C<double, 5400, 360, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 8, 3> c5400;
const FixedC2C<double, 6075, 405, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 3, 3, 3> c6075;
const FixedC2C<double, 6561, 438, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 3, 3, 3, 3, 3, 3, 3, 3> c6561;
const FixedC2C<double, 7290, 486, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 3, 3, 3, 3, 3, 2> c7290;
}  // namespace
}  // namespace sfft
