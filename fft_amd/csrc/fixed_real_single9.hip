// fixed_real_single9.hip -- compile-time plans, real FP32 (real
// length 2h), single pass: part 6 of 8 of the fast half lengths h up to 15625
// that the other files leave.
// Radices are those the runtime planner's cost model chooses at 16 elements a
// thread, so that bits and every other use of the plan stay as they were;
// about 256 threads a block; one group per block (the persistent form of these
// kernels had lost).  Bound by HBM.  Listed where faster over both directions
// with neither 3 % slower, batches of 128 MB:
// R2C forward and inverse median 1.24x (10800 114 + 127 -> 75 + 76 us, 31250 118
// + 121 -> 106 + 106), half-bin shifted 1.28x; h = 64, 72, 75, 80, 125, 200 and
// 2500 lose up to 18 % in one direction of one kind.
#include "fixed.h"

namespace sfft {
namespace {
const FixedReal<float, 120, 8, 32, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 8> r240;
const FixedReal<float, 360, 24, 11, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 8, 3> r720;
const FixedReal<float, 900, 60, 4, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 4> r1800;
const FixedReal<float, 1920, 128, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15, 8> r3840;
const FixedReal<float, 3375, 225, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 15> r6750;
const FixedReal<float, 6000, 400, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 16, 15> r12000;
const FixedReal<float, 9000, 600, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 8, 5> r18000;
const FixedReal<float, 13122, 875, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 3, 3, 3, 3, 3, 3, 3, 3, 2> r26244;
}  // namespace
}  // namespace sfft
