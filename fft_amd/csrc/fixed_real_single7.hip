// fixed_real_single7.hip -- compile-time plans, real FP32 (real
// length 2h), single pass: part 4 of 8 of the fast half lengths h up to 15625
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
const FixedReal<float, 100, 10, 26, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 10, 10> r200;
const FixedReal<float, 250, 25, 10, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 10> r500;
const FixedReal<float, 675, 45, 6, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 3> r1350;
const FixedReal<float, 1800, 120, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 8> r3600;
const FixedReal<float, 3125, 209, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 25, 5> r6250;
const FixedReal<float, 5400, 360, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 8, 3> r10800;
const FixedReal<float, 7680, 512, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 16, 15, 2> r15360;
const FixedReal<float, 12150, 1013, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 15, 15, 6, 3, 3> r24300;
}  // namespace
}  // namespace sfft
