// fixed_real_single6.hip -- compile-time plans, real FP32 (real
// length 2h), single pass: part 3 of 8 of the fast half lengths h up to 15625
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
const FixedReal<float, 96, 8, 32, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 6> r192;
const FixedReal<float, 240, 16, 16, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 15> r480;
const FixedReal<float, 625, 25, 10, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 25> r1250;
const FixedReal<float, 1620, 180, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 15, 12, 9> r3240;
const FixedReal<float, 3000, 200, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 15, 8> r6000;
const FixedReal<float, 5000, 313, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 25, 8> r10000;
const FixedReal<float, 7500, 500, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 15, 5, 4> r15000;
const FixedReal<float, 11250, 750, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 25, 15, 15, 2> r22500;
const FixedReal<float, 15625, 625, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 25, 25, 25> r31250;
}  // namespace
}  // namespace sfft
