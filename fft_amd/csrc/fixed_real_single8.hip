// fixed_real_single8.hip -- compile-time plans, real FP32 (real
// length 2h), single pass: part 5 of 8 of the fast half lengths h up to 15625
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
const FixedReal<float, 108, 12, 21, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 9> r216;
const FixedReal<float, 256, 16, 16, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 16, 16> r512;
const FixedReal<float, 750, 50, 5, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 15, 2> r1500;
const FixedReal<float, 1875, 125, 2, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 15, 5> r3750;
const FixedReal<float, 3200, 200, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 16, 8> r6400;
const FixedReal<float, 5625, 375, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 25, 15, 15> r11250;
const FixedReal<float, 8748, 972, 1, Sched<0, 0, 0, 0, kLdsPadShift>, 0, 12, 9, 9, 9> r17496;
const FixedReal<float, 12500, 834, 1, Sched<kNoPrefetch, 0, 0, 0, kLdsPadShift>, 0, 25, 25, 5, 4> r25000;
}  // namespace
}  // namespace sfft
